"""Products whose rows are dealt evenly to tiles that could hold more (a wavefront then has all of its blocks of 16 rows, or one or two fewer), and parts along k that are
dealt to the dies part by part: every tile height, the last tile full and not, one and more steps along k, against sums in 64 bits."""
import ctypes

import pytest
import torch

import plain_llama as P

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
MODES = {"store": 0, "add": 1, "gated": 2}
TILES = {"256": 0, "192": 1, "128": 2, "256 and 128": 3}
ULP = 4e-3                                                       # a bfloat16 result: half of its last place
SUMS = 1e-5                                                      # float32 sums of products of bfloat16 numbers


@pytest.fixture(scope="module")
def ops():
    from xeno_rt_amd.ops import load_ops
    return load_ops()


def rand(*shape, dtype=torch.float32, seed=0, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


def rel(got, want):
    return float((got.double() - want.double()).abs().max()) / max(1e-30, float(want.double().abs().max()))


def height(m, most):
    tiles = -(-m // most)
    return (-(-m // tiles) + 15) // 16 * 16


def route(ops, m, n, k, mode):
    """(parts along k, a tile's rows) of the product."""
    rows, columns = ctypes.c_int(), ctypes.c_int()
    parts = ops.lib.xrt_linear_parts(m, n, k, MODES[mode], 0, ctypes.byref(rows), ctypes.byref(columns))
    if parts > 1:
        return parts, rows.value
    tiles = ops.lib.xrt_linear_tiles(0 if mode == "add" else 1, m, n, k, MODES[mode])
    return 1, {0: 256, 1: 192, 2: 128, 3: 256}.get(tiles, 0)


# (m, n, k, a tile's rows at most, the rows it then has, whether k is cut)
HEIGHTS = {
    "store": [(778, 4096, 128, 128, 112, False), (900, 4096, 192, 128, 128, False), (257, 12320, 64, 128, 96, False), (390, 16640, 128, 192, 144, False),
              (778, 12320, 128, 192, 160, False), (700, 12320, 64, 192, 176, False), (778, 14344, 128, 256, 208, False), (1100, 12320, 128, 256, 224, False),
              (900, 14344, 64, 256, 240, False), (199, 8200, 4096, 192, 112, True), (257, 2048, 14336, 192, 144, True), (778, 2048, 8192, 192, 160, True),
              (520, 2048, 8192, 192, 176, True), (778, 2048, 14336, 256, 208, True), (1100, 4096, 8192, 256, 224, True)],
    "add": [(778, 8200, 2048, 128, 112, False), (257, 16640, 2048, 128, 96, False), (257, 25608, 2048, 192, 144, False), (520, 16640, 320, 192, 176, False),
            (778, 14344, 2048, 256, 208, False), (900, 14344, 2048, 256, 240, False), (199, 12320, 2048, 192, 112, True), (300, 12320, 2048, 192, 160, True),
            (333, 12320, 2048, 192, 176, True), (900, 2048, 14336, 256, 240, True)],
    "gated": [(520, 4096, 128, 128, 112, False), (257, 6152, 128, 128, 96, False), (390, 8200, 128, 192, 144, False), (700, 6152, 128, 192, 176, False),
              (778, 12320, 128, 256, 208, False), (580, 8200, 128, 256, 208, False), (700, 8200, 128, 256, 240, False), (520, 2048, 8192, 192, 176, True)]}


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("mode,size", [(mode, size) for mode in HEIGHTS for size in HEIGHTS[mode]])
def test_rows_dealt_evenly_to_tiles(ops, mode, size, packed):
    m, n, k, most, rows, cut = size
    parts, tile = route(ops, m, n, k, mode)
    assert tile == most and height(m, most) == rows and (parts > 1) == cut
    a = rand(m, k, dtype=torch.bfloat16, seed=m)
    a[m - 1] *= 3.0                                               # (the last row is what rows beyond the last are read as)
    w = rand(2 * n if mode == "gated" else n, k, dtype=torch.bfloat16, seed=n, scale=0.1)
    sums = a.double() @ w.double().t()
    matrix = w if not packed else ops.pack(w, "gated", gated_n=n) if mode == "gated" else ops.pack(w, "tiles")
    around = torch.full((m + 16, n), 7.0, dtype=torch.float32 if mode == "add" else torch.bfloat16, device=DEV)      # what lies behind the result stays
    out = around[:m]
    if mode == "gated":
        ops.linear_glu(a, matrix, out)
        assert rel(out, P.swiglu(sums[:, :n].cpu(), sums[:, n:].cpu()).to(DEV)) < ULP * 2
    elif mode == "store":
        ops.linear(a, matrix, out)
        assert rel(out, sums) < ULP * 2
        exact = torch.empty(m, n, device=DEV)
        ops.linear(a, matrix, exact)
        assert rel(exact, sums) < SUMS
    else:
        before = rand(m, n, seed=5)
        out.copy_(before)
        ops.linear(a, matrix, out, accumulate=True)
        assert rel(out, before.double() + sums) < SUMS
    assert bool((around[m:] == 7.0).all())


# The fixed array of xrt_linear_static holds the sums of few parts: where the product alone would have more of them, or parts where it had none, it is served as before.
@pytest.mark.parametrize("m,n,k,mode", [(684, 696, 11456, "add"), (780, 1440, 7104, "store"), (842, 5152, 3072, "add"), (481, 4688, 1408, "add")])
def test_products_of_the_fixed_array_whose_parts_would_not_fit(ops, m, n, k, mode):
    lib = ops.lib
    pointer = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    a, w = rand(m, k, dtype=torch.bfloat16, seed=1), rand(n, k, dtype=torch.bfloat16, seed=2, scale=0.1)
    assert int(lib.xrt_linear_workspace(pointer(a), pointer(w), 1, m, n, k, MODES[mode])) > int(lib.xrt_linear_static_floats())
    out = rand(m, n, seed=3) if mode == "add" else torch.zeros(m, n, dtype=torch.bfloat16, device=DEV)
    want = a.double() @ w.double().t() + (out.double() if mode == "add" else 0.0)
    status = lib.xrt_linear_static(pointer(a), pointer(w), 1, pointer(out), 0 if mode == "add" else 1, m, n, k, MODES[mode],
                                   ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert status == 0, lib.xrt_last_error().decode()
    assert rel(out, want) < (SUMS if mode == "add" else ULP * 2)
