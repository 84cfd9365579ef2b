"""Which products xrt_linear_static serves, and how: every one whose partial sums fit its array, by xrt_linear's own plan; larger ones in fewer parts; those that the plan of few
parts does not cut uncut, without the array. (What it refuses, and that calls leave each other alone: test_zz_no_alloc.py.)"""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
STORE, ADD = 0, 1


def library():
    from xeno_rt_amd.ops import build
    lib = ctypes.CDLL(build.find_library() or build.build())
    lib.xrt_last_error.restype = ctypes.c_char_p
    lib.xrt_linear_workspace.restype = lib.xrt_linear_static_floats.restype = ctypes.c_long
    return lib


def pointer(tensor):
    return ctypes.c_void_p(0 if tensor is None else tensor.data_ptr())


def results(lib, m, n, k, mode):
    """The product by xrt_linear_static, by xrt_linear with a workspace and without one, its true value and the floats it asks for."""
    g = torch.Generator(device="cuda").manual_seed(m)
    a = torch.randn((m, k), generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn((n, k), generator=g, device="cuda") * 0.05).to(torch.bfloat16)
    before = torch.randn((m, n), generator=g, device="cuda") if mode == ADD else torch.zeros(m, n, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    need = int(lib.xrt_linear_workspace(pointer(a), pointer(w), 1, m, n, k, mode))
    workspace = torch.empty(max(need, 1), device="cuda")
    by_static, cut, whole = (before.clone() for _ in range(3))
    assert lib.xrt_linear_static(pointer(a), pointer(w), 1, pointer(by_static), 0, m, n, k, mode, stream) == 0, lib.xrt_last_error().decode()
    assert lib.xrt_linear(pointer(a), pointer(w), 1, pointer(cut), 0, m, n, k, mode, pointer(workspace), ctypes.c_long(need), stream) == 0
    assert lib.xrt_linear(pointer(a), pointer(w), 1, pointer(whole), 0, m, n, k, mode, None, ctypes.c_long(0), stream) == 0
    true = before.double() + a.double() @ w.double().t()
    assert float((by_static - true).abs().max()) < 1e-5 * float(true.abs().max())        # float32 sums of products of bfloat16 numbers
    return by_static, cut, whole, need


# the plan of few parts would not fit, but the product's own does: two of them cut, the last not
@pytest.mark.parametrize("m,n,k,mode", [(134, 2696, 9536, ADD), (1179, 512, 14336, STORE), (1002, 4096, 2048, STORE)])
def test_what_fits_by_its_own_plan_is_served_by_it(m, n, k, mode):
    lib = library()
    by_static, cut, _, need = results(lib, m, n, k, mode)
    assert need <= int(lib.xrt_linear_static_floats()) and (need > 0) == (k != 2048)
    assert torch.equal(by_static, cut)


# cut by xrt_linear, into parts that fit or do not, but not by the plan of few parts: without the array, whatever runs beside it
@pytest.mark.parametrize("m,n,k,mode,fits", [(236, 8672, 1984, ADD, True), (826, 2368, 1408, ADD, True), (237, 9096, 1600, ADD, False), (842, 5152, 3072, ADD, False)])
def test_what_few_parts_would_not_cut_leaves_the_array_alone(m, n, k, mode, fits):
    lib = library()
    by_static, cut, whole, need = results(lib, m, n, k, mode)
    assert need > 0 and (need <= int(lib.xrt_linear_static_floats())) == fits
    assert torch.equal(by_static, whole) and not torch.equal(by_static, cut)
