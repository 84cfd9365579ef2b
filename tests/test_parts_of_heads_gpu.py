"""The kernel that adds the parts of a q/k/v projection while it prepares the heads asks for two, three or four parts at once, in as few turns as that takes: every
number of parts from 2 to 11 against the product and the preparation one after the other, which add in the same order: the same bits."""
import ctypes
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# (tokens, query heads, key/value heads, dims of a head), {parts: k}
SIZES = [(65, 4, 1, 64, {2: 256, 3: 576, 4: 1024, 5: 1600, 6: 2304, 7: 3136, 8: 4096, 9: 5184, 10: 6400, 11: 7744})]


@pytest.fixture(scope="module")
def ops():
    from xeno_rt_amd.ops import load_ops
    return load_ops()


def rand(*shape, seed, scale=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).to(torch.bfloat16).to(DEV)


@pytest.mark.parametrize("tokens,nh,nkv,hd,parts,k", [(*size[:4], parts, k) for size in SIZES for parts, k in size[4].items()])
@pytest.mark.parametrize("longest_run", [1, 65])                  # values one by one, and by workgroups of their own
def test_every_number_of_parts(ops, tokens, nh, nkv, hd, parts, k, longest_run):
    width = (nh + 2 * nkv) * hd
    rows, columns = ctypes.c_int(), ctypes.c_int()
    assert ops.lib.xrt_linear_parts(tokens, width, k, 0, 0, ctypes.byref(rows), ctypes.byref(columns)) == parts
    a, w = rand(tokens, k, seed=1), rand(width, k, seed=2, scale=k ** -0.5)
    positions = torch.arange(30, 30 + tokens, dtype=torch.int32, device=DEV)
    slots = torch.zeros(tokens, dtype=torch.int32, device=DEV)
    theta = (10000.0 ** (torch.arange(hd // 2) * 2.0 / hd)).to(DEV)
    gains = [1.0 + rand(hd, seed=s) for s in (3, 4)]
    args = dict(q_norm=gains[0], k_norm=gains[1], norm_eps=1e-5, rope_theta=theta, rope_dim=hd, rope_scale=1.0, longest_run=longest_run)

    def cache():
        return SimpleNamespace(k=torch.zeros(3, nkv, 64, hd, dtype=torch.bfloat16, device=DEV), v=torch.zeros(3, nkv, hd, 64, dtype=torch.bfloat16, device=DEV),
                               block_table=torch.tensor([[2, 0]], dtype=torch.int32, device=DEV))
    got, want = (torch.full((tokens, width), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    kv_got, kv_want = cache(), cache()
    ops.linear_qkv(a, w, got, nh, nkv, hd, positions, slots, kv=kv_got, **args)
    ops.linear(a, w, want)
    ops.qkv_prepare(want, nh, nkv, hd, positions, slots, kv=kv_want, **args)
    assert torch.equal(got, want) and torch.equal(kv_got.k, kv_want.k) and torch.equal(kv_got.v, kv_want.v)
    assert bool((kv_got.k != 0).any()) and bool((kv_got.v != 0).any())
