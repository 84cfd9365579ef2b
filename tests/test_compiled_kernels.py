"""What the compiler made of the kernels: read from the built library, without a GPU."""
import collections

import pytest

from device_code import code_objects, instructions, kernels


@pytest.fixture(scope="module")
def objects(tmp_path_factory):
    from xeno_rt_amd.ops import build
    paths = code_objects(build.find_library() or build.build(), tmp_path_factory.mktemp("code"))
    return [(path, kernels(path)) for path in paths]


# min() and max() of an int and a long are the double's in device code: row and column numbers then go through float64, exact but for some hundred instructions a kernel.
def test_products_have_no_double_precision(objects):
    products = [path for path, names in objects if any("gemm_mfma_kernel" in name for name in names)]
    assert len(products) == 1
    doubles, seen = collections.Counter(), set()
    for kernel, instruction in instructions(products[0]):
        seen.add(kernel)
        if "f64" in instruction:
            doubles[kernel] += 1
    assert sum("gemm_mfma_kernel" in (name or "") for name in seen) > 10
    assert not doubles, doubles.most_common(5)


# 512 registers a SIMD lane: up to 96 leave room for five wavefronts, up to 64 for eight.
def test_the_kernel_that_adds_parts_of_q_k_v_leaves_room_for_other_wavefronts(objects):
    of_parts = {name: fields for _, names in objects for name, fields in names.items() if "qkv_prepare_vector_kernel" in name and "Li0E" not in name}
    assert len(of_parts) > 10
    for name, fields in of_parts.items():
        assert fields["vgpr_count"] <= (64 if "Li2EEE" in name else 96), name
        assert fields["vgpr_spill_count"] == 0 and fields["private_segment_fixed_size"] == 0, name
