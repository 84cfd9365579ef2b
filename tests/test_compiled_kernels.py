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
