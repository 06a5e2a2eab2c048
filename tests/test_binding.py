"""CPU tests of the native module behind the Python entry points (csrc/torch_binding.cpp): what it refuses before it touches a
device."""
import pytest
import torch

COUNTS = {"check_operands": 5, "fp8_mm": 6, "fp8_mm_static": 5, "fp8_mm_grouped": 7, "fp8_mm_grouped_padded": 7, "quantize": 2,
          "quantize_a_grouped": 2}


@pytest.fixture(scope="module")
def native():
    from radeonflow_kernels_amd import gemm
    gemm._native.check_operands                          # loads the module, which takes the stand-in's place
    return gemm._native


@pytest.mark.parametrize("name,count", COUNTS.items())
def test_a_call_with_another_number_of_arguments_is_refused(native, name, count):
    x = torch.zeros((16, 128))
    for n in (0, count - 1, count + 1):
        with pytest.raises(TypeError, match="expected %d arguments, got %d" % (count, n)):
            getattr(native, name)(*[x] * n)
