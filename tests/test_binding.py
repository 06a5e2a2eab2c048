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


@pytest.mark.parametrize("last", [2**32 + 16, 2**31, -2**31 - 1, 2**70])
def test_row_offsets_that_32_bits_do_not_hold_are_refused(native, last):
    """2^32 + 16 used to count as 16, the number of rows, and went on to the device check."""
    x = torch.zeros((16, 128))
    with pytest.raises(ValueError, match="32 bits"):
        native.quantize_a_grouped(x, [0, last])
    with pytest.raises(ValueError, match="on the GPU"):
        native.quantize_a_grouped(x, torch.tensor([0, 16]))           # anything int() takes


def test_a_module_built_for_another_torch_says_how_to_build_it_again(tmp_path, monkeypatch):
    """A library with a symbol that this PyTorch does not have, as one built against another version would be."""
    import subprocess
    from radeonflow_kernels_amd import gemm
    src, so = tmp_path / "m.cpp", str(tmp_path / "_torch_binding.so")
    src.write_text('extern "C" int no_such_torch_symbol(); extern "C" void *PyInit__torch_binding() '
                   '{ return no_such_torch_symbol() ? nullptr : nullptr; }')
    subprocess.run(["g++", "-shared", "-fPIC", "-Wl,-z,now", "-o", so, str(src)], check=True)
    monkeypatch.setattr(gemm, "BINDING_PATH", so)
    with pytest.raises(RuntimeError, match="radeonflow_kernels_amd.build.*no_such_torch_symbol"):
        gemm._Binding().fp8_mm()
