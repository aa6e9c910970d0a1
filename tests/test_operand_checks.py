"""What the wrappers of products with fused ends refuse before anything is launched: a kernel takes addresses as they come, so an operand
in host memory or a cache that is too short must not reach it.  The native module is replaced, so nothing here needs or touches a GPU."""
import pytest
import torch

from atoma_infer_amd.kernels import ops

NH, NKV, HD, K, PAGE = 4, 2, 16, 64, 16


class OnDevice(torch.Tensor):
    """A host tensor that says that it is on the device."""
    is_cuda = property(lambda self: True)


@pytest.fixture
def launched(monkeypatch):
    names = []

    class Native:
        def __getattr__(self, name):
            def call(*_):
                if name != "atoma_gemm_few_takes":
                    names.append(name)
                return 1 if name == "atoma_gemm_few_takes" else 0
            return call

    monkeypatch.setattr(ops, "core", Native)
    monkeypatch.setattr(ops, "_stream", lambda: None)
    return names


def there(*shape, dtype=torch.float32):
    return torch.zeros(*shape, dtype=dtype).as_subclass(OnDevice)


def rotated_operands():
    w = there((NH + 2 * NKV) * HD, K, dtype=torch.bfloat16)
    return {"a": there(3, K), "w": w, "positions": there(3, dtype=torch.int32), "cos": there(9, HD // 2), "sin": there(9, HD // 2),
            "kcache": there(5, NKV, PAGE * HD), "vcache": there(5, NKV, PAGE * HD), "slot_mapping": there(3, dtype=torch.int32)}


@pytest.mark.parametrize("host", ["a", "w"])
def test_few_rows_that_end_in_the_activation_are_device_tensors(launched, host):
    operands = {"a": there(3, K), "w": there(128, K, dtype=torch.bfloat16)}
    assert ops.gemm_few_gated(**operands) is not None and launched == ["atoma_gemm_few_gated"]
    operands[host] = operands[host].as_subclass(torch.Tensor)
    with pytest.raises(ops.KernelError, match="device tensors only"):
        ops.gemm_few_gated(**operands)
    assert len(launched) == 1


@pytest.mark.parametrize("host", ["a", "w", "positions", "cos", "sin", "kcache", "vcache", "slot_mapping"])
def test_few_rows_that_end_in_the_rotation_are_device_tensors(launched, host):
    operands = rotated_operands()
    assert ops.gemm_few_rotated(**operands, page_size=PAGE, nh=NH, nkv=NKV, hd=HD) is not None and launched == ["atoma_gemm_few_rotated"]
    operands[host] = operands[host].as_subclass(torch.Tensor)
    with pytest.raises(ops.KernelError, match="device tensors only"):
        ops.gemm_few_rotated(**operands, page_size=PAGE, nh=NH, nkv=NKV, hd=HD)
    assert len(launched) == 1


def test_few_rows_that_end_in_the_rotation_leave_caches_of_two_lengths(launched):
    """To the rotation's own kernel, whose wrapper refuses them."""
    operands = rotated_operands()
    operands["vcache"] = there(4, NKV, PAGE * HD)
    assert ops.gemm_few_rotated(**operands, page_size=PAGE, nh=NH, nkv=NKV, hd=HD) is None and not launched
    qkv = there(3, (NH + 2 * NKV) * HD)
    with pytest.raises(ops.KernelError, match="cache tensors"):
        ops.rope_cache_write(qkv, operands["positions"], operands["cos"], operands["sin"], HD, operands["kcache"], operands["vcache"],
                             operands["slot_mapping"], PAGE, NH, NKV, HD, there(3, NH * HD))
    assert not launched
