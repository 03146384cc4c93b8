"""The native entry functions (``mojo_amd._call``) serve the plain calls, with the results of the Python path behind them, and decline the rest."""
import pytest
import torch

from mojo_amd import QuantizationConfig, QuantizationEncoding as QE, _lib, dequantize, qmatmul, quantize, quantize_gptq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("enc", ["Q4_0", "Q4_K", "Q5_K", "Q6_K", "GPTQ"])
@pytest.mark.parametrize("lead", [(), (1,), (2, 3), (20,)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_native_call_serves_and_equals_the_python_path(enc, lead, out_dtype):
    n, k = 264, 512
    gen = torch.Generator(device="cuda").manual_seed(len(lead))
    w = torch.empty((n, k), device="cuda").normal_(0, 0.02, generator=gen)
    a = torch.empty((*lead, k), device="cuda").normal_(generator=gen)
    config = QuantizationConfig() if enc == "GPTQ" else None
    rhs = tuple(quantize_gptq(w, config)[:3]) if enc == "GPTQ" else (quantize(QE[enc], w),)
    native = _lib.call().matmul(QE[enc], config, a, rhs, 0, out_dtype)
    assert native is not None and native.shape == (*lead, n) and native.dtype == out_dtype
    out = torch.empty((a.numel() // k, n), dtype=out_dtype, device="cuda")
    assert torch.equal(native, qmatmul(QE[enc], config, a, *rhs, out=out, out_dtype=out_dtype))  # (out= goes through Python)


def test_native_call_declines_what_is_not_plain():
    call = _lib.call().matmul
    w = quantize(QE.Q4_K, torch.randn(8, 256, device="cuda"))
    a = torch.randn(2, 256, device="cuda")
    for enc, config, lhs, rhs in ((QE.Q8_0, None, a, (w,)), (QE.Q6_K, None, a, (w,)), ("Q4_K", None, a, (w,)), (QE.Q4_K, None, a.half(), (w,)),
                                  (QE.Q4_K, None, a.t(), (w,)), (QE.Q4_K, None, a.cpu(), (w,)), (QE.Q4_K, None, a, (w, w)), (QE.Q4_K, None, a, [w]),
                                  (QE.Q4_K, None, a[:, :128].contiguous(), (w,)), (QE.Q4_K, None, a[:0], (w,)), (QE.GPTQ, None, a, (w, w, w))):
        assert call(enc, config, lhs, rhs, 0, torch.float32) is None
    assert call(QE.Q4_K, None, a, (w,), 0, torch.float16) is None
    assert _lib.call().dequantize(QE.Q4_K, None, (w[:, :100].contiguous(),), torch.float32) is None
    with pytest.raises(ValueError, match="K=128"):
        qmatmul(QE.Q4_K, None, a[:, :128].contiguous(), w)
    assert dequantize(QE.Q4_K, w, k=256).shape == (8, 256)


def test_without_the_module_the_kernels_are_the_same(monkeypatch):
    w = quantize(QE.Q4_K, torch.randn(264, 512, device="cuda"))
    a = torch.randn(3, 512, device="cuda")
    want = qmatmul(QE.Q4_K, None, a, w), dequantize(QE.Q4_K, w)
    monkeypatch.setattr(_lib, "_call", _lib._Declines())
    assert torch.equal(want[0], qmatmul(QE.Q4_K, None, a, w)) and torch.equal(want[1], dequantize(QE.Q4_K, w))
