"""Quantisers and dequantisers at the edges of their tiles, byte for byte against the oracle."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle as O
from mojo_amd import QuantizationConfig, QuantizationEncoding as QE, _lib, dequantize, qmatmul_rmsnorm, quantize, quantize_gptq

pytestmark = pytest.mark.gpu
ORACLE = {QE.Q4_0: O.Q4_0, QE.Q4_K: O.Q4_K, QE.Q5_K: O.Q5_K, QE.Q6_K: O.Q6_K}


def weights(seed, n, k):
    """Normal values with zero blocks, and runs of equal magnitude and either sign (the first extreme of a block decides its scale)."""
    rng = np.random.Generator(np.random.PCG64(seed))
    w = (0.02 * rng.standard_normal((n, k), dtype=np.float32)).astype(np.float32)
    flat = w.reshape(-1)
    flat[: flat.size // 4 // 256 * 256] = 0.0 if seed % 2 else flat[: flat.size // 4 // 256 * 256]
    tied = flat[flat.size // 2 :]
    tied[:] = np.round(tied * 50) * np.float32(0.02)
    return w


def bits(t):
    return t.cpu().view(torch.int32 if t.dtype == torch.float32 else torch.int16).numpy()


@pytest.mark.parametrize("enc", list(ORACLE))
@pytest.mark.parametrize("n,blocks", [(1, 1), (1, 3), (3, 5), (17, 4), (33, 9), (515, 37)])
def test_gguf_edges(enc, n, blocks):
    k = blocks * enc.block_parameters.elements_per_block  # (Q4_0: pieces of eight blocks with a remainder)
    w = weights(n + blocks, n, k)
    packed = O.quantize(ORACLE[enc], w)
    assert np.array_equal(quantize(enc, torch.from_numpy(w).cuda()).cpu().numpy(), packed)
    want = O.dequantize(ORACLE[enc], packed, k)
    assert np.array_equal(bits(dequantize(enc, torch.from_numpy(packed).cuda())), want.view(np.int32))
    assert np.array_equal(bits(dequantize(enc, torch.from_numpy(packed).cuda(), dtype=torch.bfloat16)), O.f32_to_bf16(want).view(np.int16))


@pytest.mark.parametrize("enc", [QE.Q4_K, QE.Q5_K, QE.Q6_K])
@pytest.mark.parametrize("scale", [1e-30, 1e-9, 1e-4, 1.0, 1e3, 1e5])
def test_codes_of_any_magnitude(enc, scale):
    """Quotients by one reciprocal per sub-block: rounded as divisions are, halves between codes among them, and with scales that are denormal or zero in fp16."""
    rng = np.random.Generator(np.random.PCG64(11))
    w = rng.standard_normal((256, 1024), dtype=np.float32)
    w[::2] = np.round(w[::2] * 6) / np.float32(6) + np.float32(1 / 12)  # few different values, so many quotients of a block that are equal or lie half way
    w[1::4, ::3] *= np.float32(1e-3)
    w = (w * np.float32(scale)).astype(np.float32)
    assert np.array_equal(quantize(enc, torch.from_numpy(w).cuda()).cpu().numpy(), O.quantize(ORACLE[enc], w))


@pytest.mark.parametrize("n,k,group", [(8, 32, 32), (72, 96, 96), (64, 512, 128), (56, 640, 160), (200, 1024, 1024), (8, 416, 32)])
def test_gptq_edges(n, k, group):
    w = weights(n + k, n, k)
    got = [t.cpu().numpy() for t in quantize_gptq(torch.from_numpy(w).cuda(), QuantizationConfig("gptq", 4, group, False, True))]
    want = O.quantize_gptq(w, group)
    for a, b in zip(got, want):
        assert np.array_equal(a.view(np.uint16) if a.dtype == np.float16 else a, b)
    qw, sc, qz, _ = want
    order = np.random.Generator(np.random.PCG64(k)).integers(0, k // group, k).astype(np.int32)
    tensors = [torch.from_numpy(qw).cuda(), torch.from_numpy(sc.view(np.float16)).cuda(), torch.from_numpy(qz).cuda()]
    for g_idx in (None, order):
        config = QuantizationConfig("gptq", 4, group, g_idx is not None, True)
        rhs = tensors + ([torch.from_numpy(g_idx).cuda()] if g_idx is not None else [])
        plain = O.dequantize_gptq(qw, sc, qz, group, g_idx)
        assert np.array_equal(bits(dequantize(QE.GPTQ, *rhs, config=config)), plain.view(np.int32))
        assert np.array_equal(bits(dequantize(QE.GPTQ, *rhs, config=config, dtype=torch.bfloat16)), O.f32_to_bf16(plain).view(np.int16))


@pytest.mark.parametrize("enc", list(ORACLE))
@pytest.mark.parametrize("n", [4, 15, 16, 17, 31, 32, 33, 65])  # a workgroup's 4096 (fp32) or 8192 (bf16) elements, with and without a rest
def test_dequantised_workgroups_with_and_without_a_rest(enc, n):
    """Block scales that are infinite or no number beside finite ones: a bf16 NaN is 0x7fc0, with either sign."""
    k = 256
    packed = O.quantize(ORACLE[enc], weights(n, n, k))
    blocks = packed.reshape(-1, O.BLOCK[ORACLE[enc]][1])
    at = 208 if enc == QE.Q6_K else 0
    for block, scale in ((1, 0x7C00), (2, 0x7E01), (len(blocks) - 1, 0xFC00)):
        blocks[block, at : at + 2] = [scale & 255, scale >> 8]
    want = O.dequantize(ORACLE[enc], packed, k)
    got = dequantize(enc, torch.from_numpy(packed).cuda())
    assert np.array_equal(np.isnan(want), got.isnan().cpu().numpy()) and np.isnan(want).any()
    assert np.array_equal(bits(got)[~np.isnan(want)], want.view(np.int32)[~np.isnan(want)])
    got = bits(dequantize(enc, torch.from_numpy(packed).cuda(), dtype=torch.bfloat16))
    assert np.array_equal(got[~np.isnan(want)], O.f32_to_bf16(want).view(np.int16)[~np.isnan(want)])
    assert (got[np.isnan(want)] & 0x7FFF == 0x7FC0).all()


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k", [32, 256, 288, 4096, 4128, 8192, 8224, 16384, 16416, 33056])  # a thread's 16, 32 and 64 values, and rows longer than those
def test_rms_normalised_rows_of_every_length(k, lhs):
    gen = torch.Generator(device="cuda").manual_seed(k)
    config = QuantizationConfig("gptq", 4, 32, False, True)
    rhs = quantize_gptq(torch.randn((40, k), device="cuda", generator=gen) * 0.02, config)[:3]
    x = (torch.randn((3, k), device="cuda", generator=gen) * torch.tensor([[1.0], [1e-3], [300.0]], device="cuda")).to(lhs)
    gamma = torch.rand(k, device="cuda", generator=gen) + 0.5
    y = x.double() / (x.double().square().mean(dim=1, keepdim=True) + 1e-5).sqrt() * gamma.double()
    w = dequantize(QE.GPTQ, *rhs, config=config).double()
    want, size = y @ w.T, y.abs() @ w.abs().T
    # The sum of squares: K / 256 additions one after the other and ten more, half of their error behind the square root, five roundings; bf16 rows are rounded once more.  The product: K / 16 additions and 32 on
    # products of up to sixteen times their size.
    bound = ((k / 512 + 10) * 2.0**-24 + (2.0**-8 if lhs == torch.bfloat16 else 0.0) + (k / 16 + 32) * 2.0**-24 * 16) * size
    assert ((qmatmul_rmsnorm(QE.GPTQ, config, x, gamma, 1e-5, *rhs).double() - want).abs() <= bound).all()


@pytest.mark.parametrize("m,n,k", [(300, 33, 256), (301, 65, 512), (300, 8, 256), (67, 3, 288)])
@pytest.mark.parametrize("offset", [0, 1, 4, 8])  # of the results, in values: 16-byte aligned or not
def test_bf16_results_anywhere(m, n, k, offset):
    gen = torch.Generator(device="cuda").manual_seed(m)
    packed = quantize(QE.Q4_0, torch.randn((n, k), device="cuda", generator=gen))
    a = torch.randn((m, k), device="cuda", generator=gen)
    lib = _lib.load()
    need = max(lib.qmm_preferred_workspace_bytes(_lib.QMM_OP_MATMUL, QE.Q4_0.code, None, _lib.QMM_F32, m, n, k, flags) for flags in (0, _lib.QMM_FLAG_OUT_BF16))
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device="cuda")
    want, got = torch.empty((m, n), device="cuda"), torch.zeros(m * n + 16, dtype=torch.bfloat16, device="cuda")
    for out, flags in ((want, 0), (got[offset:], _lib.QMM_FLAG_OUT_BF16)):
        assert lib.qmm_matmul(QE.Q4_0.code, None, a.data_ptr(), _lib.QMM_F32, m, k, (C.c_void_p * 1)(packed.data_ptr()), 1, n, out.data_ptr(), ws.data_ptr(), ws.numel(), flags,
                              torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(got[offset : offset + m * n].view(m, n), want.bfloat16())
    assert not got[:offset].any() and not got[offset + m * n :].any()


@pytest.mark.parametrize("n", [1, 7, 9, 33, 2047, 4101])
@pytest.mark.parametrize("offset", [0, 1, 2, 5, 8])  # of the results, in values
def test_results_narrowed_by_a_launch_of_their_own(n, offset):
    """One row of Q6_K with an odd number of blocks in all, which no kernel that stores bf16 itself serves: the decode kernel's fp32 results and the launch behind it, whose eights leave n mod 8 values."""
    k = 768
    packed = quantize(QE.Q6_K, torch.randn((n, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(n)))
    a = torch.randn((1, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(k))
    lib = _lib.load()
    need = [lib.qmm_preferred_workspace_bytes(_lib.QMM_OP_MATMUL, QE.Q6_K.code, None, _lib.QMM_F32, 1, n, k, flags) for flags in (0, _lib.QMM_FLAG_OUT_BF16)]
    assert need[1] >= need[0] + 4 * n  # (the fp32 results lie there)
    ws = torch.empty(need[1], dtype=torch.uint8, device="cuda")
    want, got = torch.empty(n, device="cuda"), torch.zeros(n + 16, dtype=torch.bfloat16, device="cuda")
    for out, flags in ((want, 0), (got[offset:], _lib.QMM_FLAG_OUT_BF16)):
        assert lib.qmm_matmul(QE.Q6_K.code, None, a.data_ptr(), _lib.QMM_F32, 1, k, (C.c_void_p * 1)(packed.data_ptr()), 1, n, out.data_ptr(), ws.data_ptr(), ws.numel(), flags,
                              torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(got[offset : offset + n], want.bfloat16())
    assert not got[:offset].any() and not got[offset + n :].any()


@pytest.mark.parametrize("offset", [0, 1])
def test_narrowed_values_of_every_exponent(offset):
    """Ties and their neighbours at every exponent of fp32, subnormal numbers, the largest, infinities and NaNs: one value a row, times one, through the act-order look-up kernel (whose products and
    sums are exact here) and the launch that narrows, over more results than its grid has lanes."""
    k, n = 32, 1464
    high, low = torch.tensor([0, 1, 0x7E, 0x7F]) << 16, torch.tensor([0, 1, 0x7FFF, 0x8000, 0x8001, 0xFFFF])
    values = ((torch.arange(255) << 23)[:, None, None] + high[:, None] + low).flatten()
    values = torch.cat([values, torch.tensor([0x7F800000, 0x7F800001, 0x7FC00000, 0x7FFFFFFF])])
    values = torch.cat([values[values > 0], -0x80000000 + values[values > 0]]).int().view(torch.float32).cuda()
    m = len(values)
    assert m * n > 8 * 256 * 8192
    a = torch.zeros((m, k), device="cuda")
    a[torch.arange(m), torch.arange(m) % k] = values
    rhs = (torch.full((k // 8, n), 0x22222222, dtype=torch.int32, device="cuda"), torch.ones((1, n), dtype=torch.float16, device="cuda"), torch.zeros((1, n // 8), dtype=torch.int32, device="cuda"),
           torch.zeros(k, dtype=torch.int32, device="cuda"))  # codes 2, zero point 1
    lib, cfg = _lib.load(), _lib.GptqConfig(4, 32, 1, 1)
    need = lib.qmm_matmul_workspace_bytes_flags(QE.GPTQ.code, _lib.QMM_F32, m, n, k, _lib.QMM_FLAG_OUT_BF16)
    assert 4 * m * n <= need < lib.qmm_preferred_workspace_bytes(_lib.QMM_OP_MATMUL, QE.GPTQ.code, C.byref(cfg), _lib.QMM_F32, m, n, k, _lib.QMM_FLAG_OUT_BF16)  # (no room for sorted columns)
    ws, got = torch.empty(need, dtype=torch.uint8, device="cuda"), torch.zeros(m * n + offset, dtype=torch.bfloat16, device="cuda")
    assert lib.qmm_matmul(QE.GPTQ.code, C.byref(cfg), a.data_ptr(), _lib.QMM_F32, m, k, (C.c_void_p * 4)(*[t.data_ptr() for t in rhs]), 4, n, got[offset:].data_ptr(), ws.data_ptr(), need,
                          _lib.QMM_FLAG_OUT_BF16, torch.cuda.current_stream().cuda_stream) == 0
    got = got[offset:].view(m, n).view(torch.int16)
    assert torch.equal(got, got[:, :1].expand(m, n))
    got, want, x = got[:, 0].cpu().numpy(), O.f32_to_bf16(values.cpu().numpy()).view(np.int16), values.cpu().numpy()
    assert np.array_equal(got[~np.isnan(x)], want[~np.isnan(x)])
    assert (got[np.isnan(x)] & 0x7FFF == 0x7FC0).all()


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k", [32, 256, 288, 1024, 1056, 4096, 4128, 8192, 8224, 16384, 16416, 33056])
@pytest.mark.parametrize("place", [0, 1, 2])  # the first values of a row, some in its middle, the last
def test_rms_of_rows_that_32_values_decide(k, place, lhs):
    """Nearly all of a row's squares in 32 values: a sum that leaves them out is wrong by a large factor, at whichever of a thread's values they are."""
    gen = torch.Generator(device="cuda").manual_seed(k)
    config = QuantizationConfig("gptq", 4, 32, False, True)
    rhs = quantize_gptq(torch.randn((40, k), device="cuda", generator=gen) * 0.02, config)[:3]
    first = (0, k // 64 * 32, k - 32)[place]
    x = torch.randn((3, k), device="cuda", generator=gen)
    x[:, first : first + 32] *= 1024
    x = x.to(lhs)
    gamma = torch.rand(k, device="cuda", generator=gen) + 0.5
    y = x.double() / (x.double().square().mean(dim=1, keepdim=True) + 1e-5).sqrt() * gamma.double()
    w = dequantize(QE.GPTQ, *rhs, config=config).double()
    want, size = y @ w.T, y.abs() @ w.abs().T
    # as above; a sum without those values would make the results larger by sqrt(32 * 2^20 / k), 31 times at the longest
    bound = ((k / 512 + 10) * 2.0**-24 + (2.0**-8 if lhs == torch.bfloat16 else 0.0) + (k / 16 + 32) * 2.0**-24 * 16) * size
    assert ((qmatmul_rmsnorm(QE.GPTQ, config, x, gamma, 1e-5, *rhs).double() - want).abs() <= bound).all()
