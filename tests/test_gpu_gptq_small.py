"""GPTQ with 1 .. 16 lhs rows: the kernel for few rows at the edges of its tiles (16 or 32 columns; the last one overlaps its neighbour), of its parts of K (256, up to 16 in a
group, divided evenly), of its lhs rows (1, 2, 4, 8, 16) and with every size of group, against float64 products of the dequantised weights."""
import ctypes

import pytest
import torch

from mojo_amd import QuantizationConfig, QuantizationEncoding as QE, _lib, dequantize, qmatmul, qmatmul_rmsnorm

pytestmark = pytest.mark.gpu


def tensors(n, k, group, seed=0):
    """Random words, zeros included, and scales of ordinary size."""
    gen = torch.Generator(device="cuda").manual_seed(n + 7 * k + seed)
    words = lambda *shape: torch.randint(-(2**31), 2**31, shape, device="cuda", generator=gen, dtype=torch.int64).to(torch.int32)
    scales = torch.empty((k // group, n), device="cuda").uniform_(1e-3, 4e-3, generator=gen).half()
    return QuantizationConfig("gptq", 4, group, False, False), (words(k // 8, n), scales, words(k // group, n // 8))


def rows(m, k, lhs):
    return torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m * k)).to(lhs)


def check(config, rhs, got, a, bits=22):
    want = a.double() @ dequantize(QE.GPTQ, *rhs, config=config).double().T
    # fp32 rows as two fp16 terms (2^-23 of a value), exact products, fp32 sums (some 2^-24 of their terms each, which add up like a random walk): 0.6e-7 .. 1.1e-7 of a row's
    # norm, held to 2^-22 = 2.4e-7.  bits: 8 for results rounded to bf16.
    error = ((got.double() - want).norm(dim=1) / want.norm(dim=1)).max().item()
    assert error <= 2.0**-bits, (tuple(got.shape), a.shape[1], config.group_size, a.dtype, error)


@pytest.mark.parametrize("group", [32, 64, 128, 256])
@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(1, 16, 256), (2, 24, 512), (3, 1000, 768), (4, 14344, 4096), (1, 4104, 4352), (8, 264, 8192), (7, 4200, 11008), (16, 1000, 2560), (9, 16, 14336), (12, 8200, 4096), (16, 4112, 5120)])
def test_against_float64(group, lhs, m, n, k):
    config, rhs = tensors(n, k, group)
    a = rows(min(m, 8) if lhs == torch.float32 else m, k, lhs)
    check(config, rhs, qmatmul(QE.GPTQ, config, a, *rhs), a)
    check(config, rhs, qmatmul(QE.GPTQ, config, a, *rhs, out_dtype=torch.bfloat16), a, bits=8)


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("scale", [1e-36, 1e-5, 3e4, 1e30])
def test_rows_of_other_magnitudes(lhs, scale):
    """Rows that are brought to fp16's range by a power of two, next to rows that need none and to one of zeros."""
    config, rhs = tensors(136, 4608, 128)
    a = rows(8, 4608, torch.float32)
    a[1::3] *= scale
    a[5] = 0.0
    a = a.to(lhs)
    got = qmatmul(QE.GPTQ, config, a, *rhs)
    assert (got[5] == 0).all()
    keep = [0, 1, 2, 3, 4, 6, 7]
    check(config, rhs, got[keep], a[keep])


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
def test_infinities_and_nans_keep_their_kind(lhs):
    config, rhs = tensors(64, 1024, 128)
    a = rows(4, 1024, lhs)
    a[1, 300], a[2, 5], a[3, 1000] = float("inf"), float("nan"), float("-inf")
    a[1, 299] = 1e5  # (finite next to an infinity)
    got, w = qmatmul(QE.GPTQ, config, a, *rhs), dequantize(QE.GPTQ, *rhs, config=config)
    check(config, rhs, got[:1], a[:1])
    assert got[2].isnan().all()
    for row, column, sign in ((1, 300, 1.0), (3, 1000, -1.0)):
        assert torch.equal(got[row].nan_to_num(nan=0.0, posinf=1.0, neginf=-1.0), sign * w[:, column].sign())


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
def test_small_values_next_to_a_few_large_ones(lhs):
    """Spikes of 0.2 among values of 2^-13: what a row is scaled by decides how much of those fp16 holds."""
    config, rhs = tensors(264, 4096, 128)
    a = rows(4, 4096, torch.float32) * 2.0**-13
    a[:, 5::1024] = 0.2
    # (roundings of a few large terms do not average out: 2^-21; with the small values held to 2^-25, however large the spikes are, 1.4e-6 and, bf16 with 2^-17, 1.3e-6)
    check(config, rhs, qmatmul(QE.GPTQ, config, a.to(lhs), *rhs), a.to(lhs), bits=21)
    a[:, torch.arange(4096, device="cuda") % 1024 != 5] *= 2.0**-4
    check(config, rhs, qmatmul(QE.GPTQ, config, a.to(lhs), *rhs), a.to(lhs), bits=21)
    # rows up to 7.9 times smaller than the largest, which fp32 rows share one power of two with: 2^-31 (GPTQ 2^-36) of a row's largest left out of each value, 2^-25 of all
    a *= torch.linspace(1.0, 1.0 / 7.9, a.shape[0], device="cuda")[:, None]
    check(config, rhs, qmatmul(QE.GPTQ, config, a.to(lhs), *rhs), a.to(lhs), bits=21)


@pytest.mark.parametrize("m", [1, 4, 8])
def test_a_small_workspace_gives_the_same_sums(m):
    """Groups of K side by side, added by a launch of their own, or, with less than they need, one after the other in each workgroup."""
    lib = _lib.load()
    n, k = 2056, 11008
    config, rhs = tensors(n, k, 128)
    a, out = rows(m, k, torch.bfloat16), torch.empty((m, n), device="cuda")
    want = qmatmul(QE.GPTQ, config, a, *rhs)
    cfg, ptrs = _lib.GptqConfig(4, 128, 0, 0), (ctypes.c_void_p * 3)(*(t.data_ptr() for t in rhs))
    assert lib.qmm_preferred_workspace_bytes(0, 3, ctypes.byref(cfg), 1, m, n, k, 0) >= 4 * 4 * m * n  # four groups of K, [m, n] fp32 each
    ws = torch.empty(3 * 4 * m * n, dtype=torch.uint8, device="cuda")
    assert lib.qmm_matmul(3, ctypes.byref(cfg), a.data_ptr(), 1, m, k, ptrs, 3, n, out.data_ptr(), ws.data_ptr(), ws.numel(), 0, torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(out, want)


def test_rmsnorm_in_front():
    config, rhs = tensors(520, 2048, 64)
    a, gamma = rows(3, 2048, torch.float32), 1.0 + 0.1 * torch.randn(2048, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    normal = a * torch.rsqrt((a.double() ** 2).mean(dim=1, keepdim=True) + 1e-5).float() * gamma
    check(config, rhs, qmatmul_rmsnorm(QE.GPTQ, config, a, gamma, 1e-5, *rhs), normal, bits=21)  # (and the normalisation's rounding)


@pytest.mark.parametrize("m,n,k", [(8, 8200, 8192), (24, 2048, 8192)])
def test_tiles_that_leave_lds_one_by_one(m, n, k):
    """fp32 rows, groups of K side by side, results of one tile in LDS at a time: the operands of the group serve every tile of the workgroup."""
    config, rhs = tensors(n, k, 128)
    a = rows(m, k, torch.float32)
    check(config, rhs, qmatmul(QE.GPTQ, config, a, *rhs), a)
