"""The GEMM that reads packed weights straight into the matrix cores, at the edges of its tiles (32 or 64 rows and columns), of its units
of 256 values of K and of the ways it cuts K (4 or 8 wavefronts, one or two workgroups a tile), against float64 products of the same
integers."""
import ctypes as C

import pytest
import torch

from mojo_amd import QuantizationConfig, QuantizationEncoding as QE, _lib, dequantize, qmatmul, qmatmul_grouped, quantize, quantize_gptq

pytestmark = pytest.mark.gpu


def weights(enc, group, n, k):
    gen = torch.Generator(device="cuda").manual_seed(n + k)
    w = torch.empty((n, k), device="cuda").normal_(0.0, 0.02, generator=gen)
    if enc != QE.GPTQ:
        return None, (quantize(enc, w),)
    config = QuantizationConfig("gptq", 4, group, False, True)
    qweight, scales, qzeros, _ = quantize_gptq(w, config)
    qzeros = torch.randint(-2**31, 2**31 - 1, qzeros.shape, device="cuda", dtype=torch.int64, generator=gen).int()  # every zero point
    return config, (qweight, scales, qzeros)


def check(got, enc, config, rhs, a):
    w = dequantize(enc, *rhs, config=config).double()
    x = a.double()
    if enc == QE.Q4_0:  # (multiplies with the lhs quantised to Q8_0)
        blocks = quantize(QE.Q8_0, a.float()).view(a.shape[0], -1, 34)
        scale = blocks[:, :, :2].contiguous().view(torch.float16)
        x = (scale.double() * blocks[:, :, 2:].contiguous().view(torch.int8).double()).view(a.shape)
    want, size = x @ w.T, x.abs() @ w.abs().T
    # A lhs value is two fp16 terms (2^-22) or exact (bf16); K / 16 products enter a sum one after the other, and 32 for the parts of K.
    # A GPTQ or Q4_K product may be the difference of two terms sixteen times as large (code and zero point or minimum apart).
    bound = (a.shape[1] / 16 + 32) * 2.0**-24 * 16 * size + 1e-30
    if got.dtype == torch.bfloat16:
        bound = bound + 2.0**-8 * want.abs()
    worst = ((got.double() - want).abs() / bound).max().item()
    assert worst <= 1.0, (enc, got.shape, a.shape, worst)


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("enc,group,odd", [(QE.Q4_0, 0, 32), (QE.Q4_K, 0, 0), (QE.Q5_K, 0, 0), (QE.Q6_K, 0, 0), (QE.GPTQ, 128, 128), (QE.GPTQ, 32, 32)])
def test_edges(enc, group, odd, lhs):
    for m, n, k in ((17, 40, 256), (32, 264, 512 + odd), (17, 40, 2304 + odd), (33, 2056, 2304), (33, 4104, 4352 - odd), (65, 4104, 4352), (100, 4104, 256 + odd),
                    (200, 4104, 256), (450, 264, 1024)):
        config, rhs = weights(enc, group, n, k)
        a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).to(lhs)
        a[m // 2] *= 1e-6
        a[m - 1] = 0.0
        cfg = C.byref(_lib.GptqConfig(4, group, 0, 1)) if config else None
        lib, dtype = _lib.load(), _lib.QMM_F32 if lhs == torch.float32 else _lib.QMM_BF16
        assert lib.qmm_preferred_workspace_bytes(_lib.QMM_OP_MATMUL, enc.code, cfg, dtype, m, n, k, 0) > 0
        check(qmatmul(enc, config, a, *rhs), enc, config, rhs, a)
        check(qmatmul(enc, config, a, *rhs, out_dtype=torch.bfloat16), enc, config, rhs, a)
        # with the workspace that a caller of the C interface gives (none for some: other kernels)
        need = lib.qmm_matmul_workspace_bytes(enc.code, dtype, m, n, k)
        ws, out = torch.empty(max(need, 1), dtype=torch.uint8, device="cuda"), torch.full((m, n), float("nan"), device="cuda")
        ptrs = (C.c_void_p * len(rhs))(*[t.data_ptr() for t in rhs])
        assert lib.qmm_matmul(enc.code, cfg, a.data_ptr(), dtype, m, k, ptrs, len(rhs), n, out.data_ptr(), ws.data_ptr(), need, 0,
                              torch.cuda.current_stream().cuda_stream) == 0
        check(out, enc, config, rhs, a)


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("enc,group,odd", [(QE.Q4_0, 0, 32), (QE.Q4_K, 0, 0), (QE.Q5_K, 0, 0), (QE.Q6_K, 0, 0), (QE.GPTQ, 128, 128), (QE.GPTQ, 32, 32)])
def test_shared_lhs_edges(enc, group, odd, lhs):
    """Sizes at which the wavefronts of a workgroup share the lhs: ragged last tiles of 64 rows and of 128 and 256 columns, one and two parts of K
    (of one unit, of unequal lengths), one and two workgroups a tile."""
    for m, n, k in ((200, 14344, 2048), (200, 14344, 2304 + odd), (65, 14600, 1280), (97, 11016, 2048 + odd), (449, 4104, 2304), (500, 4104, 4352 + odd),
                    (321, 11008, 256), (130, 14344, 256 + odd)):
        config, rhs = weights(enc, group, n, k)
        a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).to(lhs)
        a[m // 2] *= 1e-6
        a[m - 1] = 0.0
        check(qmatmul(enc, config, a, *rhs), enc, config, rhs, a)
        check(qmatmul(enc, config, a, *rhs, out_dtype=torch.bfloat16), enc, config, rhs, a)


@pytest.mark.parametrize("enc", [QE.Q4_0, QE.Q4_K, QE.Q5_K, QE.Q6_K])
@pytest.mark.parametrize("m,k,ns", [(17, 768, (40, 264, 1000)), (33, 2304, (4104, 2056, 40, 1, 31)), (3, 1024, (6400, 40, 6400)), (200, 2048, (14344, 14344, 264))])
def test_group_equals_separate_calls(enc, m, k, ns):
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m))
    rhs = [weights(enc, 0, n, k)[1] for n in ns]
    for got, w in zip(qmatmul_grouped(enc, a, [w[0] for w in rhs]), rhs):
        assert torch.equal(got, qmatmul(enc, None, a, *w))
        check(got, enc, None, w, a)


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("enc,group,order", [(QE.Q4_K, 0, False), (QE.Q5_K, 0, False), (QE.Q6_K, 0, False), (QE.GPTQ, 128, False), (QE.GPTQ, 32, False),
                                             (QE.GPTQ, 128, True)])
def test_rows_of_any_magnitude(enc, group, order, lhs):
    """A row is narrowed behind a power of two of its own: rows from denormal numbers (2^-140) up to 2^120, next to each other."""
    m, n, k = 33, 264, 512
    config, rhs = weights(enc, group, n, k)
    if order:
        config, rhs = QuantizationConfig("gptq", 4, group, True, True), (*rhs, torch.arange(k, device="cuda", dtype=torch.int32) // group)
    exponents = torch.tensor([(-140, -133, -126, -125, -118, -117, -110, -101, -100, -60, 0, 60, 120)[i % 13] for i in range(m)], device="cuda")
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    a = torch.ldexp(a.double(), exponents[:, None]).to(lhs)  # (rounded to the type's denormal grid where that is coarser)
    w, x = dequantize(enc, *rhs, config=config).double(), a.double()
    want, size = x @ w.T, x.abs() @ w.abs().T
    # as in check(), and the grid of denormal results
    bound = (k / 16 + 32) * 2.0**-24 * 16 * size + 2.0**-149
    worst = ((qmatmul(enc, config, a, *rhs).double() - want).abs() / bound).amax(1)
    assert worst.max().item() <= 1.0, (enc, [(int(e), round(v, 2)) for e, v in zip(exponents, worst.tolist()) if v > 1.0])


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("group,order,m,n,k", [(g, o, *s) for g, o in ((128, False), (32, False), (128, True)) for s in ((17, 264, 512), (33, 2056, 1024),
                                                                                                                       (200, 4104, 512))] + [(128, True, 6, 264, 512)])
def test_gptq_infinities_and_nans_keep_their_kind(group, order, m, n, k, lhs):
    """code - zero is one integer, so an infinity meets no difference of sums: +-inf where the weight is not zero, NaN where it is, as in the
    product of the dequantised weights; a NaN makes its row NaN; finite neighbours in such a row (1e30) and other rows are what they are."""
    config, rhs = weights(QE.GPTQ, group, n, k)
    if order:
        config, rhs = QuantizationConfig("gptq", 4, group, True, True), (*rhs, torch.arange(k, device="cuda", dtype=torch.int32) // group)
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(4)).to(lhs)
    a[1, 7], a[3, k - 1], a[4, 5], a[5, 100], a[5, 101] = float("inf"), -float("inf"), float("nan"), float("inf"), 1e30
    got = qmatmul(QE.GPTQ, config, a, *rhs)
    w, special = dequantize(QE.GPTQ, *rhs, config=config).double().cpu(), [1, 3, 4, 5]
    want, have = a[special].double().cpu() @ w.T, got[special].double().cpu()
    assert not want.isfinite().any()
    assert torch.equal(have.isnan(), want.isnan()) and torch.equal(have.isposinf(), want.isposinf())
    rest = [i for i in range(m) if i not in special]
    check(got[rest], QE.GPTQ, config, rhs, a[rest])


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("enc", [QE.Q4_K, QE.Q5_K, QE.Q6_K])
@pytest.mark.parametrize("m,n,k", [(17, 264, 512), (33, 2056, 1024), (200, 4104, 512), (40, 264, 33024)])  # (the last one: more pieces of a row than its threads hold)
def test_k_quant_rows_with_infinities_and_nans(enc, m, n, k, lhs):
    """A row with an infinity or a NaN has no finite result; what is finite in it (1e30) scales it, and rows beside it are what they are."""
    _, rhs = weights(enc, 0, n, k)
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(4)).to(lhs)
    a[1, 7], a[3, k - 1], a[4, 5], a[5, 100], a[5, 101] = float("inf"), -float("inf"), float("nan"), float("inf"), 1e30
    a[6] = float("inf")
    a[8] = float("nan")
    special = [1, 3, 4, 5, 6, 8]
    got = qmatmul(enc, None, a, *rhs)
    assert not got[special].isfinite().any() and got[[4, 8]].isnan().all()
    rest = [i for i in range(m) if i not in special]
    check(got[rest], enc, None, rhs, a[rest])


@pytest.mark.parametrize("enc,group,lhs,m,n,k", [(QE.GPTQ, 32, torch.bfloat16, 2**23 + 40, 8, 32), (QE.Q4_K, 0, torch.float32, 6000000, 1, 256)])
def test_more_row_tiles_than_a_grid_counts_apart(enc, group, lhs, m, n, k):
    """65536 row tiles and more, which are numbered through."""
    config, rhs = weights(enc, group, n, k)
    a = torch.empty((m, k), dtype=lhs, device="cuda").normal_(generator=torch.Generator(device="cuda").manual_seed(5))
    got = qmatmul(enc, config, a, *rhs)
    for x, y in zip(got.split(2**20), a.split(2**20)):
        check(x, enc, config, rhs, y)


def test_more_q4_0_rows_than_one_slice_of_the_quantiser():
    """32768 rows and some: the grid of the lhs quantiser has a second slice (K no multiple of 256 and more results than the direct GEMM serves)."""
    m, n, k = 32768 + 41, 208, 96
    _, rhs = weights(QE.Q4_0, 0, n, k)
    for lhs in (torch.float32, torch.bfloat16):
        a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(6)).to(lhs)
        check(qmatmul(QE.Q4_0, None, a, *rhs), QE.Q4_0, None, rhs, a)


@pytest.mark.parametrize("lhs,spike", [(torch.float32, 2.0**20), (torch.bfloat16, 2.0**28)])
@pytest.mark.parametrize("group", [128, 32])
def test_values_far_below_the_largest_of_their_row(group, lhs, spike):
    """Columns with values 2^20 (2^28) times the others' that no weight multiplies (code = zero): the rest of the row has to come through."""
    m, n, k = 33, 264, 1024
    config, (qweight, scales, qzeros) = weights(QE.GPTQ, group, n, k)
    columns = torch.tensor([3, 300, 801], device="cuda")
    zero = (qzeros[columns // group].repeat_interleave(8, 1) >> (4 * (torch.arange(n, device="cuda") & 7))) & 15  # stored zero; the code is one more
    scales, qzeros = scales.clone(), qzeros.clone()
    for c, z in zip(columns.tolist(), zero):
        z = (z + 1).clamp(max=15)  # (a zero point of 16 has no code: those columns of the output are left out below)
        word = qweight[c // 8] & ~(15 << (4 * (c % 8)))
        qweight[c // 8] = word | (z << (4 * (c % 8)))
    keep = ((zero + 1) <= 15).all(0)
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(6))
    a[:, columns] = spike
    a = a.to(lhs)
    rhs = (qweight, scales, qzeros)
    w, x = dequantize(QE.GPTQ, *rhs, config=config).double()[keep], a.double()
    assert keep.sum() > 100 and not w[:, columns].any()
    want, size = x @ w.T, x.abs() @ w.abs().T
    # as in check(), but code - zero is one operand: no terms sixteen times as large; a value is held to 2^-39 of its row's largest
    bound = (k / 16 + 32) * 2.0**-24 * size + 2.0**-39 * spike * w.abs().sum(1)
    worst = ((qmatmul(QE.GPTQ, config, a, *rhs)[:, keep].double() - want).abs() / bound).max().item()
    assert worst <= 1.0, worst


@pytest.mark.parametrize("enc,lhs,k", [(QE.Q4_K, torch.float32, 2**25 + 256), (QE.Q6_K, torch.float32, 2**25 + 256), (QE.Q4_K, torch.bfloat16, 2**26 + 256)])
def test_rows_whose_operands_take_more_than_32_bits_of_address(enc, lhs, k):
    """17 rows of 2^25 (fp32) or 2^26 (bf16) columns and some: a row tile's operands pass 4 GB.  The first and the last 256 columns hold most of the product, so that it is wrong by as much as it is
    large where one takes the other's place."""
    m, n = 17, 8
    assert _lib.load().qmm_preferred_workspace_bytes(_lib.QMM_OP_MATMUL, enc.code, None, _lib.QMM_F32 if lhs == torch.float32 else _lib.QMM_BF16, m, n, k, 0) > 2**32  # (the direct GEMM's)
    gen = torch.Generator(device="cuda").manual_seed(9)
    w = quantize(enc, torch.empty((n, k), device="cuda").normal_(0.0, 0.02, generator=gen))
    a = torch.empty((m, k), device="cuda").normal_(generator=gen)
    a[:, :256] *= 2.0**12
    a[:, -256:] *= 2.0**12
    a = a.to(lhs)
    plain = dequantize(enc, w, k=k)
    want = sum(x.double() @ y.double().T for x, y in zip(a.split(2**22, 1), plain.split(2**22, 1)))
    got = qmatmul(enc, None, a, w)
    # (up to 2^15 sums of a unit one after the other: 2^-24 of what is summed up each, as a random walk below 2^-15)
    assert ((got.double() - want).norm() / want.norm()).item() < 2.0**-15


# Relative error (2-norm over all results, against float64) of quantised N(0, 0.02) weights and N(0, 1) rows.  The bounds lie a tenth above what the chains of
# rounded sums give (measured, in the comment, with what longer chains and codes around another mean gave); leaving the residual of fp32 rows out would give 1.4e-4.
PRECISION = [
    ("Q4_K", 0, "bf16", 33, 4096, 4096, 1.05e-7),  # 0.9e-7 (1.9e-7)
    ("Q4_K", 0, "f32", 33, 4096, 4096, 1.9e-7),    # 1.7e-7 (3.2e-7)
    ("Q4_K", 0, "bf16", 3, 6400, 1024, 0.95e-7),   # 0.8e-7 (2.0e-7)
    ("Q5_K", 0, "bf16", 17, 4096, 4096, 1.15e-7),  # 1.0e-7 (2.2e-7)
    ("Q5_K", 0, "bf16", 33, 5120, 5120, 1.3e-7),   # 1.15e-7 (2.2e-7)
    ("Q5_K", 0, "f32", 33, 4096, 4096, 1.95e-7),   # 1.75e-7 (3.3e-7)
    ("Q5_K", 0, "bf16", 4, 6400, 1024, 1.0e-7),    # 0.9e-7 (2.2e-7)
    ("Q5_K", 0, "f32", 3, 2056, 1280, 1.9e-7),     # 1.65e-7 (2.8e-7)
    ("Q4_K", 0, "f32", 200, 11008, 4096, 2.05e-7),  # 1.85e-7 (3.3e-7)
    ("Q5_K", 0, "f32", 100, 14336, 4096, 2.1e-7),   # 1.9e-7 (3.4e-7)
    ("Q5_K", 0, "bf16", 64, 20000, 4096, 1.1e-7),   # 1.0e-7 (2.35e-7)
    ("Q5_K", 0, "f32", 64, 20000, 4096, 1.95e-7),   # 1.77e-7 (3.4e-7)
    ("Q6_K", 0, "bf16", 64, 20000, 4096, 1.07e-7),  # 0.95e-7 (1.2e-7)
    ("Q6_K", 0, "f32", 64, 8192, 8192, 1.82e-7),    # 1.65e-7 (2.1e-7)
    ("Q6_K", 0, "bf16", 17, 4096, 4096, 1.07e-7),  # 0.97e-7 (1.17e-7)
    ("Q6_K", 0, "bf16", 33, 11008, 4096, 1.07e-7),  # 0.96e-7 (1.12e-7)
    ("Q6_K", 0, "f32", 9, 4096, 4096, 1.8e-7),     # 1.6e-7 (2.1e-7)
    ("Q6_K", 0, "f32", 33, 11008, 4096, 1.8e-7),   # 1.6e-7 (2.05e-7)
    ("Q6_K", 0, "f32", 5, 6400, 1024, 1.15e-7),    # 1.0e-7 (the direct GEMM: 1.55e-7)
    ("GPTQ", 128, "bf16", 33, 4096, 4096, 0.72e-7),  # 0.64e-7
    ("GPTQ", 128, "f32", 33, 4096, 4096, 1.35e-7),   # 1.22e-7
    ("GPTQ", 32, "bf16", 300, 11008, 4096, 1.0e-7),  # 0.9e-7 (one chain over K: 2.0e-7)
    ("GPTQ", 32, "bf16", 100, 5120, 5120, 1.1e-7),   # 1.0e-7 (1.2e-7)
    ("Q4_0", 0, "bf16", 700, 5120, 5120, 1.4e-7),    # 1.0e-7 (2.3e-7)
]


@pytest.mark.parametrize("enc,group,lhs,m,n,k,limit", PRECISION)
def test_precision(enc, group, lhs, m, n, k, limit):
    enc, gen = QE[enc], torch.Generator(device="cuda").manual_seed(n + k + m)
    w = torch.empty((n, k), device="cuda").normal_(0.0, 0.02, generator=gen)
    a = torch.randn((m, k), device="cuda", generator=gen).to(torch.float32 if lhs == "f32" else torch.bfloat16)
    config = QuantizationConfig("gptq", 4, group, False, True) if enc == QE.GPTQ else None
    rhs = quantize_gptq(w, config)[:3] if config else (quantize(enc, w),)
    x = a.double()
    if enc == QE.Q4_0:
        blocks = quantize(QE.Q8_0, a.float()).view(m, -1, 34)
        x = (blocks[:, :, :2].contiguous().view(torch.float16).double() * blocks[:, :, 2:].contiguous().view(torch.int8).double()).view(m, k)
    want = x @ dequantize(enc, *rhs, config=config).double().T
    error = ((qmatmul(enc, config, a, *rhs).double() - want).norm() / want.norm()).item()
    assert error <= limit, (enc, lhs, m, n, k, error)


@pytest.mark.parametrize("enc", ["Q4_K", "Q5_K"])
@pytest.mark.parametrize("lhs", ["bf16", "f32"])
@pytest.mark.parametrize("m,n", [(40, 6200), (64, 20000), (200, 6200)])
def test_scales_of_any_size(enc, lhs, m, n):
    """The offsets of the sub-blocks are two fp16 terms in units of a power of two that suits the larger of the block's two scales: any pair of them, zeros
    and negative ones among them."""
    enc, k = QE[enc], 512
    gen = torch.Generator(device="cuda").manual_seed(n + m)
    w = quantize(enc, torch.empty((n, k), device="cuda").normal_(0.0, 0.02, generator=gen))
    scales = w.view(n, k // 256, -1)[:, :, :4].contiguous().view(torch.float16)
    kinds = torch.tensor([0.0, 2.0**-24, -3 * 2.0**-20, 0.02, -1.0, 700.0, -1000.0], device="cuda").half()
    scales.copy_(kinds[torch.randint(len(kinds), scales.shape, device="cuda", generator=gen)])
    w.view(n, k // 256, -1)[:, :, :4] = scales.view(torch.uint8).view(n, k // 256, 4)
    a = torch.randn((m, k), device="cuda", generator=gen).to(torch.float32 if lhs == "f32" else torch.bfloat16)
    out, x = qmatmul(enc, None, a, w).double(), a.double()
    # d sc q and dmin mn apart: with the other scale zero
    no_min, no_d = w.clone(), w.clone()
    no_min.view(n, k // 256, -1)[:, :, 2:4] = 0
    no_d.view(n, k // 256, -1)[:, :, :2] = 0
    parts = [dequantize(enc, t).double() for t in (no_min, no_d)]
    size = x.abs() @ (parts[0].abs() + parts[1].abs()).T
    # 32 roundings of a chain and 22 bits of an operand, all in one direction; the mean of the codes (half their range) doubles what the sums hold
    assert ((out - x @ (parts[0] + parts[1]).T).abs() <= 2.0**-24 * 2 * (32 + 4) * size).all()
