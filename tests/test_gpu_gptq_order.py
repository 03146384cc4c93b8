"""Act-order GPTQ with several lhs rows (columns sorted by group, then the kernels for plain groups): edges of the sort (K / 16 columns per
wavefront, groups of 32 .. K), of the column slabs (8, 16, 32), of the row counts at which the plain kernels change, groups of uneven
size (served by the look-up kernel), workspaces with and without room for the sorted matrix; against float64 products."""
import ctypes as C

import pytest
import torch

from mojo_amd import QuantizationConfig, QuantizationEncoding as QE, _lib, dequantize, qmatmul, quantize_gptq

pytestmark = pytest.mark.gpu


def act_order(n, k, group, seed, any_codes=True):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    w = torch.empty((n, k), device="cuda").normal_(0.0, 0.02, generator=gen)
    qweight, scales, qzeros, g_idx = quantize_gptq(w, QuantizationConfig("gptq", 4, group, False, True))
    if any_codes:
        qweight = torch.randint(-2**31, 2**31 - 1, qweight.shape, device="cuda", dtype=torch.int64, generator=gen).int()
        qzeros = torch.randint(-2**31, 2**31 - 1, qzeros.shape, device="cuda", dtype=torch.int64, generator=gen).int()
    return QuantizationConfig("gptq", 4, group, True, True), (qweight, scales, qzeros, g_idx[torch.randperm(k, device="cuda", generator=gen)].contiguous())


def check(got, config, rhs, a, sorted_columns=False):
    w = dequantize(QE.GPTQ, *rhs, config=config).double()
    x = a.double()
    want, size = x @ w.T, x.abs() @ w.abs().T
    # A weight is exact (code and zero point apart: a product of up to sixteen times its size), a lhs value two fp16 terms (2^-22) or exact; the
    # look-up kernel adds K / 16 products one after the other and sixteen sums, the others K / 16 products and 32 sums.
    bound = (a.shape[1] / 16 + 32) * 2.0**-24 * 16 * size + 1e-30
    if got.dtype == torch.bfloat16:
        bound = bound + 2.0**-8 * want.abs()
    worst = ((got.double() - want).abs() / bound).max().item()
    assert worst <= 1.0, (got.shape, a.shape, worst)
    if got.dtype == torch.float32 and sorted_columns:
        # Over all results the roundings average out: eight matrix-core sums of a group one after the other, K / 128 groups (K / 32 of the
        # smallest) and eight parts of K, each off by 2^-24 / sqrt(3) of the sum so far; an fp32 lhs value by 2^-23 / sqrt(3).
        chain = 16 + a.shape[1] / min(config.group_size, 128)
        rms = ((got.double() - want).norm() / ((x * x) @ (w * w).T).sqrt().norm()).item()
        assert rms <= (2.0**-24 * chain**0.5 + (2.0**-23 if a.dtype == torch.float32 else 0)) / 3**0.5, (got.shape, a.shape, rms)


def c_call(config, rhs, a, need):
    """The C entry point with a workspace of `need` bytes."""
    m, (k, n) = a.shape[0], (a.shape[1], rhs[0].shape[1])
    ws, out = torch.empty(max(need, 1), dtype=torch.uint8, device="cuda"), torch.full((m, n), float("nan"), device="cuda")
    ptrs = (C.c_void_p * 4)(*[t.data_ptr() for t in rhs])
    cfg = C.byref(_lib.GptqConfig(4, config.group_size, 1, 1))
    assert _lib.load().qmm_matmul(QE.GPTQ.code, cfg, a.data_ptr(), _lib.QMM_F32 if a.dtype == torch.float32 else _lib.QMM_BF16, m, k, ptrs, 4, n, out.data_ptr(),
                                  ws.data_ptr(), need, 0, torch.cuda.current_stream().cuda_stream) == 0
    return out


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k,group", [(3, 72, 256, 32), (5, 8, 32, 32), (6, 40, 1056, 32), (17, 264, 1024, 1024), (16, 136, 5120, 128), (33, 136, 5376, 256),
                                         (9, 72, 10240, 128), (20, 40, 10496, 64), (20, 24, 32768, 32), (130, 1032, 2304, 128), (600, 4104, 512, 128),
                                         (40, 72, 256, 32), (40, 8, 32, 32), (40, 40, 1056, 32), (1, 40, 14336, 32), (2, 72, 10240, 128), (4, 72, 10240, 128)])
def test_edges(m, n, k, group, lhs):
    config, rhs = act_order(n, k, group, m)
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).to(lhs)
    cfg, dtype = C.byref(_lib.GptqConfig(4, group, 1, 1)), _lib.QMM_F32 if lhs == torch.float32 else _lib.QMM_BF16
    room = _lib.load().qmm_preferred_workspace_bytes(_lib.QMM_OP_MATMUL, QE.GPTQ.code, cfg, dtype, m, n, k, 0)
    sorted_columns = room > n * k // 2  # (room for the sorted matrix)
    assert sorted_columns or m < 20
    check(qmatmul(QE.GPTQ, config, a, *rhs), config, rhs, a, sorted_columns)
    check(qmatmul(QE.GPTQ, config, a, *rhs, out_dtype=torch.bfloat16), config, rhs, a)
    least = _lib.load().qmm_matmul_workspace_bytes(QE.GPTQ.code, dtype, m, n, k)
    for need in (room, max(room - 1, least), least):
        check(c_call(config, rhs, a, need), config, rhs, a)


@pytest.mark.parametrize("m,n,k", [(9, 6400, 1024), (16, 512, 512), (8, 1024, 4096), (12, 2056, 1280)])
def test_few_rows_keep_their_fp32_precision(m, n, k):
    """Codes around a zero point of 8, as quantised weights have them: a kernel that sums codes and zero points apart loses two bits to the difference."""
    config, rhs = act_order(n, k, 128, m, any_codes=False)
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m))
    check(qmatmul(QE.GPTQ, config, a, *rhs), config, rhs, a, sorted_columns=True)


# Relative error (2-norm, against float64) of the sorted columns, a tenth above what they have; the look-up kernel's in the comment
@pytest.mark.parametrize("m,n,k,group,most", [(6, 18944, 4096, 128, 1.34e-7),  # 2.75e-7
                                              (4, 5504, 18944, 128, 1.46e-7),  # 5.7e-7
                                              (2, 11648, 12032, 32, 1.67e-7),  # 4.7e-7
                                              (5, 16472, 7936, 32, 1.3e-7)])   # 3.8e-7
def test_few_rows_of_large_matrices_keep_their_precision(m, n, k, group, most):
    config, rhs = act_order(n, k, group, m, any_codes=False)
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m))
    want = a.double() @ dequantize(QE.GPTQ, *rhs, config=config).double().T
    error = ((qmatmul(QE.GPTQ, config, a, *rhs).double() - want).norm() / want.norm()).item()
    assert error <= most, error


@pytest.mark.parametrize("change", ["one column", "one group empty", "out of range"])
def test_uneven_groups(change):
    m, n, k, group = 37, 264, 2048, 128
    config, (qweight, scales, qzeros, g_idx) = act_order(n, k, group, 5)
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(2))
    if change == "one column":
        g_idx[7] = (g_idx[7] + 1) % (k // group)
    elif change == "one group empty":
        g_idx[g_idx == 3] = 4
    else:  # (clamped to the last group)
        g_idx[g_idx == k // group - 1] = 10**6
        rhs = (qweight, scales, qzeros, g_idx.clamp(max=k // group - 1))
        check(qmatmul(QE.GPTQ, config, a, qweight, scales, qzeros, g_idx), config, rhs, a)
        return
    check(qmatmul(QE.GPTQ, config, a, qweight, scales, qzeros, g_idx), config, (qweight, scales, qzeros, g_idx), a)


def test_replayed_from_a_graph():
    config, rhs = act_order(264, 1024, 128, 9)
    a = torch.randn((40, 1024), device="cuda")
    want = qmatmul(QE.GPTQ, config, a, *rhs)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = qmatmul(QE.GPTQ, config, a, *rhs)
    for i in range(3):
        a.copy_(torch.randn((40, 1024), device="cuda"))
        rhs[3].copy_(rhs[3][torch.randperm(1024, device="cuda")])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, qmatmul(QE.GPTQ, config, a, *rhs))
        assert not torch.equal(got, want)


@pytest.mark.parametrize("n,k,group", [(8200, 4096, 128), (8200, 4128, 32), (8200, 8704, 128),  # slabs of 32 columns: 4, 8, 16 columns of K a lane
                                       (4104, 4096, 512), (4104, 8192, 128), (4104, 14336, 128),  # of 16
                                       (40, 16384, 128), (40, 18944, 128), (40, 26112, 128),  # of 8, up to where words and order fill a compute unit
                                       (40, 26240, 128), (40, 28672, 32)])  # beyond: the sort as a launch of its own
def test_slabs(n, k, group):
    config, rhs = act_order(n, k, group, 3)
    a = torch.randn((20, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(4)).bfloat16()
    check(qmatmul(QE.GPTQ, config, a, *rhs), config, rhs, a, sorted_columns=True)
    uneven = rhs[3].clone()
    uneven[k - 1] = (uneven[k - 1] + 1) % (k // group)
    rhs = (*rhs[:3], uneven)
    check(qmatmul(QE.GPTQ, config, a, *rhs), config, rhs, a)


@pytest.mark.parametrize("n,k,group", [(12296, 5120, 128), (12296, 4608, 32),  # slabs of 32 columns
                                       (12296, 8704, 128), (4104, 9120, 32), (4104, 16384, 128), (2056, 20480, 64),  # of 16
                                       (2056, 20608, 128), (2056, 28672, 32)])  # of 8
def test_slabs_with_the_sort_apart(n, k, group):
    """More slabs than compute units, each with its order too large for two to a compute unit."""
    test_slabs(n, k, group)


@pytest.mark.parametrize("n,k,group", [(4104, 8704, 128), (4104, 4096, 128), (2056, 9088, 128)])  # the widest slabs of which there is one for each compute unit
def test_one_slab_a_compute_unit(n, k, group):
    test_slabs(n, k, group)


@pytest.mark.parametrize("n,k", [(8200, 4096), (4104, 4096), (40, 16384), (2056, 20608)])  # slabs of 32, 16, 8 columns, the sort apart
@pytest.mark.parametrize("words", [1, 2, 3])
def test_qweight_at_any_multiple_of_four(n, k, words):
    config, rhs = act_order(n, k, 128, 3)
    a = torch.randn((20, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(4)).bfloat16()
    moved = torch.empty(rhs[0].numel() + words, dtype=torch.int32, device="cuda")[words:].view(rhs[0].shape)
    moved.copy_(rhs[0])
    assert moved.data_ptr() % 16 == 4 * words
    got = qmatmul(QE.GPTQ, config, a, moved, *rhs[1:])
    check(got, config, rhs, a, sorted_columns=True)
    assert torch.equal(got, qmatmul(QE.GPTQ, config, a, *rhs))


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(33, 8200, 4096), (41, 8200, 4128),  # slabs of 32 columns: 8 bf16 rows of the lhs a workgroup, 4 of fp32
                                   (23, 4104, 4096), (21, 4104, 14336),  # of 16: 4 and 2
                                   (35, 40, 4096), (22, 40, 26112),  # of 8: 2 and 1
                                   (33, 8200, 160), (23, 4104, 2080), (21, 4104, 4512),  # rows of words that fill part of a turn
                                   (21, 2056, 20480), (23, 2056, 20608), (25, 12296, 4608),  # the sort as a launch of its own
                                   (600, 1032, 2048), (300, 4104, 4128)])  # more rows than the last round of the slabs has room for: a preparation of their own
def test_rows_of_the_lhs_beside_the_slabs(m, n, k, lhs):
    """Rows whose largest value is anywhere, an infinity, none at all (zeros), tiny, and what is left of a workgroup's rows."""
    config, rhs = act_order(n, k, 32, m)
    gen = torch.Generator(device="cuda").manual_seed(m)
    a = torch.randn((m, k), device="cuda", generator=gen)
    a[torch.arange(m), torch.randint(0, k, (m,), device="cuda", generator=gen)] = 300.0
    a[2] = 0.0
    a[3] *= 2.0**-100
    a[m - 1, k - 1] = -1000.0
    a = a.to(lhs)
    broken = a.clone()
    broken[5, 0], broken[6, k - 1], broken[11, k // 2] = float("inf"), float("-inf"), float("nan")
    got = qmatmul(QE.GPTQ, config, broken, *rhs)
    rows = [r for r in range(m) if r not in (5, 6, 11)]
    check(got[rows], config, rhs, a[rows])
    assert not torch.isfinite(got[[5, 6, 11]]).any()
    assert torch.equal(got[2], torch.zeros_like(got[2]))
    assert torch.equal(got[rows], qmatmul(QE.GPTQ, config, a, *rhs)[rows])


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(13, 4056, 18176),  # the sort apart, no place left for the rows: a preparation behind it
                                   (13, 7400, 8064),  # room for a few workgroups that zero, not for as many as there could be
                                   (42, 24440, 8192),  # rounds of slabs, and a few places more than the last one has
                                   (2500, 2056, 20480)])  # thousands of rows, the sort apart
def test_rows_of_the_lhs_and_places_beside_the_slabs(m, n, k, lhs):
    test_rows_of_the_lhs_beside_the_slabs(m, n, k, lhs)
