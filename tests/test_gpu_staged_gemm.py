"""The GEMM whose lhs and packed weights go to LDS by themselves, at the edges of its tiles (64, 96 or 128 rows, 64, 128 or 256 columns), of its units of 256
values of K and of the ways it cuts K (one to four parts a workgroup, one or two workgroups a tile), against float64 products of the same integers."""
import ctypes as C

import pytest
import torch

from mojo_amd import QuantizationEncoding as QE, _lib, dequantize, qmatmul, qmatmul_grouped
from test_gpu_direct_gemm import check, weights

pytestmark = pytest.mark.gpu

# (rows, columns, K): one unit and several, parts of unequal lengths; a row and a column short of a tile and beyond one
SIZES = ((79, 5128, 4352), (97, 4104, 4352), (100, 14344, 256), (129, 11016, 2304), (161, 14344, 1280), (200, 4104, 4352), (255, 14336, 512), (257, 6152, 2304), (330, 8200, 768),
         (385, 14328, 1024), (641, 4104, 2304), (700, 9000, 512), (1300, 4104, 768))


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("enc,group", [(QE.Q4_K, 0), (QE.Q5_K, 0), (QE.Q6_K, 0), (QE.GPTQ, 128), (QE.GPTQ, 256), (QE.GPTQ, 32)])
def test_edges(enc, group, lhs):
    for m, n, k in SIZES:
        config, rhs = weights(enc, group, n, k)
        a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).to(lhs)
        a[m // 2] *= 1e-6
        a[m - 1] = 0.0
        check(qmatmul(enc, config, a, *rhs), enc, config, rhs, a)
        check(qmatmul(enc, config, a, *rhs, out_dtype=torch.bfloat16), enc, config, rhs, a)


@pytest.mark.parametrize("lhs,m,n,k,limit", [(torch.bfloat16, 160, 11008, 4096, 0.75e-7), (torch.bfloat16, 190, 11008, 2816, 0.76e-7), (torch.float32, 160, 14336, 4096, 1.33e-7),
                                               (torch.float32, 160, 11008, 5376, 1.37e-7)])
def test_folded_sums(lhs, m, n, k, limit):
    """Sums over four units of K that are added up in others (16, 11 and 21 units): a tenth above 0.67e-7, 0.69e-7, 1.21e-7 and 1.25e-7, where one chain over 16 has 1.03e-7
    (fp32 rows: 1.43e-7)."""
    config, rhs = weights(QE.GPTQ, 128, n, k)
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m + k)).to(lhs)
    want = a.double() @ dequantize(QE.GPTQ, *rhs, config=config).double().T
    assert ((qmatmul(QE.GPTQ, config, a, *rhs).double() - want).norm() / want.norm()).item() <= limit


@pytest.mark.parametrize("n", [2048 + 1, 14336 - 3])
def test_odd_columns(n):
    """K-quants take any number of columns: rows of the result that begin at any multiple of four bytes."""
    for enc in (QE.Q4_K, QE.Q6_K):
        _, rhs = weights(enc, 0, n, 1024)
        a = torch.randn((190, 1024), device="cuda", generator=torch.Generator(device="cuda").manual_seed(n)).bfloat16()
        check(qmatmul(enc, None, a, *rhs), enc, None, rhs, a)


def test_misaligned_gptq_words():
    """qweight may lie at any multiple of four bytes, which is what loads of 16 bytes to LDS want."""
    config, rhs = weights(QE.GPTQ, 128, 14336, 1024)
    a = torch.randn((200, 1024), device="cuda", generator=torch.Generator(device="cuda").manual_seed(3)).bfloat16()
    words = torch.empty(rhs[0].numel() + 1, dtype=torch.int32, device="cuda")
    words[1:] = rhs[0].flatten()
    moved = (words[1:].view(rhs[0].shape), *rhs[1:])
    lib = _lib.load()
    cfg = C.byref(_lib.GptqConfig(4, 128, 0, 1))
    need = lib.qmm_preferred_workspace_bytes(_lib.QMM_OP_MATMUL, QE.GPTQ.code, cfg, _lib.QMM_BF16, 200, 14336, 1024, 0)
    ws, out = torch.empty(need, dtype=torch.uint8, device="cuda"), torch.full((200, 14336), float("nan"), device="cuda")
    ptrs = (C.c_void_p * 3)(*[t.data_ptr() for t in moved])
    assert lib.qmm_matmul(QE.GPTQ.code, cfg, a.data_ptr(), _lib.QMM_BF16, 200, 1024, ptrs, 3, 14336, out.data_ptr(), ws.data_ptr(), need, 0,
                          torch.cuda.current_stream().cuda_stream) == 0
    check(out, QE.GPTQ, config, moved, a)


@pytest.mark.parametrize("group,m,n,k", [(128, 200, 14336, 1024), (32, 200, 14336, 1024), (128, 1000, 14336, 4096), (128, 161, 14344, 1280)])
@pytest.mark.parametrize("words", [1, 2, 3])
def test_misaligned_gptq_words_give_the_same_bits(group, m, n, k, words):
    config, rhs = weights(QE.GPTQ, group, n, k)
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).bfloat16()
    moved = torch.empty(rhs[0].numel() + words, dtype=torch.int32, device="cuda")[words:].view(rhs[0].shape)
    moved.copy_(rhs[0])
    assert moved.data_ptr() % 16 == 4 * words
    assert torch.equal(qmatmul(QE.GPTQ, config, a, moved, *rhs[1:]), qmatmul(QE.GPTQ, config, a, *rhs))


@pytest.mark.parametrize("m,n,k", [(300, 8192, 512), (700, 14336, 1024), (1500, 4096, 768)])
def test_q6_k_between_multiples_of_four(m, n, k):
    _, (w,) = weights(QE.Q6_K, 0, n, k)
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).bfloat16()
    moved = torch.empty(w.numel() + 2, dtype=torch.uint8, device="cuda")[2:].view(w.shape)
    moved.copy_(w)
    check(qmatmul(QE.Q6_K, None, a, moved), QE.Q6_K, None, (w,), a)
    check(qmatmul(QE.Q6_K, None, a, moved, out_dtype=torch.bfloat16), QE.Q6_K, None, (w,), a)


@pytest.mark.parametrize("m,n,k", [(190, 8193, 256), (190, 8193, 768), (300, 4097, 2304), (700, 14337, 1280), (200, 8194, 768)])
def test_q6_k_with_an_odd_number_of_blocks(m, n, k):
    """In the last bytes of a buffer: no kernel may look beyond them for what it multiplies."""
    _, (w,) = weights(QE.Q6_K, 0, n, k)
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).bfloat16()
    whole = torch.full(((w.numel() + 2047) // 1024 * 1024,), 255, dtype=torch.uint8, device="cuda")
    start = (whole.numel() - w.numel()) // 4 * 4
    moved = whole[start:start + w.numel()].view(w.shape)
    moved.copy_(w)
    check(qmatmul(QE.Q6_K, None, a, moved), QE.Q6_K, None, (w,), a)


def test_matrices_together_sum_as_alone():
    """q | k | v in one launch: the bits of three calls of their own."""
    for enc in (QE.Q4_K, QE.Q5_K, QE.Q6_K):
        for m, ns, k in ((200, (4096, 1024, 1024), 4096), (300, (4104, 4104), 2304)):
            mats = [weights(enc, 0, n, k)[1][0] for n in ns]
            a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).bfloat16()
            for got, w in zip(qmatmul_grouped(enc, a, mats), mats):
                assert torch.equal(got, qmatmul(enc, None, a, w))


@pytest.mark.parametrize("enc,m,n,count,k", [(QE.Q4_K, 385, 5120, 3, 4096), (QE.Q5_K, 193, 5120, 3, 4096), (QE.Q4_K, 228, 5632, 2, 1024), (QE.Q4_K, 540, 4096, 3, 1024)])
def test_a_tile_for_several_matrices_keeps_their_sums(enc, m, n, count, k):
    """Sizes at which matrices together would take 128 rows a wavefront where each alone takes 64 or 96, with codes around their middle."""
    w = weights(enc, 0, n, k)[1][0]
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).bfloat16()
    alone = qmatmul(enc, None, a, w)
    for got in qmatmul_grouped(enc, a, [w] * count):
        assert torch.equal(got, alone)


# Relative error of (enc, group, rows, n, k, lhs): the float32 sums of the kernel that served the call before, by 1.08
@pytest.mark.parametrize("enc,group,m,n,k,lhs,most", [
    (QE.Q4_K, 0, 96, 4096, 4096, torch.bfloat16, 1.06e-7), (QE.Q4_K, 0, 200, 14336, 4096, torch.bfloat16, 2.2e-7), (QE.Q4_K, 0, 200, 4096, 4096, torch.float32, 2.04e-7),
    (QE.Q5_K, 0, 64, 14336, 4096, torch.bfloat16, 1.35e-7), (QE.Q6_K, 0, 500, 4096, 14336, torch.bfloat16, 1.5e-7), (QE.GPTQ, 128, 400, 4096, 4096, torch.bfloat16, 0.86e-7),
    (QE.GPTQ, 32, 300, 4096, 4096, torch.bfloat16, 0.85e-7), (QE.GPTQ, 128, 800, 14336, 4096, torch.float32, 1.7e-7)])
def test_precision(enc, group, m, n, k, lhs, most):
    from mojo_amd import QuantizationConfig, dequantize, quantize, quantize_gptq

    gen = torch.Generator(device="cuda").manual_seed(5)
    w = torch.empty((n, k), device="cuda").normal_(0.0, 0.02, generator=gen)
    config = QuantizationConfig("gptq", 4, group, False, True) if enc == QE.GPTQ else None
    rhs = quantize_gptq(w, config)[:3] if config else (quantize(enc, w),)
    a = torch.randn((m, k), device="cuda", generator=gen).to(lhs)
    want = a.double() @ dequantize(enc, *rhs, config=config).double().T
    assert ((qmatmul(enc, config, a, *rhs).double() - want).norm() / want.norm()).item() < most


# The same of calls whose parts of K would be longer or joined in another order than in the direct or shared kernel: the error of that kernel, and what its order
# of joining the parts is worth (0.3 %)
@pytest.mark.parametrize("enc,group,m,n,k,lhs,most", [
    (QE.GPTQ, 32, 202, 12192, 1024, torch.float32, 0.9592e-7), (QE.GPTQ, 32, 360, 13248, 1792, torch.float32, 1.0652e-7), (QE.GPTQ, 32, 66, 14336, 4096, torch.float32, 1.1225e-7),
    (QE.GPTQ, 128, 786, 2248, 512, torch.bfloat16, 0.4073e-7), (QE.GPTQ, 128, 60, 14336, 4096, torch.bfloat16, 0.6657e-7), (QE.GPTQ, 128, 1330, 728, 2048, torch.float32, 1.1498e-7),
    (QE.Q6_K, 0, 252, 15480, 512, torch.bfloat16, 1.0096e-7), (QE.Q4_K, 0, 481, 6144, 1024, torch.float32, 1.6326e-7), (QE.Q4_K, 0, 385, 5120, 4096, torch.bfloat16, 1.2078e-7),
    (QE.Q5_K, 0, 193, 5120, 4096, torch.bfloat16, 1.0544e-7), (QE.Q4_K, 0, 200, 4096, 4096, torch.bfloat16, 1.9066e-7), (QE.Q5_K, 0, 481, 7104, 512, torch.bfloat16, 2.0712e-7)])
def test_no_less_exact_than_the_kernel_before(enc, group, m, n, k, lhs, most):
    test_precision(enc, group, m, n, k, lhs, 1.003 * most)


def test_rows_of_more_than_2_to_the_23_columns():
    """Row tiles whose operands lie half a gigabyte apart, eight of them and one row: bf16 rows of 2^23 + 256 columns.  The first and the last 256 columns hold most of the product."""
    m, n, k = 513, 8, 2**23 + 256
    config, rhs = weights(QE.GPTQ, 128, n, k)
    gen = torch.Generator(device="cuda").manual_seed(4)
    a = torch.empty((m, k), dtype=torch.bfloat16, device="cuda").normal_(generator=gen)
    a[:, :256] *= 2.0**12
    a[:, -256:] *= 2.0**12
    plain = dequantize(QE.GPTQ, *rhs, config=config)
    want = sum(x.double() @ y.double().T for x, y in zip(a.split(2**19, 1), plain.split(2**19, 1)))
    got = qmatmul(QE.GPTQ, config, a, *rhs)
    # (2^14 sums of a unit one after the other and their parts: 2^-24 of what is summed up each, as a random walk below 2^-15)
    assert ((got.double() - want).norm() / want.norm()).item() < 2.0**-15
