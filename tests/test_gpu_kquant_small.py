"""Q4_0, Q4_K, Q5_K and Q6_K (and GPTQ, where it has the same rules) with 1 .. 64 lhs rows: the small-batch kernel at the edges of its tiles (16 weight rows), of its groups of K (up to 16 super-blocks, divided
evenly) and of its lhs rows (2, 4, 8, 16), against float64 products of the dequantised weights."""
import ctypes

import pytest
import torch

from mojo_amd import QuantizationConfig, QuantizationEncoding as QE, dequantize, qmatmul, qmatmul_grouped, qmatmul_swiglu, quantize
from mojo_amd import _lib

pytestmark = pytest.mark.gpu
ENCODINGS = ("Q4_K", "Q5_K", "Q6_K")


def packed(enc, n, k, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(n + 7 * k + seed)
    return quantize(QE[enc], torch.empty((n, k), device="cuda").normal_(0.0, 0.02, generator=gen))


def rows(m, k, lhs):
    return torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m * k)).to(lhs)


def check(enc, got, w, a, bits=22):
    want = a.double() @ dequantize(QE[enc], w).double().T
    # fp32 rows as two fp16 terms (2^-23 of a value), exact products, fp32 sums (some 2^-24 of their terms each, which add up like a random walk): 0.7e-7 .. 1.3e-7 of a row's
    # norm, held to 2^-22 = 2.4e-7.  bits: 8 for results rounded to bf16.
    error = ((got.double() - want).norm(dim=1) / want.norm(dim=1)).max().item()
    assert error <= 2.0**-bits, (enc, tuple(got.shape), a.shape[1], a.dtype, error)


@pytest.mark.parametrize("enc", ENCODINGS)
@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
# (18 rows of one block: with 17 the number of Q6_K blocks is odd, which is not this kernel's, see below)
@pytest.mark.parametrize("m,n,k", [(2, 18, 256), (3, 1000, 768), (4, 4104, 4096), (5, 40, 4352), (8, 264, 8192), (7, 4200, 11008), (16, 1001, 2560), (9, 16, 14336), (12, 8200, 512), (16, 4112, 5120)])
def test_against_float64(enc, lhs, m, n, k):
    w, a = packed(enc, n, k), rows(min(m, 8) if lhs == torch.float32 else m, k, lhs)
    check(enc, qmatmul(QE[enc], None, a, w), w, a)
    check(enc, qmatmul(QE[enc], None, a, w, out_dtype=torch.bfloat16), w, a, bits=8)


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(1, 8200, 512), (1, 1000, 18944), (2, 18, 256), (2, 4104, 4096), (3, 1000, 768), (4, 17, 14336), (5, 40, 4352), (8, 264, 8192), (7, 4200, 11008), (9, 4112, 1024), (16, 1001, 2048),
                                   (12, 1000, 14336)])
def test_q4_0(lhs, m, n, k):
    """The lhs quantised to Q8_0 by every wavefront for itself: the codes of the package's quantiser, exact sums over blocks."""
    w, a = packed("Q4_0", n, k), rows(min(m, 8) if lhs == torch.float32 else m, k, lhs)
    a[0, :32] *= 1e-30
    a[-1, 32:64] = 0.0
    a[0, 64:96] = torch.tensor([127.0, *[x + 0.5 for x in range(-15, 16)]], device="cuda").to(lhs)  # halves between codes
    blocks = quantize(QE.Q8_0, a.float()).view(a.shape[0], -1, 34)
    x = (blocks[:, :, :2].contiguous().view(torch.float16).double() * blocks[:, :, 2:].contiguous().view(torch.int8).double()).view(a.shape)
    want = x @ dequantize(QE.Q4_0, w).double().T
    for got, bits in ((qmatmul(QE.Q4_0, None, a, w), 22), (qmatmul(QE.Q4_0, None, a, w, out_dtype=torch.bfloat16), 8)):
        assert ((got.double() - want).norm(dim=1) / want.norm(dim=1)).max().item() <= 2.0**-bits
    ws = [w, packed("Q4_0", n + 16, k, 1)]
    if m in (4, 8):
        for got, v in zip(qmatmul_grouped(QE.Q4_0, a, ws), ws):
            assert torch.equal(got, qmatmul(QE.Q4_0, None, a, v))


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("enc,n,k", [("Q4_K", 8200, 512), ("Q4_K", 9001, 2048), *((e, n, k) for e in ("Q5_K", "Q6_K") for n, k in ((4104, 4096), (2064, 11008), (264, 14336), (2050, 256), (8192, 18944)))])
def test_one_row(enc, lhs, n, k):
    """The matrices on which this kernel serves one row."""
    w, a = packed(enc, n, k), rows(1, k, lhs)
    check(enc, qmatmul(QE[enc], None, a, w), w, a)
    check(enc, qmatmul(QE[enc], None, a, w, out_dtype=torch.bfloat16), w, a, bits=8)
    if enc != "Q4_K":
        up = packed(enc, n, k, 1)
        g, u = (qmatmul(QE[enc], None, a, x).double() for x in (w, up))
        # the same sums but for how a long K is added up (2^-22); exp, the quotient and two products in fp32 (8 units of 2^-24)
        want = g / (1 + torch.exp(-g)) * u
        assert ((qmatmul_swiglu(QE[enc], a, w, up).double() - want).norm() / want.norm()).item() <= 2.0**-21


@pytest.mark.parametrize("enc", ENCODINGS)
@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("scale", [1e-36, 1e-5, 3e4, 1e30])
def test_rows_of_other_magnitudes(enc, lhs, scale):
    """Rows that are brought to fp16's range by a power of two, next to rows that need none and to one of zeros."""
    w, a = packed(enc, 136, 4608), rows(8, 4608, torch.float32)
    a[1::3] *= scale
    a[5] = 0.0
    a = a.to(lhs)
    got = qmatmul(QE[enc], None, a, w)
    assert (got[5] == 0).all()
    keep = [0, 1, 2, 3, 4, 6, 7]
    check(enc, got[keep], w, a[keep])


@pytest.mark.parametrize("enc", ENCODINGS)
@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
def test_small_values_next_to_a_few_large_ones(enc, lhs):
    """Spikes of 0.2 among values of 2^-13: what a row is scaled by decides how much of those fp16 holds."""
    w, a = packed(enc, 264, 4096), rows(8, 4096, torch.float32) * 2.0**-13
    a[:, 5::1024] = 0.2
    # (roundings of a few large terms do not average out: 2^-21; with the small values held to 2^-25, however large the spikes are, 1.4e-6 and, bf16 with 2^-17, 1.3e-6)
    check(enc, qmatmul(QE[enc], None, a.to(lhs), w), w, a.to(lhs), bits=21)
    a[:, torch.arange(4096, device="cuda") % 1024 != 5] *= 2.0**-4
    check(enc, qmatmul(QE[enc], None, a.to(lhs), w), w, a.to(lhs), bits=21)
    # rows up to 7.9 times smaller than the largest, which fp32 rows share one power of two with: 2^-31 (GPTQ 2^-36) of a row's largest left out of each value, 2^-25 of all
    a *= torch.linspace(1.0, 1.0 / 7.9, a.shape[0], device="cuda")[:, None]
    check(enc, qmatmul(QE[enc], None, a.to(lhs), w), w, a.to(lhs), bits=21)


@pytest.mark.parametrize("enc", ENCODINGS)
@pytest.mark.parametrize("m,k", [(4, 4096), (8, 11008), (3, 8448)])
def test_group_gated_pair_and_parts_of_k_give_the_same_sums(enc, m, k):
    ns = (1032, 520, 40)
    ws, a = [packed(enc, n, k, i) for i, n in enumerate(ns)], rows(m, k, torch.bfloat16)
    alone = [qmatmul(QE[enc], None, a, w) for w in ws]  # (a long K: its groups side by side, added by a launch of their own)
    for got, want in zip(qmatmul_grouped(QE[enc], a, ws), alone):  # (one after the other in each workgroup)
        assert torch.equal(got, want)
    gate, up = packed(enc, 520, k, 5), packed(enc, 520, k, 6)
    g, u = (qmatmul(QE[enc], None, a, w).double() for w in (gate, up))
    # the same sums; exp, the quotient and two products in fp32 (8 units of 2^-24)
    assert torch.allclose(qmatmul_swiglu(QE[enc], a, gate, up).double(), g / (1 + torch.exp(-g)) * u, rtol=2.0**-21, atol=1e-30)


@pytest.mark.parametrize("enc", ("Q4_0",) + ENCODINGS)
@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(2, 1, 512), (4, 7, 512), (1, 8, 8448), (8, 9, 512), (3, 17, 4608), (16, 15, 1024), (4, 2056, 4096), (20, 23, 512), (4, 4099, 512)])
def test_gated_pair_in_tiles_of_eight_rows_of_each_matrix(enc, lhs, m, n, k):
    """Eight rows of gate and of up share a tile of the matrix cores: the sums of a call with one matrix, at the edges of such tiles (silu: some 2^-24 for each of its steps)."""
    gate, up, a = packed(enc, n, k), packed(enc, n, k, 1), rows(m, k, lhs)
    g, u = qmatmul(QE[enc], None, a, gate).double(), qmatmul(QE[enc], None, a, up).double()
    assert torch.allclose(qmatmul_swiglu(QE[enc], a, gate, up).double(), g / (1 + torch.exp(-g)) * u, rtol=2.0**-21, atol=1e-30)


@pytest.mark.parametrize("enc", ("Q4_0",) + ENCODINGS)
@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(8, 2816, 1024), (16, 2815, 1024), (12, 9721, 2560), (20, 4850, 1024), (16, 6130, 4608), (8, 11007, 512),  # pairs of whole tiles: more than four rows
                                   (4, 2816, 1024), (2, 4862, 1024), (3, 2801, 512)])  # eight rows of each matrix, as many a workgroup as in pairs
def test_gated_pair_dealt_in_pairs_of_tiles(enc, lhs, m, n, k):
    """A workgroup with two items for a result, or twice as many tiles as there are places for: the sums of a call with one matrix, with a last tile that is ragged or has no second half."""
    gate, up, a = packed(enc, n, k), packed(enc, n, k, 1), rows(m, k, lhs)
    g, u = qmatmul(QE[enc], None, a, gate).double(), qmatmul(QE[enc], None, a, up).double()
    assert torch.allclose(qmatmul_swiglu(QE[enc], a, gate, up).double(), g / (1 + torch.exp(-g)) * u, rtol=2.0**-21, atol=1e-30)


def test_q6_k_at_every_multiple_of_four_and_an_odd_last_block():
    """Blocks of 210 bytes: rows that begin at 0 and at 2 mod 4 alternate with an odd number of blocks; a matrix of an odd number of them in all is left to the kernels
    that read its last one exactly."""
    for n, k, lead in ((32, 768, 4), (33, 1536, 8), (33, 768, 0), (24, 1280, 12)):
        w, a = packed("Q6_K", n, k), rows(4, k, torch.float32)
        buffer = torch.zeros(w.numel() + 16, dtype=torch.uint8, device="cuda")
        at = buffer[lead : lead + w.numel()].view(w.shape)
        at.copy_(w)
        check("Q6_K", qmatmul(QE.Q6_K, None, a, at), w, a, bits=20)  # (the last shape goes to kernels with more rounding: 4e-7)


def test_workspace_is_what_the_parts_of_k_need():
    lib = _lib.load()
    need = lib.qmm_preferred_workspace_bytes(0, 1, None, 0, 4, 4096, 14336, 0)
    assert need >= 4 * 4 * 4096 * 4  # four groups of K, [4, 4096] fp32 each


@pytest.mark.parametrize("enc,m,n,k", [("Q6_K", 16, 4104, 14336), ("Q4_K", 16, 28680, 8192)])
def test_tiles_that_leave_lds_a_few_at_a_time(enc, m, n, k):
    """Groups of K side by side, results of some of a workgroup's tiles in LDS at a time: the operands of the group serve all of them."""
    w, a = packed(enc, n, k), rows(m, k, torch.bfloat16)
    check(enc, qmatmul(QE[enc], None, a, w), w, a)


@pytest.mark.parametrize("enc", ("Q4_0", *ENCODINGS))
@pytest.mark.parametrize("m,n,k", [(48, 2048, 768), (48, 3072, 768), (64, 2560, 1024), (64, 3584, 1024), (40, 4352, 1024), (17, 6144, 1024), (17, 6144, 1280), (32, 8192, 1280), (32, 6144, 1536), (16, 14336, 768)])
def test_on_both_sides_of_the_lines_for_a_short_k(enc, m, n, k):
    """Tiles of lhs rows side by side, or the direct GEMM where a compute unit would get too many of them."""
    w, a = packed(enc, n, k), rows(m, k, torch.bfloat16)
    if enc == "Q4_0":
        blocks = quantize(QE.Q8_0, a.float()).view(m, -1, 34)
        a = (blocks[:, :, :2].contiguous().view(torch.float16).double() * blocks[:, :, 2:].contiguous().view(torch.int8).double()).view(m, k)
    check(enc, qmatmul(QE[enc], None, rows(m, k, torch.bfloat16), w), w, a)


@pytest.mark.parametrize("m", [9, 16])
def test_no_matrix_is_too_large_for_a_short_k(m):
    """fp32 rows side by side whatever the number of weights, up to K = 4096."""
    w, a = packed("Q4_K", 65544, 4096), rows(m, 4096, torch.float32)
    got = qmatmul(QE.Q4_K, None, a, w)
    for part in (slice(0, 4112), slice(65544 - 4112, 65544)):
        check("Q4_K", got[:, part], w[part], a)


def alone(encoding, config, a, rhs, step):
    """The rows of `a` in calls of `step` rows, the last of which repeats rows of the one before."""
    m, out = a.shape[0], []
    for r in range(0, m, step):
        first = max(0, min(r, m - step))
        out.append(qmatmul(encoding, config, a[first : first + step].contiguous(), *rhs)[r - first :])
    return torch.cat(out)


def tile_calls():
    everywhere = ((16, 256), (1000, 1536), (136, 4608), (264, 14336), (1032, 11008))
    for enc in ("Q4_0", "GPTQ", *ENCODINGS):
        for lhs, each in ((torch.float32, 8), (torch.bfloat16, 16)):
            for tiles in (2, 3, 4):
                if enc == "GPTQ" or (lhs == torch.float32 and (tiles == 2 or enc == "Q4_0")):
                    shapes = everywhere
                elif enc == "Q4_0" or (lhs == torch.bfloat16 and tiles == 2):  # (the others go to other kernels)
                    shapes = ((16, 256), (1000, 1536), (264, 14336))
                else:
                    shapes = ((16, 256), (1000, 768), (264, 14336))
                for n, k in shapes:
                    yield enc, lhs, each, n, k, tiles


@pytest.mark.parametrize("enc,lhs,rows_each,n,k,tiles", list(tile_calls()))
def test_tiles_of_lhs_rows(enc, lhs, rows_each, n, k, tiles):
    """More rows than a workgroup takes: the sums of calls with the rows of one; a last tile of one row and a full one; results in bf16; in a group; with less memory than groups of K need."""
    config, more = None, ()
    if enc == "GPTQ":
        gen = torch.Generator(device="cuda").manual_seed(n + k)
        words = lambda *shape: torch.randint(-(2**31), 2**31, shape, device="cuda", generator=gen, dtype=torch.int64).to(torch.int32)
        config, rhs = QuantizationConfig("gptq", 4, 128, False, False), (words(k // 8, n), torch.empty((k // 128, n), device="cuda").uniform_(1e-3, 4e-3, generator=gen).half(), words(k // 128, n // 8))
    else:
        rhs, more = (packed(enc, n, k),), (packed(enc, n + 16, k, 1),)
    encoding, lib = QE[enc], _lib.load()
    for m in (rows_each * (tiles - 1) + 1, rows_each * tiles):
        a = rows(m, k, lhs)
        a[m - 1] *= 3.0 if enc == "Q4_0" else 1e30  # (a row that is scaled on its way to fp16; Q8_0 scales are fp16)
        want = alone(encoding, config, a, rhs, rows_each)
        assert torch.equal(qmatmul(encoding, config, a, *rhs), want)
        assert torch.equal(qmatmul(encoding, config, a, *rhs, out_dtype=torch.bfloat16), want.bfloat16())
        if more:
            for got, w in zip(qmatmul_grouped(encoding, a, [*rhs, *more]), (rhs, more)):
                assert torch.equal(got, alone(encoding, config, a, w, rows_each))
        out, ptrs = torch.empty((m, n), device="cuda"), (ctypes.c_void_p * len(rhs))(*(t.data_ptr() for t in rhs))
        cfg = _lib.GptqConfig(4, 128, 0, 0) if config else None
        kind = _lib.QMM_F32 if lhs == torch.float32 else _lib.QMM_BF16
        ws = torch.empty(max(256, lib.qmm_matmul_workspace_bytes(encoding.code, kind, m, n, k)), dtype=torch.uint8, device="cuda")
        assert lib.qmm_matmul(encoding.code, cfg and ctypes.byref(cfg), a.data_ptr(), kind, m, k, ptrs, len(rhs), n, out.data_ptr(), ws.data_ptr(), ws.numel(), 0, torch.cuda.current_stream().cuda_stream) == 0
        assert torch.equal(out, want)
