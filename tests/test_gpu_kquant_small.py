"""Q4_0, Q4_K, Q5_K and Q6_K with 1 .. 16 lhs rows: the small-batch kernel at the edges of its tiles (16 weight rows), of its groups of K (up to 16 super-blocks, divided
evenly) and of its lhs rows (2, 4, 8, 16), against float64 products of the dequantised weights."""
import pytest
import torch

from mojo_amd import QuantizationEncoding as QE, dequantize, qmatmul, qmatmul_grouped, qmatmul_swiglu, quantize
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
    w, a = packed(enc, n, k), rows(min(m, 8) if lhs == torch.float32 else m, k, lhs)  # (from nine fp32 rows on other kernels serve the call)
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
