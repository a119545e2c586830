"""fp32 GEMM on bf16 pieces (sgemm_x3.hip): tile edges, cut-short K stages,
layouts, unaligned rows, batches and K splits, and the values the pieces
cannot carry (infinities, NaN, overflow, rows near the subnormals).

Bar: with S = |A| |B| (the sum of the product magnitudes), each output is
within (K/32 + 12) 2^-24 S of the exact one: one rounding of the running sum
per 32 k, six per stage of the products, two for alpha / the K split, and
under 2^-24 S left out of the products.
"""
import ctypes as C

import pytest

from test_sgemm_plan import plan

pytestmark = pytest.mark.gpu


def _gh():
    import ghostflow_hip
    return ghostflow_hip


def _operands(torch, dev, m, n, k, ta, tb, seed, pad=0, scale=1.0):
    """op(A) [m, k], op(B) [k, n] and the stored forms, `pad` floats between
    rows and (with pad) a base 4 bytes off 16-byte alignment."""
    g = torch.Generator(device=dev)
    g.manual_seed(seed)

    def stored(r, c):
        ld = c + pad
        buf = torch.randn(r * ld + 1, device=dev, generator=g) * scale
        off = 1 if pad else 0
        return buf, off, ld, buf[off:off + r * ld].view(r, ld)[:, :c]

    a = stored(k, m) if ta else stored(m, k)
    b = stored(n, k) if tb else stored(k, n)
    opa = a[3].t() if ta else a[3]
    opb = b[3].t() if tb else b[3]
    return a, b, opa, opb


def _sgemm(torch, gh, a, b, m, n, k, ta, tb, out, alpha=1.0, beta=0.0, bias=None):
    L = gh.lib()
    rc = L.gfh_sgemm(int(ta), int(tb), m, n, k, alpha, a[0].data_ptr() + 4 * a[1], a[2], b[0].data_ptr() + 4 * b[1],
                     b[2], beta, out.data_ptr(), out.shape[1], None if bias is None else bias.data_ptr(),
                     torch.cuda.current_stream().cuda_stream)
    assert rc == 0, L.gfh_last_error()


def _check(torch, got, opa, opb, k):
    ref = opa.double() @ opb.double()
    s = opa.double().abs() @ opb.double().abs()
    assert ((got.double() - ref).abs() <= (k / 32 + 12) * 2.0 ** -24 * s).all(), \
        float(((got.double() - ref).abs() / s).max())


# remainders of rows, columns and K on the 32 x 64, 64 x 64, 128 x 64 and 128 x
# 128 tiles, and on the 256 x 128 one, whole and with K split
# (test_sgemm_plan.py checks which tiles these are)
SHAPES = [(17, 70, 33), (32, 640, 1000), (40, 100, 63), (65, 129, 97), (64, 64, 32), (130, 257, 64), (500, 500, 95),
          (1000, 700, 45), (700, 1500, 401), (2000, 1100, 129), (4100, 2050, 70), (96, 512, 4099)]
LARGE = [(4090, 4090, 1000), (4000, 4000, 401), (5000, 3000, 129), (2050, 2050, 525), (900, 1000, 8201),
         (2000, 2060, 4099)]


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k", SHAPES + LARGE)
def test_edges_and_layouts(torch_dev, m, n, k, ta, tb):
    import torch
    gh = _gh()
    for pad in (0, 3):
        a, b, opa, opb = _operands(torch, torch_dev, m, n, k, ta, tb, m + n + k, pad)
        out = torch.full((m, n + pad), 7.0, device=torch_dev)
        _sgemm(torch, gh, a, b, m, n, k, ta, tb, out)
        _check(torch, out[:, :n], opa, opb, k)
        assert (out[:, n:] == 7.0).all()


@pytest.mark.parametrize("m,n,k", [(48, 192, 2048), (300, 260, 1056), (33, 64, 8190), (700, 1700, 5000),
                                   (130, 1579, 4515), (84, 960, 3520)])
def test_epilogue_and_split_k(torch_dev, m, n, k):
    """alpha, beta and bias on shapes whose K is split; three calls in a row
    (the arrival counters return to zero) give the same bits."""
    import torch
    gh = _gh()
    a, b, opa, opb = _operands(torch, torch_dev, m, n, k, 0, 1, k)
    bias = torch.randn(n, device=torch_dev)
    c0 = torch.randn(m, n, device=torch_dev)
    plain = torch.empty(m, n, device=torch_dev)
    _sgemm(torch, gh, a, b, m, n, k, 0, 1, plain)
    _check(torch, plain, opa, opb, k)
    want = (plain * 0.7 + c0 * -1.3) + bias
    for _ in range(3):
        out = c0.clone()
        _sgemm(torch, gh, a, b, m, n, k, 0, 1, out, 0.7, -1.3, bias)
        assert torch.equal(out, want)


@pytest.mark.parametrize("m,n,k,ba,bb,batch", [(70, 50, 40, 6, 3, 6), (130, 300, 100, 5, 5, 5), (64, 65, 33, 1, 4, 4),
                                               (300, 200, 65, 2, 1, 3)])
def test_batches_modulo(torch_dev, m, n, k, ba, bb, batch):
    import torch
    gh = _gh()
    for ta, tb in ((0, 0), (0, 1), (1, 0), (1, 1)):
        a = torch.randn((ba,) + ((k, m) if ta else (m, k)), device=torch_dev)
        b = torch.randn((bb,) + ((n, k) if tb else (k, n)), device=torch_dev)
        out = torch.empty(batch, m, n, device=torch_dev)
        rc = gh.lib().gfh_sgemm_strided_batched(ta, tb, m, n, k, 1.0, a.data_ptr(), a.shape[2], m * k, ba, b.data_ptr(),
                                                b.shape[2], n * k, bb, 0.0, out.data_ptr(), n, m * n, batch, None,
                                                torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        for i in range(batch):
            x, y = a[i % ba], b[i % bb]
            _check(torch, out[i], x.t() if ta else x, y.t() if tb else y, k)


@pytest.mark.parametrize("m,n,k,ba,bb,batch", [(32, 345, 1742, 2, 2, 2), (411, 140, 2100, 3, 1, 6), (40, 100, 4100, 4, 2, 4),
                                               (500, 64, 4096, 2, 2, 2)])
def test_batches_split_k(torch_dev, m, n, k, ba, bb, batch):
    """Batches whose K is split: every slice's own partials and counters, with
    alpha, beta and a bias, the same bits from call to call."""
    import torch
    for ta, tb in ((0, 0), (0, 1), (1, 0), (1, 1)):
        assert plan(m, n, k, ta, tb, batch)[2] > 1
        a = torch.randn((ba,) + ((k, m) if ta else (m, k)), device=torch_dev)
        b = torch.randn((bb,) + ((n, k) if tb else (k, n)), device=torch_dev)
        bias, c0 = torch.randn(n, device=torch_dev), torch.randn(batch, m, n, device=torch_dev)

        def call(out, alpha, beta, bias):
            rc = _gh().lib().gfh_sgemm_strided_batched(
                ta, tb, m, n, k, alpha, a.data_ptr(), a.shape[2], m * k, ba, b.data_ptr(), b.shape[2], n * k, bb, beta,
                out.data_ptr(), n, m * n, batch, bias, torch.cuda.current_stream().cuda_stream)
            assert rc == 0
            return out

        plain = call(torch.empty_like(c0), 1.0, 0.0, None)
        for i in range(batch):
            x, y = a[i % ba], b[i % bb]
            _check(torch, plain[i], x.t() if ta else x, y.t() if tb else y, k)
        want = (plain * 0.7 + c0 * -1.3) + bias
        for _ in range(3):
            assert torch.equal(call(c0.clone(), 0.7, -1.3, bias.data_ptr()), want)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0)])
def test_whole_24_bits(torch_dev, ta, tb):
    """A permutation matrix returns the other operand's bits: all three pieces
    of every value arrive."""
    import torch
    gh = _gh()
    n = 96
    x = torch.randn(n, n, device=torch_dev) * torch.logspace(-20, 20, n, device=torch_dev)
    perm = torch.eye(n, device=torch_dev)[torch.randperm(n, generator=torch.Generator().manual_seed(1)).to(torch_dev)]
    for left in (True, False):
        a, b = (perm, x) if left else (x, perm)
        got = gh.sgemm(a.t().contiguous() if ta else a.contiguous(), b.t().contiguous() if tb else b.contiguous(),
                       trans_a=bool(ta), trans_b=bool(tb))
        idx = perm.argmax(1)
        assert torch.equal(got, x[idx] if left else x[:, idx.argsort()])


@pytest.mark.parametrize("tb", [0, 1])
def test_non_finite_values(torch_dev, tb):
    """An infinity or NaN reaches exactly the outputs it reaches in fp32 (an
    infinite term's sum is infinite, not NaN), and finite outputs stay within
    the bound; sums that overflow give the infinity."""
    import torch
    gh = _gh()
    m, n, k = 150, 140, 70
    a = torch.randn(m, k, device=torch_dev)
    b = torch.randn(k, n, device=torch_dev).abs() + 0.5
    a[3, 5] = float("inf")
    a[77, 9] = float("-inf")
    a[140, 69] = float("nan")
    a[20, :] = 3e38
    a[21, :] = 3.4e38  # rounds up to infinity as a bf16
    a[21, 1:] = 0.0
    b[0, 100] = 0.25
    got = gh.sgemm(a, b.t().contiguous() if tb else b, trans_b=bool(tb))
    ref = a.double() @ b.double()
    ref = torch.where(ref.abs() > 3.4028235677973366e38, ref.sign() * float("inf"), ref)
    assert torch.equal(got.isnan(), ref.isnan())
    assert torch.equal(got.isinf(), ref.isinf())
    assert torch.equal(got[got.isinf()].double(), ref[ref.isinf()])
    fin = ref.isfinite()
    s = torch.nan_to_num(a.double().abs(), 0, 0, 0) @ b.double().abs()
    assert ((got.double() - ref).abs()[fin] <= ((k / 2 + 12) * 2.0 ** -24 * s)[fin]).all()


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0)])
def test_tiny_rows(torch_dev, ta, tb):
    """Rows whose low pieces would fall below the subnormals keep fp32
    precision: against 64 bits, relative to S."""
    import torch
    gh = _gh()
    m, n, k = 70, 66, 64
    a, b, opa, opb = _operands(torch, torch_dev, m, n, k, ta, tb, 3)
    opa.mul_(2.0 ** -118)
    opb.mul_(2.0 ** 40)
    opa[5:9].mul_(2.0 ** 100)
    out = torch.empty(m, n, device=torch_dev)
    _sgemm(torch, gh, a, b, m, n, k, ta, tb, out)
    ref = opa.double() @ opb.double()
    s = opa.double().abs() @ opb.double().abs()
    # (the f32 chain: one rounding per 2 k)
    assert ((out.double() - ref).abs() <= (k / 2 + 4) * 2.0 ** -24 * s).all()


def test_group_equals_separate_products(torch_dev):
    """The SwiGLU's gate and up share a launch: h from the block equals h from
    separate linears within the bound carried through silu * up."""
    import torch
    gh = _gh()
    m, hid, inter = 100, 192, 320
    x = torch.randn(m, hid, device=torch_dev)
    w = [torch.randn(inter, hid, device=torch_dev) * 0.1 for _ in range(2)]
    bb = [torch.randn(inter, device=torch_dev) for _ in range(2)]
    wd = torch.randn(hid, inter, device=torch_dev)
    _, h = gh.swiglu(x, w[0], bb[0], w[1], bb[1], wd, None, want_h=True)
    g, u = (x.double() @ wi.double().t() + bi.double() for wi, bi in zip(w, bb))
    eps = (hid / 32 + 13) * 2.0 ** -24
    sg, su = (x.double().abs() @ wi.double().abs().t() + bi.double().abs() for wi, bi in zip(w, bb))
    ref = torch.nn.functional.silu(g) * u
    bound = eps * (1.1 * sg * u.abs() + g.abs() * su) + 8 * 2.0 ** -24 * ref.abs() + 1e-30
    assert ((h.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("over", [0, 5])
@pytest.mark.parametrize("operand,ta,tb", [("a", 0, 0), ("a", 0, 1), ("a", 1, 0), ("b", 0, 0), ("b", 0, 1), ("b", 1, 1)])
def test_offset_limits(torch_dev, operand, ta, tb, over):
    """Leading dimensions at the limits of the tiles' 32-bit offsets, 2^22 for a
    k-contiguous operand and 2^23 for a k-major one, and just beyond, where
    64-bit ones take their place."""
    import torch
    kmajor = ta if operand == "a" else not tb
    m, k, n = 263, 171 if kmajor else 1003, 270
    assert plan(m, n, k, ta, tb) is not None
    ld = (1 << (23 if kmajor else 22)) + over
    _big_ld(torch, torch_dev, operand, m, n, k, ta, tb, ld)


def test_offset_limit_of_the_largest_tile(torch_dev):
    import torch
    m, n, k = 2050, 2050, 525
    assert plan(m, n, k)[:2] == (256, 128)
    _big_ld(torch, torch_dev, "a", m, n, k, 0, 0, 1 << 22)


def _big_ld(torch, dev, operand, m, n, k, ta, tb, ld):
    def stored(rows, cols, wide):
        w = ld if wide else cols
        x = torch.as_strided(torch.empty((rows - 1) * w + cols, device=dev), (rows, cols), (w, 1))
        return x.copy_(torch.randn(rows, cols, device=dev))

    a = stored(*((k, m) if ta else (m, k)), operand == "a")
    b = stored(*((n, k) if tb else (k, n)), operand == "b")
    out = torch.empty(m, n, device=dev)
    rc = _gh().lib().gfh_sgemm(ta, tb, m, n, k, C.c_float(1.0), a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0),
                               C.c_float(0.0), out.data_ptr(), n, None, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    _check(torch, out, (a.t() if ta else a).contiguous(), (b.t() if tb else b).contiguous(), k)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k", [(70, 130, 96), (300, 200, 40), (33, 64, 2100)])
def test_small_elements_beside_large_ones(torch_dev, m, n, k, ta, tb):
    """Elements down to the fp32 subnormals keep their 24 bits next to elements
    near 1 in the same row: products of theirs are the output where the other
    operand is zero at the large ones.  Each output within the bar, plus the
    rounding of a subnormal result."""
    import torch
    g = torch.Generator().manual_seed(m + k)
    for e in (-112, -120, -127, -145):
        small = torch.randn(m, k, dtype=torch.float64, generator=g) * 2.0 ** e
        small[:, ::8] = torch.randn(m, (k + 7) // 8, dtype=torch.float64, generator=g)
        other = torch.randn(k, n, dtype=torch.float64, generator=g) * 2.0 ** 60
        other[::8, :n // 2] = 0.0
        for a64, b64 in ((small, other), (other.t(), small.t())):
            opa, opb = a64.float(), b64.float()
            a = (opa.t() if ta else opa).contiguous().to(torch_dev)
            b = (opb.t() if tb else opb).contiguous().to(torch_dev)
            got = _gh().sgemm(a, b, trans_a=bool(ta), trans_b=bool(tb)).cpu().double()
            ref, s = opa.double() @ opb.double(), opa.double().abs() @ opb.double().abs()
            assert ((got - ref).abs() <= (k / 32 + 12) * 2.0 ** -24 * s + 2.0 ** -148).all(), \
                (e, float(((got - ref).abs() / s).max()))


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_large_sums(torch_dev, ta, tb):
    """Values and sums up to the largest fp32 ones, finite ones within the f32
    chain's bound (they leave the range of the pieces)."""
    import torch
    m, n, k = 70, 66, 64
    for ea, eb in ((110, 10), (60, 60), (0, 120), (50, 46)):
        a, b, opa, opb = _operands(torch, torch_dev, m, n, k, ta, tb, ea)
        opa.mul_(2.0 ** ea)
        opb.mul_(2.0 ** eb)
        out = torch.empty(m, n, device=torch_dev)
        _sgemm(torch, _gh(), a, b, m, n, k, ta, tb, out)
        ref, s = opa.double() @ opb.double(), opa.double().abs() @ opb.double().abs()
        assert out.isfinite().all()
        assert ((out.double() - ref).abs() <= (k / 2 + 4) * 2.0 ** -24 * s).all()
