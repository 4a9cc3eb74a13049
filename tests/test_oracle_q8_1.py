"""Pins the oracle's F32 -> Q8_1 quantiser (ggml-cuda quantize_q8_1
arithmetic) by its invariants and exact special cases."""
import numpy as np


def _split(q8, nblk):
    b = q8.reshape(-1, nblk, 36)
    d = b[..., 0:2].copy().view(np.uint16)[..., 0]
    s = b[..., 2:4].copy().view(np.uint16)[..., 0]
    qs = b[..., 4:].view(np.int8)
    return d, s, qs


def test_invariants(O):
    rng = np.random.default_rng(5)
    x = (rng.standard_normal((3, 4096)) * rng.uniform(0.01, 100, size=(3, 1))).astype(np.float32)
    q8 = O.quantize_q8_1(x)
    d16, s16, qs = _split(q8, 4096 // 32)
    d = O.f16_bits_to_f32(d16)
    xb = x.reshape(3, -1, 32)
    amax = np.abs(xb).max(-1)
    assert np.abs(qs.astype(np.int32)).max() <= 127
    # d is half(amax/127) with the f32 quotient
    assert (d16 == O.f32_to_f16_bits((amax / np.float32(127)).astype(np.float32))).all()
    # the largest-magnitude value maps to +-127
    imax = np.abs(xb).argmax(-1)
    top = np.take_along_axis(qs.astype(np.int32), imax[..., None], -1)[..., 0]
    sign = np.sign(np.take_along_axis(xb, imax[..., None], -1)[..., 0])
    assert (top == 127 * sign).all()
    # rounding error at most half a step of the f32 scale
    d32 = (amax / np.float32(127)).astype(np.float64)
    err = np.abs(xb.astype(np.float64) - d32[..., None] * qs)
    assert (err <= d32[..., None] * 0.5 * (1 + 1e-6)).all()
    # ds.y is half of the block sum
    ssum = xb.astype(np.float64).sum(-1)
    s = O.f16_bits_to_f32(s16).astype(np.float64)
    assert (np.abs(s - ssum) <= np.abs(ssum) * 2.0 ** -10 + 1e-6).all()


def test_zero_blocks_and_padding(O):
    x = np.zeros((1, 1024), dtype=np.float32)
    x[0, 100] = 3.0
    q8 = O.quantize_q8_1(x, k_padded=2048)
    assert q8.shape == (1, 2048 // 32 * 36)
    d16, s16, qs = _split(q8, 64)
    # block 3 holds the only non-zero value
    nz = [i for i in range(64) if d16[0, i] != 0]
    assert nz == [3]
    assert (qs[0, [i for i in range(64) if i != 3]] == 0).all()
    assert (s16[0, 32:] == 0).all() and (d16[0, 32:] == 0).all()


def test_exact_multiples_roundtrip(O):
    rng = np.random.default_rng(9)
    q = rng.integers(-127, 128, size=(2, 512)).astype(np.int32)
    q[:, ::32] = 127  # every block reaches amax = 127 * 2^-e
    for e in (0, 3, 10):
        x = (q * 2.0 ** -e).astype(np.float32)
        d16, _, qs = _split(O.quantize_q8_1(x), 16)
        assert (qs.reshape(2, -1) == q).all()
        assert (O.f16_bits_to_f32(d16) == np.float32(2.0 ** -e)).all()


def test_division_by_127_identity(O):
    """The GPU quantiser's division-free d = amax/127 (product with the
    rounded reciprocal plus one fma correction) must equal the IEEE quotient.
    Every 61st float bit pattern here (35M values, a few seconds); the
    same function run with stride 1 over [0, 0x7f800000) is the exhaustive
    check and reports no mismatch either.  A planted error -- the correction
    step dropped -- is caught by the same sample."""
    L = O.lib()
    assert L.orc_check_div127(0, 0x7F800000, 61) == 0
    # the first 2^20 patterns (zero and the subnormals) exhaustively
    assert L.orc_check_div127(0, 1 << 20, 1) == 0
    # without the correction (q0 alone) many quotients are off by one ulp
    rcp = np.float32(1.0 / 127.0)
    a = np.random.default_rng(0).uniform(1e-3, 1e3, 100000).astype(np.float32)
    assert ((a * rcp).astype(np.float32) != a / np.float32(127)).sum() > 1000


def _rounded_sum(x, r):
    """fma(x, r, 1.5 * 2^23) in float32: x * r (at most 48 bits) plus the
    constant is formed in float64, where only bits below 2^-29 of the sum can
    be lost; a sum that lands on a half-integer that way is moved back to its
    side of it, so that the second rounding is that of the exact sum."""
    magic = 12582912.0
    p = x.astype(np.float64) * r.astype(np.float64)  # exact: 24 + 24 bits
    s = p + magic
    lost = p - (s - magic)  # exact
    tie = s - np.floor(s) == 0.5
    s = np.where(tie & (lost > 0), np.nextafter(s, np.inf), s)
    s = np.where(tie & (lost < 0), np.nextafter(s, -np.inf), s)
    return s.astype(np.float32)


def _bounded_round_wrong(d, xs, below, above):
    """The in-launch quantiser's rounding: r any float within one ulp of 1/d
    (the accuracy of v_rcp_f32), the bounds r0 = r (1 - below) and r1 = r
    (1 + above) rounded to float32, one fma with each onto 1.5 * 2^23; where
    both sums agree their low byte is the q8.  Returns (the number of agreeing
    values whose byte differs from ggml's roundf(x / d) with the IEEE
    quotient, the share of values that do not agree)."""
    d = np.float32(d)
    q = np.float32(xs / d)
    q_ref = (np.sign(q) * np.floor(np.abs(q).astype(np.float64) + 0.5)).astype(np.int64) & 0xFF
    near = np.float32(1.0) / d
    wrong, differ = 0, 0
    for r in (near, np.nextafter(near, np.float32(0)), np.nextafter(near, np.float32(np.inf))):
        if abs(float(r) * float(d) - 1.0) > 2.0 ** -23:
            continue  # further than one ulp from 1/d
        m0 = _rounded_sum(xs, np.float32(r * np.float32(1.0 - below))).view(np.uint32)
        m1 = _rounded_sum(xs, np.float32(r * np.float32(1.0 + above))).view(np.uint32)
        same = m0 == m1
        wrong += int(np.sum(same & ((m0 & 0xFF) != q_ref)))
        differ += int(np.sum(~same))
    return wrong, differ / (3 * xs.size)


def _tie_adversaries(rng, d, n=4000):
    """x whose x/d lies within a few units of 2^-20 of a half-integer."""
    k = rng.integers(-127, 127, size=n) + 0.5
    off = rng.integers(-64, 65, size=n) * 2.0 ** -20
    return (np.float32(d) * (k + off)).astype(np.float32)


def test_bounded_rounding_is_safe():
    """quantize_lanes takes a byte only where the sums with both bounds agree:
    r is within 2^-23 of 1/d, the bounds' own rounding and the quotient's are
    2^-24 each, so bounds 1.25 and 1.5 * 2^-22 from r hold the rounded quotient
    strictly between them.  Over random and near-tie quotients, block maxima
    from 2^-100 (below which the kernel divides) to 2^57 and the reciprocals a
    one-ulp rcp can return no agreeing byte is wrong; bounds that allow for
    none of those errors are wrong somewhere; and on ordinary values few
    disagree (the kernel's exact path)."""
    rng = np.random.default_rng(42)
    tight_wrong = 0
    for i in range(300):
        amax = np.float32(2.0 ** rng.uniform(-100, 57))
        d = np.float32(amax / np.float32(127.0))
        plain = rng.uniform(-1, 1, 2000).astype(np.float32) * amax
        xs = np.concatenate([plain, _tie_adversaries(rng, d)]).astype(np.float32)
        xs = xs[np.abs(xs) <= amax]
        assert _bounded_round_wrong(d, xs, 1.25 * 2.0 ** -22, 1.5 * 2.0 ** -22)[0] == 0
        assert _bounded_round_wrong(d, plain, 1.25 * 2.0 ** -22, 1.5 * 2.0 ** -22)[1] < 0.01
        tight_wrong += _bounded_round_wrong(d, xs, 0.0, 2.0 ** -23)[0]
    assert tight_wrong > 0


def test_bounded_rounding_on_generic_ties():
    """The values next to every tie of blocks whose d is no power of two: x
    from a few floats below (k + 1/2) d to a few above, so that the IEEE
    quotient falls on, just under and just over the half-integer."""
    rng = np.random.default_rng(43)
    for _ in range(40):
        d = np.float32(np.float32(2.0 ** rng.uniform(-20, 20)) / np.float32(127.0))
        ties = ((np.arange(-127, 127) + 0.5) * np.float64(d)).astype(np.float32)
        steps = [ties]
        up, down = ties, ties
        for _ in range(6):
            up, down = np.nextafter(up, np.float32(np.inf)), np.nextafter(down, np.float32(-np.inf))
            steps += [up, down]
        xs = np.concatenate(steps)
        assert _bounded_round_wrong(d, xs, 1.25 * 2.0 ** -22, 1.5 * 2.0 ** -22)[0] == 0
