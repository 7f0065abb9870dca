"""The exact fp16 / fp32 identities the prefill GEMM's operand builds rely on
(csrc/mcpm_prefill.hip), checked exhaustively on the CPU: every scale, code
and field position the Q4_K and Q6_K formats allow.  A byte permute reads a
code byte t as the fp16 number 1024 + t; one fused multiply-add then forms
the weight operand, a code times its sub-block scale over 64, which meets an
activation code times 64.  The constants and masks are read from the kernel's
source, so that it cannot change without these checks.  Each check computes
the fused operation exactly (float64 holds every intermediate here exactly) and
rounds once to fp16, as v_pk_fma_f16 does, and compares with the exact product
the reference's integer arithmetic uses."""
import os
import re

import numpy as np

from conftest import ROOT

F16 = np.float16
SRC = open(os.path.join(ROOT, "minicpm5.cpp_amd", "csrc", "mcpm_prefill.hip")).read()


def r16(x):
    """Round a float64 (exact here) once to fp16, back to float64."""
    return np.float64(F16(x))


def fma16(a, b, c):
    return r16(np.float64(a) * np.float64(b) + np.float64(c))


def const(pattern):
    """The numbers at the groups of the one place in the kernel that matches."""
    m = re.findall(pattern, SRC)
    assert len(m) == 1, f"{pattern}: {len(m)} places in the kernel"
    return [float(v) if "." in v else int(v, 16) for v in (m[0] if isinstance(m[0], tuple) else (m[0],))]


def splat(*values):
    """splat2's conversion to fp16; every constant has to be exact in it."""
    assert all(r16(v) == v for v in values)
    return values


N = r"(-?[0-9.]+)f"
X = r"(0x[0-9a-f]+)u"
[X_SCALE] = const(rf"static_cast<_Float16>\({N} \* static_cast<float>\(static_cast<int8_t>")


def test_activation_operands_exact():
    """Codes -127..127 (the quantizers clamp to them) times 64, and sums of 16 of them, are exact in fp16."""
    assert X_SCALE == 64
    for x in range(-127, 128):
        assert r16(X_SCALE * x) == 64 * x
    for bs in range(-16 * 127, 16 * 127 + 1):
        assert r16(bs) == bs


def test_q4k_operands_exact():
    """Q4_K, scales 0..63: sc/64 and sc/1024 from fp16 1024 + sc, offsets -1024 times them; low nibble t = q,
    high nibble read in place t = 16q: the operand is q*sc/64 for every q, and times 64 x the integer q*sc*x."""
    a1, a2 = splat(*const(rf"sa = __builtin_elementwise_fma\(ha, splat2\({N}\), splat2\({N}\)\)"))
    b1, b2 = splat(*const(rf"sb = __builtin_elementwise_fma\(hb, splat2\({N}\), splat2\({N}\)\)"))
    am, bm = splat(*const(rf"ma = sa \* splat2\({N}\), mb = sb \* splat2\({N}\)"))
    for sc in range(64):
        s_lo, s_hi = fma16(1024 + sc, a1, a2), fma16(1024 + sc, b1, b2)
        m_lo, m_hi = r16(s_lo * am), r16(s_hi * bm)
        assert (s_lo, s_hi, m_lo, m_hi) == (sc / 64, sc / 1024, -16 * sc, -sc)
        for q in range(16):
            assert fma16(1024 + q, s_lo, m_lo) == fma16(1024 + 16 * q, s_hi, m_hi) == q * sc / 64
            for x in (-127, -1, 1, 126, 127):
                assert np.float64(q * sc / 64) * (X_SCALE * x) == q * sc * x


def test_q4k_scale_and_min_fields():
    """The lane's scale and min bytes, masked without a branch, are the format's sub-block scales 2g, 2g+1 and
    mins 4g .. 4g+3 (K-halves 0 and 1; 0 in the others), and 1024 + mn - 1024 is mn."""
    num = r"([0-9a-fx]+)u"
    sh4 = re.search(rf"sh4 = g < 2 \? {num} : {num}, m4a = g < 2 \? {num} : {num}, m4b = g < 2 \? {num} : {num};", SRC)
    shm = re.search(rf"shm = g == 1 \? {num} : {num}, mma = g == 0 \? {num} : g == 1 \? {num} : {num},\s+mmb = g == 1 \? {num} : {num};", SRC)
    assert sh4 and shm
    assert "const uint32_t sw = ((s0 >> sh4) & m4a) | (s2 & m4b);" in SRC
    assert "const uint32_t mw = ((s1 >> shm) & mma) | ((s2 >> 4) & mmb);" in SRC
    assert "sel4a = 0x04000400u | (0x00010001u * 2u * (g & 1)), sel4b = sel4a + 0x00010001u;" in SRC
    assert "const h2 o1024 = splat2(1024.0f);" in SRC
    c = [int(v, 0) for v in sh4.groups()]
    d = [int(v, 0) for v in shm.groups()]
    rng = np.random.default_rng(3)
    raws = [rng.integers(0, 256, 12) for _ in range(2000)] + [np.full(12, v) for v in (0, 0x0f, 0x3f, 0x40, 0x80, 0xc0, 0xf0, 0xff)]
    for raw in raws:
        b = [int(v) for v in raw]
        sc = [b[j] & 63 if j < 4 else (b[j + 4] & 15) | (b[j - 4] >> 6) << 4 for j in range(8)]
        mn = [b[j + 4] & 63 if j < 4 else b[j + 4] >> 4 | (b[j] >> 6) << 4 for j in range(8)]
        s0, s1, s2 = (int.from_bytes(bytes(b[4 * i:4 * i + 4]), "little") for i in range(3))
        for g in range(4):
            sw = ((s0 >> c[0 if g < 2 else 1]) & c[2 if g < 2 else 3]) | (s2 & c[4 if g < 2 else 5])
            byte = lambda w, i: w >> 8 * i & 255
            assert [byte(sw, 2 * (g & 1)), byte(sw, 2 * (g & 1) + 1)] == sc[2 * g:2 * g + 2]
            mw = ((s1 >> d[0 if g == 1 else 1]) & d[2 if g == 0 else 3 if g == 1 else 4]) | ((s2 >> 4) & d[5 if g == 1 else 6])
            assert [byte(mw, i) for i in range(4)] == (mn[4 * g:4 * g + 4] if g < 2 else [0] * 4)
    for m in range(64):
        assert r16(np.float64(1024 + m) - 1024) == m


def test_q6k_operands_exact():
    """Q6_K, signed scales -128..127 as u = sc + 128: a field at bit p of its
    byte reads as t = code*2^p and takes s = sc*2^-p/64 = (1024 + u)*(2^-p/64)
    - 18*2^-p and m = -16*sc*2^-p = (1024 + u)*(-16*2^-p) + 18432*2^-p; then
    fma(1024 + t, s, m) == code*sc/64 for the low nibbles (p = 0, 4) and the
    2-bit high fields (p = 0, 2, 4, 6), times 64 x an integer."""
    fl1, fl0, fa1, fa0 = const(rf"fl = odd \? {N} : {N}, fa = odd \? {N} : {N};")
    sl = const(rf"sl1 = splat2\(fl \* {N}\), sl2 = splat2\({N} \* fl\), ol1 = splat2\({N} \* fl\), ol2 = splat2\({N} \* fl\)")
    sa = const(rf"sa1 = splat2\(fa \* {N}\), sa2 = splat2\({N} \* fa\), oa1 = splat2\({N} \* fa\), oa2 = splat2\({N} \* fa\)")
    assert (fl0, fl1, fa0, fa1) == (1.0, 2.0 ** -4, 2.0 ** -2, 2.0 ** -6)
    # low nibbles and the high codes' first field at bit 0 or 4, their second at bit 2 or 6
    fields = [(0, 16, fl0, sl), (4, 16, fl1, sl), (0, 4, fl0, sl), (4, 4, fl1, sl), (2, 4, fa0, sa), (6, 4, fa1, sa)]
    o1, o2 = splat(*const(rf"ac = h2bits\(__builtin_elementwise_fma\(hp, splat2\({N}\), splat2\({N}\)\)\)"))
    for sc in range(-128, 128):
        h = 1024 + sc + 128
        for p, codes, f, k in fields:
            assert f == 2.0 ** -p
            c1, c2, m1, m2 = splat(f * k[0], k[1] * f, k[2] * f, k[3] * f)
            s, m = fma16(h, c1, c2), fma16(h, m1, m2)
            assert s == sc * f / 64 and m == -16 * sc * f
            for q in range(codes):
                assert fma16(1024 + q * 2 ** p, s, m) == q * sc / 64
                for x in (-127, -1, 127):
                    assert np.float64(q * sc / 64) * (X_SCALE * x) == q * sc * x
        # the offset operand's pair entries
        assert fma16(h, o1, o2) == -2 * sc


def test_sums_stay_exact_in_fp32():
    """An MFMA's sum over a lane group's 32 bytes (or the 16 bsums) is an integer below 2^24 at every step,
    whatever the order: the terms' magnitudes add up to less."""
    x, bs = 127, 16 * 127
    assert 32 * 15 * 63 * x < 2 ** 24              # Q4_K's isum
    assert 16 * 63 * bs < 2 ** 24                  # Q4_K's min sum
    assert 32 * 15 * 128 * x < 2 ** 23             # Q6_K's S: low nibbles
    assert 32 * 3 * 128 * x + 2 * 2 * 128 * bs < 2 ** 22  # Q6_K's T: high fields and the offset pair


def test_q6k_split_is_the_reference_sum():
    """fma(16, T, S), rounded once, is the reference's int32 lane sum sum(sc*q*x) - 32*C converted to float, at
    random blocks and at the extremes."""
    assert re.search(r"__builtin_fmaf\(16\.0f, T\[j\]\[i\], S\[j\]\[i\]\)", SRC)
    rng = np.random.default_rng(7)
    cases = [(rng.integers(-128, 128, 16), rng.integers(0, 64, 32), rng.integers(-127, 128, 256)) for _ in range(3000)]
    for sc in (-128, 127):
        for q in (0, 15, 48, 63):
            for x in (-127, 127):
                cases.append((np.full(16, sc), np.full(32, q), np.full(256, x)))
    for i, (sc, q, x) in enumerate(cases):
        m = i % 8  # lane group m: bytes 4m .. 4m+3 of each 32-byte group, 16-value sub-block 2s + m/4
        xl = np.concatenate([x[32 * s + 4 * m:32 * s + 4 * m + 4] for s in range(8)])
        scl = np.repeat(sc[[2 * s + m // 4 for s in range(8)]], 4)
        bs = x.reshape(16, 16).sum(axis=1)
        C = int(sc[2 * m] * bs[2 * m] + sc[2 * m + 1] * bs[2 * m + 1])
        want = int((scl * q * xl).sum()) - 32 * C
        S = int((scl * (q & 15) * xl).sum())
        T = int((scl * (q >> 4) * xl).sum()) - 2 * C
        assert abs(S) < 2 ** 23 and abs(T) < 2 ** 22
        assert np.float32(np.float64(16) * T + S) == np.float32(np.int32(want))
