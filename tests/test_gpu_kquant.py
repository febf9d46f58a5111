"""Q4_K / Q6_K on the GPU (woolly_gguf::dequantize, dequantize.rs:380-536):
dequantization bit for bit against the oracle and the closed forms the oracle
is pinned on, ragged element counts, unaligned outputs, every byte random (f16
fields included), the short-data error; the GEMV (dequantize-then-dot, no
reference kernel) against the f64 oracle at the north-star bar."""
import numpy as np
import pytest

from tests._gpu import down, gemv, up
from tests._oracle import max_abs, rel_l2
from tests.test_oracle_kquant import f16b, np_q4_k, np_q6_k, q4k_block, q6k_block
from woolly_amd import WoollyHipError, gguf, ops, synth
from woolly_amd.device import DeviceBuffer

pytestmark = pytest.mark.gpu
Q4_K, Q6_K = 12, 14
TS = {Q4_K: 144, Q6_K: 210}


def bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


def same(a, b):
    with np.errstate(invalid="ignore"):
        return np.all((bits(a) == bits(b)) | (np.isnan(a) & np.isnan(b)))


def gpu_dequant(t, data, n, out_offset=0):
    db, dp = up(data)
    ob = DeviceBuffer(4 * n + out_offset + 16)
    ops.dequantize(t, dp, data.nbytes, n, ob.ptr + out_offset)
    return down(ob, np.float32, n, out_offset)


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("n", [1, 255, 256, 257, 4096 + 100, 1 << 20])
def test_kquant_dequant_bit_exact(gpu, orc, t, n):
    print(f"[case] kquant dequant type={t} n={n}", flush=True)
    nb = (n + 255) // 256
    data = synth.quantized_weight(t, nb, 256, seed=n + 7 * t)
    got = gpu_dequant(t, data, n)
    st, ref = orc.dequantize(t, data, n)
    assert st == 0 and same(got, ref)


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("doff,off", [(0, 0), (4, 4), (0, 4), (4, 0), (2, 0), (1, 0)])
@pytest.mark.parametrize("blocks,tail", [(8192, 0), (8193, 0), (16384, 0), (16385, -3), (24577, -1)])
def test_kquant_dequant_passes(gpu, orc, t, doff, off, blocks, tail):
    """Around the blocks of one and two passes of the whole grid (256 CUs x 8
    workgroups x 4 wavefronts), with partial last blocks and quads; blocks of
    all byte values, data (doff) and output (off) 16-byte aligned or past it,
    each by itself."""
    n = 256 * blocks + tail
    data = np.random.default_rng(blocks + t).integers(0, 256, blocks * TS[t], dtype=np.uint8)
    db, dp = up(data, offset=doff)
    ob = DeviceBuffer(4 * n + off + 16)
    ops.dequantize(t, dp, data.nbytes, n, ob.ptr + off)
    st, ref = orc.dequantize(t, data, n)
    assert st == 0 and same(down(ob, np.float32, n, off), ref)


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
def test_kquant_dequant_random_bytes_unaligned_out(gpu, orc, t):
    """Every byte random (d / dmin may be NaN, inf or subnormal); output at a
    4-byte (not 16-byte) aligned address."""
    rng = np.random.default_rng(11 + t)
    n = 300 * 256 - 5
    data = rng.integers(0, 256, 300 * TS[t], dtype=np.uint8)
    got = gpu_dequant(t, data, n, out_offset=4)
    st, ref = orc.dequantize(t, data, n)
    assert st == 0 and same(got, ref)
    assert same(got, (np_q4_k if t == Q4_K else np_q6_k)(data)[:n])


def test_kquant_closed_forms_on_gpu(gpu):
    # Q4_K 6-bit scale packing: scales 5, 14, 10, 23, 17, 61, 63, 50 per 32 elements
    sb = np.array([0x05, 0x87, 0x03, 0x0A, 0xC0, 0x05, 0x11, 0x40, 0x0F, 0x3F, 0x80, 0x0C], np.uint8)
    v = gpu_dequant(Q4_K, q4k_block(sb, 1.0, 0.0, np.full(128, 0x11, np.uint8)), 256)
    assert v.reshape(8, 32)[:, 0].tolist() == [5.0, 14.0, 10.0, 23.0, 17.0, 61.0, 63.0, 50.0]
    # even elements take the low nibble, dmin added last
    v = gpu_dequant(Q4_K, q4k_block(np.full(12, 0xFF, np.uint8), 0.5, 0.25, np.full(128, 0x21, np.uint8)), 256)
    assert np.all(v[0::2] == np.float32(31.75)) and np.all(v[1::2] == np.float32(63.25))
    # Q6_K: qh = 0xFF gives q = 48 everywhere except the last element (q = 0)
    v = gpu_dequant(Q6_K, q6k_block(np.zeros(128, np.uint8), np.full(64, 0xFF, np.uint8),
                                    np.ones(16, np.uint8), 0.5), 256)
    assert np.all(v[:255] == np.float32(0.125)) and v[255] == np.float32(-0.25)
    # unsigned scales
    v = gpu_dequant(Q6_K, q6k_block(np.zeros(128, np.uint8), np.zeros(64, np.uint8),
                                    np.full(16, 0xC8, np.uint8), 0.5), 256)
    assert np.all(v == np.float32(-50.0))


def test_kquant_short_data_is_invalid_tensor_info(gpu):
    with pytest.raises(gguf.InvalidTensorInfo):
        gguf.dequantize(np.zeros(2 * 144 - 1, np.uint8), gguf.GGMLType.Q4_K, 257)
    v = gguf.dequantize(synth.quantized_weight(Q6_K, 2, 256, seed=5), gguf.GGMLType.Q6_K, 300)
    assert v.shape == (300,)


# (m, k): ragged row counts, one to 56 blocks per row
GEMV_SHAPES = [(1, 256), (63, 512), (300, 4096), (1024, 4096), (97, 14336)]


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("m,k", GEMV_SHAPES)
def test_kquant_gemv_parity(gpu, orc, t, m, k):
    print(f"[case] kquant gemv type={t} m={m} k={k}", flush=True)
    w = synth.quantized_weight(t, m, k, seed=m + k + t)
    x = synth.activations(k, seed=m * 5 + k)
    got = gemv(t, w, x, m, k)
    ref = orc.matvec_f64(t, w, x, m, k)[1]
    r, a = rel_l2(got, ref), max_abs(got, ref)
    print(f"[result] kquant t={t} {m}x{k} rel_l2={r:.3e} max_abs={a:.3e}", flush=True)
    assert r <= 1e-4 and a <= 1e-3


def test_kquant_gemv_matches_dequantized_dot(gpu):
    """The GEMV is the dequantization followed by the dot product: the same
    numbers as the GPU's own dequantized matrix times x, within f32 summation."""
    m, k = 200, 2048
    w = synth.quantized_weight(Q6_K, m, k, seed=4)
    x = synth.activations(k, seed=5)
    deq = gpu_dequant(Q6_K, w, m * k).reshape(m, k).astype(np.float64)
    got = gemv(Q6_K, w, x, m, k)
    assert rel_l2(got, deq @ x.astype(np.float64)) <= 1e-6


# K = 2048 .. 16384: 1 .. 4 K-segments of the matrix-core kernel (Q6_K at
# K = 14336: four segments of 14 blocks that start 4, 8, 12 bytes past a
# 16-byte boundary); K = 2560 and 5120 (Q6_K rows not a multiple of 16 bytes)
# run on the simple kernel
MFMA_K = [2048, 2560, 4096, 5120, 8192, 12288, 14336, 16384]


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("k", MFMA_K)
def test_kquant_mfma_matches_simple_kernel(gpu, orc, t, k):
    print(f"[case] kquant mfma type={t} k={k}", flush=True)
    m = 200
    w = synth.quantized_weight(t, m, k, seed=k + t)
    x = synth.activations(k, seed=k + 1)
    got = gemv(t, w, x, m, k)
    prev = ops.gemv_select(ops.GEMV_STREAM)
    try:
        simple = gemv(t, w, x, m, k)
    finally:
        ops.gemv_select(prev)
    ref = orc.matvec_f64(t, w, x, m, k)[1]
    for name, y in (("auto", got), ("simple", simple)):
        r, a = rel_l2(y, ref), max_abs(y, ref)
        print(f"[result] kquant {name} t={t} k={k} rel_l2={r:.3e} max_abs={a:.3e}", flush=True)
        assert r <= 1e-4 and a <= 1e-3
    assert rel_l2(got, simple) <= 1e-5


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("scale", [1e-30, 1e30])
def test_kquant_mfma_activation_scales(gpu, orc, t, scale):
    m, k = 256, 4096
    w = synth.quantized_weight(t, m, k, seed=31)
    x = (synth.activations(k, seed=32) * np.float32(scale)).astype(np.float32)
    got = gemv(t, w, x, m, k)
    ref = orc.matvec_f64(t, w, x, m, k)[1]
    assert rel_l2(got, ref) <= 1e-4


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
def test_kquant_mfma_nonfinite_and_zero_chunks(gpu, orc, t):
    m, k = 128, 4096
    w = synth.quantized_weight(t, m, k, seed=33)
    x = synth.activations(k, seed=34)
    x[:512] = 0.0
    got = gemv(t, w, x, m, k)
    assert rel_l2(got, orc.matvec_f64(t, w, x, m, k)[1]) <= 1e-4
    x[700] = np.inf
    got = gemv(t, w, x, m, k)
    ref = orc.matvec_f32(t, w, x, m, k)[1]
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    fin = ~np.isnan(ref)
    assert np.array_equal(np.isinf(got[fin]), np.isinf(ref[fin]))
    assert np.array_equal(np.sign(got[fin]), np.sign(ref[fin]))


# ---------------------------------------------------------------- prefill
# More than 16 tokens: the matrix is repacked into stage records of 64 elements
# (quants, sub-block scales in fp16, d in f32) and multiplied on the matrix cores.
# (m, n, k): one to 56 super-blocks per row, ragged token and row counts,
# token tiles of 16 .. 128, split-K
KQ_MATMUL = [(3, 300, 4096), (8, 1024, 2048), (17, 768, 256), (64, 129, 4096), (130, 200, 512),
             (257, 384, 1024), (512, 256, 14336)]


# every token tile (32, 64, 128), partial tiles, odd row counts (stage records
# that start 8 bytes off a 16-byte boundary), one super-block per row, and
# tiles shared by two workgroups of the stream-K grid (14337 and 5000 rows)
KQ_EDGES = [(17, 1, 256), (32, 255, 256), (33, 257, 768), (64, 301, 512), (65, 513, 2304), (128, 1001, 1024),
            (129, 14337, 256), (257, 5000, 1280),
            # 7 and 8 super-blocks per workgroup and tile: products accumulated over 64 and over 128 elements
            (300, 2560, 14336), (300, 2561, 14336)]


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("m,n,k", KQ_EDGES)
def test_kquant_matmul_edges(gpu, orc, t, m, n, k):
    """Per-output error of about k roundings of f32 sums of the terms' size:
    rel-L2 <= 2e-6 with f32 activations, whose lo limbs carry bits (without
    them 1e-4); bfloat16 activations give the widened ones' bits."""
    print(f"[case] kquant edges type={t} m={m} n={n} k={k}", flush=True)
    w = synth.quantized_weight(t, n, k, seed=n + k + t)
    x = synth.activations(m * k, seed=m + t).reshape(m, k)
    rows = sorted({0, m // 2, m - 1})
    ref = orc.matmul_rows_f64(t, w, n, k, x, m, np.array(rows))
    assert rel_l2(kq_matmul(t, w, x, m, n, k)[rows], ref) <= 2e-6
    xw = (x.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)  # bf16 values
    assert np.array_equal(kq_matmul_bf16(t, w, xw, m, n, k), kq_matmul(t, w, xw, m, n, k))


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("m,n,k", [(64, 256, 2048), (30, 512, 1024), (100, 300, 1024), (300, 2561, 14336)])
def test_kquant_matmul_bf16_wide_range(gpu, orc, t, m, n, k):
    """bf16 rows spanning 2^-60 .. 2^4, zeros and a row of only tiny values
    among them: the hi limbs alone give the bits of the widened f32 call (an
    element below 2^-17 of the scaled row rounds to an fp16 subnormal, and what
    is left of it, at most half of the smallest subnormal, rounds to 0)."""
    rng = np.random.default_rng(77 + t)
    w = synth.quantized_weight(t, n, k, seed=5 + t)
    x = (np.exp2(rng.uniform(-60.0, 4.0, size=(m, k))) * rng.choice([-1.0, 1.0], size=(m, k))).astype(np.float32)
    x[:, ::97] = 0.0
    x[1] *= np.float32(2.0 ** -30)
    xw = (x.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)
    got = kq_matmul_bf16(t, w, xw, m, n, k)
    assert np.array_equal(got, kq_matmul(t, w, xw, m, n, k))
    rows = sorted({0, 1, m // 2, m - 1})
    for r, ref in zip(rows, orc.matmul_rows_f64(t, w, n, k, xw, m, np.array(rows))):
        assert rel_l2(got[r], ref) <= 2e-6


@pytest.mark.parametrize("m,n,k", [(40, 512, 1024), (100, 512, 1024), (300, 8448, 1024), (130, 2560, 14336)])
def test_q6k_products_of_one_sign(gpu, orc, m, n, k):
    """Scales of 255 and quants at the ends (+-8160), and 137 x 30 = 4110, whose
    fp16 rounding is 2 off, against activations half a ulp of fp16 off: every
    product of a row has one sign, and so has x_lo w_lo, at most 2^-22 of x w.
    The first two shapes, sums of one super-block, form it, the others leave it
    out.  Each output within a rounding per 64 elements, and 2^-22 for those."""
    w = np.zeros((n, k // 256, 210), np.uint8)
    w[..., 192:208] = 255
    w[1::3, :, 192:208] = 137
    # q - 32 = -32 (all bits clear); 30 with scale 137; 31.  Byte 191's missing high
    # pair makes element 255 a quant of 0..15: its group's scale is 0
    w[1::3, :, 0:128] = 0xEE
    w[2::3, :, 0:128] = 0xFF
    w[1::3, :, 128:192] = 0xFF
    w[2::3, :, 128:192] = 0xFF
    w[..., 207] = 0
    w[..., 208:210] = f16b(2.0 ** -10)
    x = np.full((m, k), 1 + 2.0 ** -11, np.float32)
    x[1::2] *= np.float32(-3.0)
    got = kq_matmul(Q6_K, w.reshape(-1), x, m, n, k)
    rows = np.array(sorted({0, 1, m // 2, m - 1}))
    ref = orc.matmul_rows_f64(Q6_K, w.reshape(-1), n, k, x, m, rows)
    err = np.max(np.abs(got[rows] - ref) / np.abs(ref))
    print(f"[result] q6_k one sign m={m} n={n} k={k} err={err:.3e}", flush=True)
    # short: 16 f32 roundings that grow with the sum to at most 2^-24 of it, 2^-25 rms each
    assert err <= (1.2e-7 if n == 512 else 2.0 ** -22 + k / 64 * 2.0 ** -24)


# one to three super-blocks per workgroup, in tiles of 32, 64 and (Q4_K) 128 tokens
KQ_SHORT = [(20, 2048, 1024), (50, 1024, 2048), (64, 2048, 1024), (100, 2048, 1024), (150, 3000, 2816), (130, 4096, 1280)]


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("m,n,k", KQ_SHORT)
def test_kquant_short_sums(gpu, orc, t, m, n, k):
    """Short sums hide no rounding.  In units of one f32 rounding of a normal
    variate (2.53e-8 rms, relative): the 22-bit activations add 5.6, the f32
    sum of a super-block's four chains 2.2, the planes' 1, and the matrix cores,
    which round four times per product at the size of the chain, 4.8 with the lo
    limbs first: sqrt(13.6) = 0.93e-7.  Two products of lo limbs between the x_hi
    w_hi of a chain's steps make that 8.5: 1.05e-7, and x_lo w_lo left out 1.08e-7."""
    w = synth.quantized_weight(t, n, k, seed=n + k + t)
    x = synth.activations(m * k, seed=m + t).reshape(m, k)
    r = rel_l2(kq_matmul(t, w, x, m, n, k), orc.matmul_rows_f64(t, w, n, k, x, m, np.arange(m)))
    print(f"[result] kquant short sums t={t} m={m} n={n} k={k} rel_l2={r:.3e}", flush=True)
    assert r <= 1.04e-7


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
def test_kquant_nonfinite_scales(gpu, orc, t):
    """A block scale d of inf (in a block with zero quants) or NaN makes its
    row NaN, as (d * s) * q does where s or q is 0; the other rows are untouched."""
    m, n, k = 40, 96, 1024
    w = synth.quantized_weight(t, n, k, seed=5 + t).reshape(n, -1, TS[t]).copy()
    x = synth.activations(m * k, seed=6).reshape(m, k)
    base = kq_matmul(t, w.reshape(-1), x, m, n, k)
    at = 12 if t == Q4_K else 208
    w[7, 2, at:at + 2] = f16b(np.inf)
    w[50, 0, at:at + 2] = f16b(np.nan)
    got = kq_matmul(t, w.reshape(-1), x, m, n, k)
    assert np.all(np.isnan(got[:, [7, 50]]))
    rest = [r for r in range(n) if r not in (7, 50)]
    assert np.array_equal(got[:, rest], base[:, rest])


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("m", [40, 130])
def test_kquant_infinite_scales(gpu, orc, t, m):
    """d of +-inf in a block without a zero scale or quant: the row is +-inf
    where every product has one sign, as in the reference; NaN with one zero
    quant or scale anywhere in the block, or with products of both signs."""
    n, k = 96, 1024
    w = synth.quantized_weight(t, n, k, seed=15 + t).reshape(n, -1, TS[t]).copy()
    x = np.abs(synth.activations(m * k, seed=16)).reshape(m, k) + np.float32(0.01)
    rng = np.random.default_rng(t)

    def block(d):
        if t == Q4_K:
            return q4k_block(np.full(12, 0xFF, np.uint8), d, 0.5, rng.integers(1, 16, 128, dtype=np.uint8) * 17)
        # no high bits: q - 32 is -32 .. -17 (the last element has no other choice)
        return q6k_block(rng.integers(0, 256, 128, dtype=np.uint8), np.zeros(64, np.uint8),
                         rng.integers(1, 256, 16, dtype=np.uint8), d)

    rows = [3, 7, 20, 21, 22, 60, 95]
    plain = w.copy()
    for i, r in enumerate(rows):
        b = block(-np.inf if r == 7 else np.inf)
        if i == 2:                     # a zero quant (Q6_K: 32) among the first 64 elements
            if t == Q4_K:
                b[16] = 0x10
            else:
                b[0], b[128] = 0, 0x02
        elif i == 3:                   # among the last 64 (Q6_K: element 250)
            if t == Q4_K:
                b[143] = 0x01
            else:
                b[122], b[190] = 0, 0x80
        elif i == 4:                   # a zero scale
            if t == Q4_K:
                b[0] &= 0xC0
            else:
                b[207] = 0
        elif i == 5:                   # 64 elements' products of the other sign
            x[:, 768:832] *= -1
        w[r, (0, 1, 2, 3, 0, 3, 2)[i]] = b
    base = kq_matmul(t, plain.reshape(-1), x, m, n, k)
    got = kq_matmul(t, w.reshape(-1), x, m, n, k)
    for tok in (0, m - 1):
        with np.errstate(all="ignore"):
            ref = orc.matvec_f32(t, w.reshape(-1), x[tok], n, k)[1]
        assert np.array_equal(np.isnan(got[tok]), np.isnan(ref))
        inf = np.isinf(ref)
        assert inf[[3, 7]].all() and np.array_equal(got[tok][inf], ref[inf])
    rest = [r for r in range(n) if r not in rows]
    assert np.array_equal(got[:, rest], base[:, rest])


def kq_matmul(t, w, x, m, n, k, w_offset=0):
    wb, wp = up(w, offset=w_offset)
    xb, xp = up(x)
    yb = DeviceBuffer(4 * m * n)
    wsz = ops.matmul_workspace_bytes(t, n, k, m)
    ws = DeviceBuffer(max(wsz, 1))
    ops.quantized_matmul(t, wp, w.nbytes, n, k, xp, m, yb.ptr, ws, wsz)
    return down(yb, np.float32, m * n).reshape(m, n)


def kq_matmul_bf16(t, w, xw, m, n, k):
    """xw: f32 values that bfloat16 holds exactly."""
    wb, wp = up(w)
    xb, xp = up((xw.view(np.uint32) >> 16).astype(np.uint16))
    yb = DeviceBuffer(4 * m * n)
    wsz = ops.matmul_x_workspace_bytes(t, n, k, m, ops.TYPE_BF16)
    ws = DeviceBuffer(wsz)
    ops.quantized_matmul_x(t, wp, w.nbytes, n, k, xp, ops.TYPE_BF16, m, yb.ptr, ws, wsz)
    return down(yb, np.float32, m * n).reshape(m, n)


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("m,n,k", KQ_MATMUL)
def test_kquant_matmul_parity(gpu, orc, t, m, n, k):
    print(f"[case] kquant matmul type={t} m={m} n={n} k={k}", flush=True)
    w = synth.quantized_weight(t, n, k, seed=n + k + t)
    x = synth.activations(m * k, seed=m + t).reshape(m, k)
    got = kq_matmul(t, w, x, m, n, k)
    ref = orc.matmul_rows_f64(t, w, n, k, x, m, np.arange(m))
    r, a = rel_l2(got, ref), max_abs(got, ref)
    print(f"[result] kquant matmul t={t} rel_l2={r:.3e} max_abs={a:.3e}", flush=True)
    assert r <= 2e-6 and a <= 1e-3   # k roundings of f32 sums, as test_kquant_matmul_edges


@pytest.mark.parametrize("t,rows_per_group", [(Q4_K, 64), (Q6_K, 32)])
def test_kquant_repack_many_row_groups(gpu, t, rows_per_group):
    """A matrix with more row groups than a grid has in y (65535), one
    super-block per row: its last rows give the bits of the same rows alone."""
    m, k, base = 17, 256, 1024
    n = rows_per_group * 65536 + 37
    print(f"[case] kquant repack type={t} n={n}", flush=True)
    part = synth.quantized_weight(t, base, k, seed=600 + t).reshape(base, TS[t])
    w = part[np.arange(n) % base]
    x = synth.activations(m * k, seed=601).reshape(m, k)
    last = np.arange(n - base, n)
    got = kq_matmul(t, w.reshape(-1), x, m, n, k)
    assert same(np.ascontiguousarray(got[:, last]), kq_matmul(t, w[last].reshape(-1), x, m, base, k))
    assert same(np.ascontiguousarray(got[:, :base]), kq_matmul(t, part.reshape(-1), x, m, base, k))


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
def test_kquant_matmul_matches_gemv(gpu, t):
    """The several-token path (5 tokens) and the per-token GEMV agree on every token."""
    m, n, k = 5, 520, 4096
    w = synth.quantized_weight(t, n, k, seed=77 + t)
    x = synth.activations(m * k, seed=78).reshape(m, k)
    got = kq_matmul(t, w, x, m, n, k)
    for i in range(m):
        assert rel_l2(got[i], gemv(t, w, x[i], n, k)) <= 1e-5


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("hidden,n_ff,m", [(256, 512, 1), (512, 1024, 4), (4096, 1024, 64), (256, 20480, 5),
                                          (256, 768, 70), (512, 20480, 257), (4096, 14336, 130),
                                          (1024, 4096, 1000), (1792, 4096, 900)])
def test_kquant_ffn_parity(gpu, orc, t, hidden, n_ff, m):
    """The SwiGLU FFN layer on K-quant weights: decode (fused gate/up GEMV) and
    prefill (RMSNorm packed into the GEMM's activations, SwiGLU in the epilogue
    of gate and up in one pass or in the second packing, matrices repacked into
    the workspace)."""
    print(f"[case] kquant ffn t={t} hidden={hidden} n_ff={n_ff} m={m}", flush=True)
    L = synth.ffn_layer(t, hidden, n_ff, m, seed=hidden + n_ff + t)
    bufs = {name: up(v) for name, v in L.items()}
    ob = DeviceBuffer(4 * m * hidden)
    wsz = ops.ffn_workspace_bytes(hidden, n_ff, m, ggml_type=t)
    ws = DeviceBuffer(wsz)
    ops.ffn_swiglu(t, bufs["gate"][1], bufs["up"][1], bufs["down"][1], hidden, n_ff,
                   bufs["gamma"][1], 1e-5, bufs["x"][1], m, ob.ptr, ws.ptr, wsz)
    got = down(ob, np.float32, m * hidden).reshape(m, hidden)
    rows = sorted({0, m // 2, m - 1})
    ref = orc.ffn_rows_f64(t, L["gate"], L["up"], L["down"], hidden, n_ff, L["gamma"], 1e-5, L["x"], rows)
    r, a = rel_l2(got[rows], ref), max_abs(got[rows], ref)
    rms = float(np.sqrt(np.mean(ref ** 2)))
    print(f"[result] kquant ffn rel_l2={r:.3e} max_abs={a:.3e} rms={rms:.3e}", flush=True)
    # two products behind each other, 2e-6 each as test_kquant_matmul_edges
    assert r <= 4e-6 and a <= 1e-3 * max(1.0, rms / 300.0)


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("hidden,n_ff,m", [(4096, 14336, 130), (512, 20480, 257)])
def test_kquant_ffn_workspace_sizes(gpu, orc, t, hidden, n_ff, m):
    """Gate and up run in one pass here.  A workspace with room for one
    converted matrix at a time is enough (unprepared matrices then run one after
    the other where the scratch does not hold both); prepared handles give the
    same bits in it as in the queried size; a byte less is refused."""
    print(f"[case] kquant ffn workspace t={t} hidden={hidden} n_ff={n_ff} m={m}", flush=True)
    up256 = lambda v: (v + 255) // 256 * 256
    conv = lambda n, k: up256(n * (k // 32 * 20 + (k // 256 + 7) // 8 * 8 * 2) if t == Q4_K else n * k // 16 * 20)
    rest = [ops.matmul_workspace_bytes(t, *nk, m) - conv(*nk) for nk in ((n_ff, hidden), (hidden, n_ff))]
    least = up256(4 * m * hidden) + 3 * up256(4 * m * n_ff) + max(conv(n_ff, hidden), conv(hidden, n_ff)) + max(rest)
    full = ops.ffn_workspace_bytes(hidden, n_ff, m, ggml_type=t)
    # the query's extra: gate and up side by side, beyond the scratch that the one pass leaves
    assert full == least + max(0, 2 * conv(n_ff, hidden) - 2 * up256(4 * m * n_ff) - max(conv(n_ff, hidden), conv(hidden, n_ff)))
    L = synth.ffn_layer(t, hidden, n_ff, m, seed=hidden + n_ff + t)
    bufs = {name: up(v) for name, v in L.items()}

    def run(ptrs, wsz):
        ob, ws = DeviceBuffer(4 * m * hidden), DeviceBuffer(wsz)
        ops.ffn_swiglu(t, *ptrs, hidden, n_ff, bufs["gamma"][1], 1e-5, bufs["x"][1], m, ob.ptr, ws.ptr, wsz)
        return down(ob, np.float32, m * hidden).reshape(m, hidden)

    plain = [bufs[n][1] for n in ("gate", "up", "down")]
    base = run(plain, full)
    rows = sorted({0, m // 2, m - 1})
    ref = orc.ffn_rows_f64(t, L["gate"], L["up"], L["down"], hidden, n_ff, L["gamma"], 1e-5, L["x"], rows)
    for got in (base, run(plain, least)):
        assert rel_l2(got[rows], ref) <= 4e-6   # two products behind each other, 2e-6 each as above
    with pytest.raises(WoollyHipError) as e:
        run(plain, least - 1)
    assert e.value.status == 3
    hw = [ops.Weight(t, *((n_ff, hidden) if n != "down" else (hidden, n_ff)), L[n]) for n in ("gate", "up", "down")]
    for h in hw:
        h.prepare_prefill()
    for wsz in (full, least):
        assert same(run([h.ptr for h in hw], wsz), base)
    # one prepared, the other converted in the scratch
    assert same(run([hw[0].ptr, plain[1], hw[2].ptr], full), base)
    assert same(run([plain[0], hw[1].ptr, plain[2]], full), base)
    for h in hw:
        h.free()


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
def test_kquant_matmul_unaligned_weights(gpu, orc, t):
    """Weights 4 bytes past a 16-byte boundary cannot be repacked with 16-byte
    loads: the call takes one GEMV per token instead, same results."""
    m, n, k = 6, 256, 2048
    w = synth.quantized_weight(t, n, k, seed=91 + t)
    x = synth.activations(m * k, seed=92).reshape(m, k)
    got = kq_matmul(t, w, x, m, n, k, w_offset=4)
    ref = orc.matmul_rows_f64(t, w, n, k, x, m, np.arange(m))
    assert rel_l2(got, ref) <= 1e-4 and max_abs(got, ref) <= 1e-3
    assert rel_l2(got, kq_matmul(t, w, x, m, n, k)) <= 1e-5


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
def test_kquant_prepared_prefill(gpu, orc, t):
    """wh_weight_prepare_prefill converts a handle's blocks once (the reference's
    convert-once cache, dequantization_cache.rs:121-165); matmul and FFN calls
    on the handle's data then skip the per-call conversion and give the same
    bits as the converting call, at the north-star bar against the f64 oracle.
    Preparing again is a no-op; a Q4_0 handle needs no copy."""
    m, n, k = 64, 512, 4096
    w = synth.quantized_weight(t, n, k, seed=500 + t)
    x = synth.activations(m * k, seed=501).reshape(m, k)
    plain = kq_matmul(t, w, x, m, n, k)
    wh = ops.Weight(t, n, k, w)
    size = wh.prepare_prefill()
    # 40 or 80 bytes per 64 elements; Q4_K: then the fp16 dmin table with rows of k / 256 rounded up to 8
    assert size == (n * (k // 32 * 20 + (k // 256 + 7) // 8 * 8 * 2) if t == Q4_K else n * k // 16 * 20)
    assert wh.prepare_prefill() == size
    xb, xp = up(x)
    yb = DeviceBuffer(4 * m * n)
    wsz = ops.matmul_workspace_bytes(t, n, k, m)
    ws = DeviceBuffer(wsz)
    ops.quantized_matmul(t, wh.ptr, wh.nbytes, n, k, xp, m, yb.ptr, ws, wsz)
    got = down(yb, np.float32, m * n).reshape(m, n)
    assert same(got, plain)
    ref = orc.matmul_rows_f64(t, w, n, k, x, m, np.arange(m))
    assert rel_l2(got, ref) <= 1e-4 and max_abs(got, ref) <= 1e-3
    # the FFN layer with prepared gate / up / down handles against the converting call
    hidden, n_ff, mf = 4096, 1024, 64
    L = synth.ffn_layer(t, hidden, n_ff, mf, seed=510 + t)
    bufs = {name: up(v) for name, v in L.items()}
    wsz = ops.ffn_workspace_bytes(hidden, n_ff, mf, ggml_type=t)
    ws = DeviceBuffer(wsz)
    ob = DeviceBuffer(4 * mf * hidden)
    ops.ffn_swiglu(t, bufs["gate"][1], bufs["up"][1], bufs["down"][1], hidden, n_ff,
                   bufs["gamma"][1], 1e-5, bufs["x"][1], mf, ob.ptr, ws.ptr, wsz)
    base = down(ob, np.float32, mf * hidden)
    hw = {name: ops.Weight(t, *((n_ff, hidden) if name != "down" else (hidden, n_ff)), L[name])
          for name in ("gate", "up", "down")}
    for h in hw.values():
        assert h.prepare_prefill() > 0
    ob2 = DeviceBuffer(4 * mf * hidden)
    ops.ffn_swiglu(t, hw["gate"].ptr, hw["up"].ptr, hw["down"].ptr, hidden, n_ff,
                   bufs["gamma"][1], 1e-5, bufs["x"][1], mf, ob2.ptr, ws.ptr, wsz)
    assert same(down(ob2, np.float32, mf * hidden), base)
    for h in hw.values():
        h.free()
    wh.free()
    q = ops.Weight(2, 64, 256, synth.quantized_weight(2, 64, 256, seed=1))
    assert q.prepare_prefill() == 0
    q.free()
