"""GPU parity of the Q4_0 tile32-compact dequant-GEMM (qattn_q4_matmul, replacing the reference's
compact batch matmul, src/webgpu/quant-matmul.ts:267-307) against the f64 oracle, through the C ABI,
and of its fused gate/up + SwiGLU form (qattn_q4_matmul_swiglu).

Tolerance, per element: the fp32 sum of K exact products (f16 x f16 products are exact in fp32)
errs by at most (K + 2) u32 * sum_k |x_k w_k| (u32 = 2^-24), and the final fp16 rounding by half an
ulp: |y - exact| <= 2^-11 |exact| + (K + 2) 2^-24 (|x| |w|^T) + 2^-25 (fp16 subnormal spacing).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def random_compact(rng, n, k, scale_lo=0.002, scale_hi=0.05):
    """A tile32-compact tensor of random Q4_0 records; rows past n in the last tile stay zero."""
    tiles, kb = -(-n // 32), k // 32
    rec = np.zeros((tiles, kb, 32, 20), np.uint8)
    scales = rng.uniform(scale_lo, scale_hi, size=(tiles, kb, 32)).astype(np.float16)
    scales *= np.where(rng.random(scales.shape) < 0.5, -1, 1).astype(np.float16)
    rec[..., 0:2] = scales.view(np.uint8).reshape(tiles, kb, 32, 2)
    rec[..., 4:20] = rng.integers(0, 256, size=(tiles, kb, 32, 16), dtype=np.uint8)
    flat = rec.reshape(-1, 20)
    rows = (np.arange(tiles)[:, None, None] * 32 + np.arange(32)[None, None, :]).repeat(kb, axis=1).reshape(-1)
    flat[rows >= n] = 0
    return flat.reshape(-1)


def run_q4(ctx, x, packed, k, n, ldx=None, ldy=None):
    m = x.shape[0]
    ldx = k if ldx is None else ldx
    ldy = -(-n // 8) * 8 if ldy is None else ldy
    xs = np.zeros((max(m, 1), ldx), np.float16)
    xs[:m, :k] = x
    bx, bw = ctx.upload(xs.view(np.uint16)), ctx.upload(packed)
    by = ctx.alloc(max(m, 1) * ldy * 2)
    by.fill_u16(0x7E00)  # NaN: every valid element must be written
    ctx.q4_matmul(bx.ptr, m, k, bw.ptr, packed.size, n, by.ptr, ldx=ldx, ldy=ldy)
    ctx.synchronize()
    y = by.read(np.uint16, (max(m, 1), ldy)).view(np.float16)
    for b in (bx, bw, by):
        b.free()
    return y[:m]


def check(oracle, y, x, packed, k, n, label):
    exact = oracle.q4_matmul(x, packed, k, n)
    w = oracle.q40_compact_weights(packed, k, n).astype(np.float64)
    mag = np.abs(x.astype(np.float64)) @ np.abs(w).T
    bound = 2.0 ** -11 * np.abs(exact) + (k + 2) * 2.0 ** -24 * mag + 2.0 ** -25
    got = y[:, :n].astype(np.float64)
    err = np.abs(got - exact)
    print(f"[{label}] max|err| {err.max():.3e}  max err/bound {np.max(err / bound):.3f}", flush=True)
    assert np.isfinite(got).all(), label
    assert (err <= bound).all(), label


@pytest.mark.parametrize("m,k,n", [(1, 32, 1), (130, 96, 70), (64, 128, 128), (257, 2048, 1024),
                                   (33, 3072, 1024), (1280, 1024, 4096)])
def test_q4_matmul_matches_oracle(ctx, oracle, m, k, n):
    rng = np.random.default_rng(m * 7 + k + n)
    packed = random_compact(rng, n, k)
    x = rng.standard_normal((m, k)).astype(np.float16)
    y = run_q4(ctx, x, packed, k, n)
    check(oracle, y, x, packed, k, n, f"q4 {m}x{k}x{n}")


def test_q4_matmul_strides_and_untouched_padding(ctx, oracle):
    rng = np.random.default_rng(1)
    m, k, n = 70, 160, 40
    packed = random_compact(rng, n, k)
    x = rng.standard_normal((m, k)).astype(np.float16)
    y = run_q4(ctx, x, packed, k, n, ldx=k + 24, ldy=n + 8)
    check(oracle, y, x, packed, k, n, "q4 strided")
    assert np.isnan(y[:, n:].astype(np.float32)).all()  # columns past N are not written


def test_q4_matmul_reference_format_vector(ctx, oracle):
    # The reference's packing test (tests/prepacked-format.test.ts:13-22) as weights: row 0 holds
    # q - 8 (scale 1), row 1 holds 2 (7 - q) (scale 2); x = e_j picks column j.
    def block(scale_bits, quants):
        b = bytearray(18)
        b[0:2] = bytes(scale_bits)
        for i in range(16):
            b[2 + i] = quants[i] | (quants[i + 16] << 4)
        return bytes(b)
    first = block([0x00, 0x3C], [i & 15 for i in range(32)])
    second = block([0x00, 0x40], [15 - (i & 15) for i in range(32)])
    packed, k, n = oracle.pack_q40_tile32([(32, 1, first), (32, 1, second)])
    x = np.eye(32, dtype=np.float16)
    y = run_q4(ctx, x, packed, k, n).astype(np.float64)
    assert np.array_equal(y[:, 0], [(j & 15) - 8 for j in range(32)])
    assert np.array_equal(y[:, 1], [2 * (7 - (j & 15)) for j in range(32)])


def run_q4_swiglu(ctx, x, packed, k, n_inter, ldy=None):
    m = x.shape[0]
    ldy = n_inter if ldy is None else ldy
    bx, bw = ctx.upload(np.ascontiguousarray(x).view(np.uint16)), ctx.upload(packed)
    by = ctx.alloc(max(m, 1) * ldy * 2)
    by.fill_u16(0x7E00)
    ctx.q4_matmul_swiglu(bx.ptr, m, k, bw.ptr, packed.size, n_inter, by.ptr, ldy=ldy)
    ctx.synchronize()
    y = by.read(np.uint16, (max(m, 1), ldy)).view(np.float16)
    for b in (bx, bw, by):
        b.free()
    return y[:m]


@pytest.mark.parametrize("m,k,n_inter", [(1, 32, 64), (130, 96, 128), (257, 1024, 3072), (1100, 256, 3072)])
def test_q4_matmul_swiglu_equals_the_two_launches(ctx, oracle, m, k, n_inter):
    """The fused gate/up projection + SwiGLU (one launch) against the launches it replaces: the
    projection into [m, 2 n_inter] (checked against the oracle's product here too), then
    qattn_swiglu -- equal bit for bit -- and within one fp16 step of the f64 SwiGLU restatement
    (oracle/model_ref.py, ops.ts:81-88) of that projection."""
    import model_ref as mr
    rng = np.random.default_rng(m + k + n_inter)
    packed = random_compact(rng, 2 * n_inter, k)
    x = rng.standard_normal((m, k)).astype(np.float16)
    gate_up = run_q4(ctx, x, packed, k, 2 * n_inter)
    check(oracle, gate_up, x, packed, k, 2 * n_inter, f"gate_up {m}x{k}x{2 * n_inter}")
    dg, do = ctx.upload(np.ascontiguousarray(gate_up).view(np.uint16)), ctx.alloc(m * n_inter * 2)
    ctx.swiglu(dg.ptr, do.ptr, m, width=n_inter)
    ctx.synchronize()
    two = do.read(np.uint16, (m, n_inter))
    dg.free()
    do.free()
    fused = run_q4_swiglu(ctx, x, packed, k, n_inter, ldy=n_inter + 8)
    assert np.isnan(fused[:, n_inter:].astype(np.float32)).all()  # columns past n_inter are not written
    assert np.array_equal(fused[:, :n_inter].view(np.uint16), two)
    ref = mr.swiglu(gate_up, n_inter).astype(np.float64)
    got = fused[:, :n_inter].astype(np.float64)
    step = np.maximum(np.spacing(np.maximum(np.abs(got), np.abs(ref)).astype(np.float16)).astype(np.float64), 2.0 ** -24)
    assert (np.abs(got - ref) / step).max() <= 1


def test_q4_rows_do_not_depend_on_the_launch_shape(ctx, oracle):
    """Three kernels serve one projection, chosen by the launch's size: 32-row blocks whose wavefronts
    share K, then tiles of 64 x 128, then of 256 x 128.  Every output element is computed the same
    way in all three (the same K blocks and MFMA order), so rows 0..63 of a 64-row, a 300-row and
    an 1100-row launch are equal bit for bit -- the model's batch invariance rests on this -- for
    the plain and the fused gate/up projections."""
    rng = np.random.default_rng(5)
    k, n = 256, 4096
    packed = random_compact(rng, n, k)
    x = rng.standard_normal((1100, k)).astype(np.float16)
    big = run_q4(ctx, x, packed, k, n)          # 576 tiles of 64 x 128: 256 x 128 tiles
    mid = run_q4(ctx, x[:300], packed, k, n)    # 160 tiles of 64 x 128
    small = run_q4(ctx, x[:64], packed, k, n)   # 256 blocks of 32 x 32
    check(oracle, big, x, packed, k, n, "q4 1100 rows")
    check(oracle, small, x[:64], packed, k, n, "q4 64 rows")
    assert np.array_equal(big[:64].view(np.uint16), small.view(np.uint16))
    assert np.array_equal(mid[:64].view(np.uint16), small.view(np.uint16))
    big_f = run_q4_swiglu(ctx, x, packed, k, n // 2)
    mid_f = run_q4_swiglu(ctx, x[:300], packed, k, n // 2)
    small_f = run_q4_swiglu(ctx, x[:64], packed, k, n // 2)
    assert np.array_equal(big_f[:64].view(np.uint16), small_f.view(np.uint16))
    assert np.array_equal(mid_f[:64].view(np.uint16), small_f.view(np.uint16))


def test_q4_chunked_k_rows_do_not_depend_on_the_launch_shape(ctx, oracle):
    """K = 3072 spans three chunks of 1024 columns, summed in chunk order by every kernel: the
    small kernel with the chunks side by side (64 rows: 256 blocks of 16 x 16), the direct kernel
    with one wavefront folding the chunks in turn (300 rows: 320 blocks of 32 x 32, too many chunk
    wavefronts), 64 x 128 tiles (1100 rows) and 128 x 128 tiles (2600 rows: 168) with a group of
    wavefronts per chunk.  Rows 0..63 agree bit for bit."""
    rng = np.random.default_rng(6)
    k, n = 3072, 1024
    packed = random_compact(rng, n, k)
    x = rng.standard_normal((2600, k)).astype(np.float16)
    small = run_q4(ctx, x[:64], packed, k, n)
    check(oracle, small, x[:64], packed, k, n, "q4 chunked 64 rows")
    for m in (300, 1100, 2600):
        got = run_q4(ctx, x[:m], packed, k, n)
        assert np.array_equal(got[:64].view(np.uint16), small.view(np.uint16)), m
    check(oracle, got[:200], x[:200], packed, k, n, "q4 chunked 2600 rows (first 200)")


def test_q4_matmul_invalid_arguments(ctx, qattn):
    buf = ctx.alloc(1 << 16)
    good = dict(m=4, k=64, n=8, w_bytes=qattn.lib().qattn_q4_compact_bytes(64, 8), ldx=64, ldy=8, x_off=0)
    for bad in (dict(k=48), dict(w_bytes=100), dict(ldx=60), dict(ldy=12), dict(x_off=8), dict(n=0)):
        a = dict(good, **bad)
        with pytest.raises(qattn.QattnError) as e:
            ctx.q4_matmul(buf.ptr + a["x_off"], a["m"], a["k"], buf.ptr, a["w_bytes"], a["n"], buf.ptr,
                          ldx=a["ldx"], ldy=a["ldy"])
        assert e.value.code == qattn.EINVAL, bad
    # the fused entry point: n_inter a multiple of 64, y rows of n_inter, the weight 2 n_inter rows
    w128 = qattn.lib().qattn_q4_compact_bytes(64, 128)
    for n_inter, ldy, w_bytes in ((32, 64, w128), (96, 96, qattn.lib().qattn_q4_compact_bytes(64, 192)), (64, 56, w128),
                                  (64, 64, w128 - 20)):
        with pytest.raises(qattn.QattnError) as e:
            ctx.q4_matmul_swiglu(buf.ptr, 4, 64, buf.ptr, w_bytes, n_inter, buf.ptr, ldy=ldy)
        assert e.value.code == qattn.EINVAL, (n_inter, ldy, w_bytes)
    buf.free()


# (m, k, n): each launch takes another kernel or tile of the dispatch, at its edges: ragged last tiles
# in M and N, K blocks that are no multiple of the loops' four and eight, N no multiple of 8.
TILE_CASES = [
    (50, 1024, 4096, False), (50, 992, 1501, False), (33, 1024, 6144, True),  # 32-row blocks
    (300, 2048, 1024, False), (500, 3072, 1023, False), (150, 1056, 384, True),  # one wavefront per block
    (150, 3072, 2048, True), (33, 4160, 96, False),  # five chunks
    (50, 2048, 1000, False), (64, 3072, 1023, False), (40, 4096, 9, False),  # 16 x 16 blocks
    (65, 2048, 1000, False), (33, 4096, 1400, False),  # 16 x 32 blocks
    (65, 96, 6001, False),      # 64 x 128 tiles, one row past a tile, N odd
    (1025, 1024, 4096, False),  # 256 x 128
    (500, 160, 12300, False),   # 256 x 128, K padded to 8 blocks, N = 8 k + 4
    (4100, 64, 4352, False),    # shallow K: 128 x 128 where 256 x 256 leaves its last round empty
    (2100, 1024, 4096, False),  # 256 x 256
    (2570, 32, 4100, False),    # 256 x 256, one K block
    (1900, 1056, 520, False),    # a chunk of 32 K blocks and one of a single block, folded, 64 x 128
    (2100, 2048, 1024, False),  # two chunks, 128 x 128
    (4200, 3072, 1000, False),  # three chunks, folded, 128 x 256
    (200, 1024, 6144, True), (1030, 1024, 6144, True), (1300, 1024, 6144, True),  # n: gate + up rows
    (2100, 96, 6144, True), (23000, 32, 384, True), (5000, 1120, 384, True), (700, 2048, 6144, True),
]


# K above 1024 in every way to run its chunks: a group per chunk, or folded in one.
TALL_CASES = [
    (64, 2048, 10240, True), (65, 3072, 1000, False),
    (1500, 2048, 1000, False), (320, 2048, 6144, True), (600, 2048, 6144, True), (4200, 2048, 1000, False),  # two chunks
    (1500, 3072, 1000, False), (320, 3072, 6144, True), (2200, 3072, 1024, False), (600, 3072, 6144, True),  # three
    (8300, 1088, 1000, False), (1400, 2080, 6144, True), (1200, 3072, 6144, True),  # folded
]


@pytest.mark.parametrize("m,k,n,swiglu", TILE_CASES + TALL_CASES)
def test_q4_tiled_launches_equal_small_launches_bit_for_bit(ctx, m, k, n, swiglu):
    """All rows of a launch against the same rows in launches of at most 32, which take the kernels
    for small launches (themselves checked against the oracle): equal bit for bit.  Where both are the
    same kernel (at most 33 to 64 rows) this holds only that a row does not depend on its place."""
    rng = np.random.default_rng(m + k + n)
    packed = random_compact(rng, n, k)
    x = rng.standard_normal((m, k)).astype(np.float16)
    run = (lambda v: run_q4_swiglu(ctx, v, packed, k, n // 2)) if swiglu else (lambda v: run_q4(ctx, v, packed, k, n))
    cols = n // 2 if swiglu else n
    whole = run(x)[:, :cols].view(np.uint16)
    starts = sorted(set(list(range(0, m, 32 * max(1, m // 512))) + [max(0, m - 32)]))
    for a in starts:
        small = run(x[a:a + 32])[:, :cols].view(np.uint16)
        assert np.array_equal(whole[a:a + 32], small), (a, np.argwhere(whole[a:a + 32] != small)[:4])


@pytest.mark.parametrize("m,k,n", [(15, 1024, 4096), (50, 2048, 1000), (300, 3072, 1024), (1419, 1024, 4096),
                                   (2100, 2048, 1024)])
def test_q4_weights_need_only_4_byte_alignment(ctx, m, k, n):
    rng = np.random.default_rng(m + k)
    packed = random_compact(rng, n, k)
    x = rng.standard_normal((m, k)).astype(np.float16)
    bx, bw = ctx.upload(x.view(np.uint16)), ctx.upload(np.concatenate([np.zeros(4, np.uint8), packed]))
    by = ctx.alloc(m * n * 2)
    ctx.q4_matmul(bx.ptr, m, k, bw.ptr + 4, packed.size, n, by.ptr)
    ctx.synchronize()
    y = by.read(np.uint16, (m, n))
    for b in (bx, bw, by):
        b.free()
    assert np.array_equal(y, run_q4(ctx, x, packed, k, n).view(np.uint16))


@pytest.mark.parametrize("k", [3072, 3104, 4096, 5120, 8192])
@pytest.mark.parametrize("m", [5, 100, 300, 500, 1419, 3000, 4200])
def test_q4_sums_restart_every_1024_columns(ctx, m, k):
    """fp32 sums over K are chains of 1,024 columns, added in order, so a chain's rounding bound does not
    grow with K.  Column 0 contributes 2^30 and column 0 of the last chunk takes it away again; the
    chunks between hold ones.  A chain that carried 2^30 (spacing 128) into a block of ones would lose
    its 32; chains of their own keep every one: the result is the count of ones, exactly."""
    n, kb, last = 1024, k // 32, (k - 1) // 1024 * 32
    rec = np.zeros((n // 32, kb, 32, 20), np.uint8)
    rec[..., 4:20] = 0x88  # q - 8 = 0
    rec[:, [0, last], 0::2, 0:2] = np.array([8192], np.float16).view(np.uint8)
    rec[:, [0, last], 0::2, 4] = 0x8C  # column 0: (12 - 8) * 8192 = 2^15
    rec[:, 32:last, 0::2, 0:2] = np.array([1], np.float16).view(np.uint8)
    rec[:, 32:last, 0::2, 4:20] = 0x99
    x = np.ones((m, k), np.float16)
    x[:, 0], x[:, 32 * last] = 2.0 ** 15, -(2.0 ** 15)
    x[1::2] *= -1
    y = run_q4(ctx, x, rec.reshape(-1), k, n).astype(np.float64)
    expected = np.zeros((m, n))
    expected[:, 0::2] = np.where(np.arange(m) % 2, -1.0, 1.0)[:, None] * (32 * last - 1024)
    assert np.array_equal(y, expected)


# (m, k, n, swiglu): wide outputs, whose launches go by the rows that a tile would pad
WIDE_CASES = [(64, 96, 65600, False), (40, 32, 65664, True), (65, 160, 40000, False), (128, 64, 65664, True),
              (257, 1024, 20000, False), (384, 32, 33000, False), (300, 64, 33024, True),
              (50, 1056, 33100, False), (128, 1120, 33000, False), (100, 2080, 33024, True)]


@pytest.mark.parametrize("m,k,n,swiglu", WIDE_CASES)
def test_q4_wide_launches_equal_their_columns_alone(ctx, m, k, n, swiglu):
    """A projection to many columns against launches over 128 weight rows of it (64 gate and 64 up rows),
    which take the kernels for small outputs: equal bit for bit."""
    rng = np.random.default_rng(m + k + n)
    packed = random_compact(rng, n, k)
    x = rng.standard_normal((m, k)).astype(np.float16)
    tiles = packed.reshape(-(-n // 32), -1)
    cols = n // 2 if swiglu else n
    whole = (run_q4_swiglu(ctx, x, packed, k, cols) if swiglu else run_q4(ctx, x, packed, k, n))[:, :cols]
    for c in (0, cols // 64 // 2 * 64, (cols - 1) // 64 * 64):
        if swiglu:
            part = np.concatenate([tiles[c // 32:c // 32 + 2], tiles[(cols + c) // 32:(cols + c) // 32 + 2]])
            alone, width = run_q4_swiglu(ctx, x, part.reshape(-1), k, 64), 64
        else:
            width = min(128, n - c)
            alone = run_q4(ctx, x, tiles[c // 32:c // 32 + 4].reshape(-1), k, width)
        assert np.array_equal(whole[:, c:c + width].view(np.uint16), alone[:, :width].view(np.uint16)), c


@pytest.mark.parametrize("m,k,n", [(40, 4096, 9), (33, 4096, 1400), (33, 4160, 96), (9, 8192, 200), (40, 8224, 64)])
def test_q4_long_k_matches_oracle(ctx, oracle, m, k, n):
    """The kernels of small launches with more than three chunks of K, which other launches are compared with."""
    rng = np.random.default_rng(m + k + n)
    packed = random_compact(rng, n, k)
    x = rng.standard_normal((m, k)).astype(np.float16)
    check(oracle, run_q4(ctx, x, packed, k, n), x, packed, k, n, f"q4 {m}x{k}x{n}")


@pytest.mark.parametrize("m,k,n_inter", [(40, 2048, 192), (17, 3072, 192), (40, 4096, 192), (5, 4160, 128)])
def test_q4_long_k_swiglu_equals_the_two_launches(ctx, oracle, m, k, n_inter):
    test_q4_matmul_swiglu_equals_the_two_launches(ctx, oracle, m, k, n_inter)


# One case for every kernel and way to run the chunks of K, ragged in M and N.
STRIDED_CASES = [(50, 1024, 1500), (70, 992, 4090), (150, 96, 6001), (1025, 1024, 4091), (500, 160, 12301), (2100, 64, 1021),
                 (2100, 1024, 4090), (50, 2048, 1001), (65, 3072, 1003), (300, 2048, 1021), (1500, 2048, 1001),
                 (2100, 2048, 1021), (4200, 2048, 1000), (1500, 3072, 1019), (2200, 3072, 1020), (1900, 1056, 517),
                 (4200, 3072, 1005), (8300, 1088, 1001), (50, 3072, 1001), (40, 4096, 100), (65, 2048, 1001),
                 (33, 4096, 1401), (150, 3072, 1021)]


@pytest.mark.parametrize("m,k,n", STRIDED_CASES)
def test_q4_strided_rows_equal_compact_ones(ctx, m, k, n):
    """x rows inside a wider matrix (NaN between them, nothing after the last one's K columns but NaN) and y
    rows inside a wider one: the same bits, and no column past N written."""
    rng = np.random.default_rng(m + k + n)
    packed = random_compact(rng, n, k)
    x = rng.standard_normal((m, k)).astype(np.float16)
    compact = run_q4(ctx, x, packed, k, n)
    ldx, ldy = k + 40, -(-n // 8) * 8 + 24
    wide = np.full((m + 1, ldx), np.nan, np.float16)
    wide[:m, :k] = x
    bx, bw, by = ctx.upload(wide.view(np.uint16)), ctx.upload(packed), ctx.alloc((m + 1) * ldy * 2)
    by.fill_u16(0x7E01)
    ctx.q4_matmul(bx.ptr, m, k, bw.ptr, packed.size, n, by.ptr, ldx=ldx, ldy=ldy)
    ctx.synchronize()
    y = by.read(np.uint16, (m + 1, ldy))
    for b in (bx, bw, by):
        b.free()
    assert np.array_equal(y[:m, :n], compact[:, :n].view(np.uint16))
    assert (y[:, n:] == 0x7E01).all() and (y[m] == 0x7E01).all()
