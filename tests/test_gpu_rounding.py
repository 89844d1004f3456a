"""The roundings of the residual add + RMSNorm (qattn_rmsnorm) and of the QK norm + RoPE
(qattn_qk_norm_rope*), bit for bit against a host restatement of their arithmetic: embeddings stored
before there were fused projections stay equal, and a row does not depend on the kernel that computed it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F32 = np.float32


def fma(a, b, c):
    """a b + c of f32 values in 64 bits: the product is exact there, and the sum is rounded far below the
    f32 or fp16 rounding that the caller applies."""
    return a.astype(np.float64) * b.astype(np.float64) + c.astype(np.float64)


def test_rmsnorm_with_residual_bits(ctx):
    rows, width, eps = 8000, 1024, 1e-6
    rng = np.random.default_rng(3)
    x, r = (rng.standard_normal((rows, width)).astype(np.float16) for _ in range(2))
    w = (1 + 0.1 * rng.standard_normal(width)).astype(F32)
    bx, br, bw = ctx.upload(x.view(np.uint16)), ctx.upload(r.view(np.uint16)), ctx.upload(w)
    bo = ctx.alloc(rows * width * 2)
    ctx.rmsnorm(bx.ptr, bw.ptr, bo.ptr, rows, width, residual_ptr=br.ptr, eps=eps)
    ctx.synchronize()
    got_x, got = bx.read(np.uint16, (rows, width)), bo.read(np.uint16, (rows, width))
    for b in (bx, br, bw, bo):
        b.free()
    s = x.astype(F32) + r.astype(F32)
    # lane l sums columns 8 l .. + 7 and 512 + 8 l .. + 7, the first pair's squares as fma(s0, s0, s1 s1)
    lanes = np.concatenate([s[:, :512].reshape(rows, 64, 8), s[:, 512:].reshape(rows, 64, 8)], axis=-1)
    ss = fma(lanes[..., 0], lanes[..., 0], lanes[..., 1] * lanes[..., 1]).astype(F32)
    for e in range(2, 16):
        ss = fma(lanes[..., e], lanes[..., e], ss).astype(F32)
    for d in (32, 16, 8, 4, 2, 1):
        ss = ss + ss[:, np.arange(64) ^ d]
    inv = F32(1) / np.sqrt(ss[:, :1] / F32(width) + F32(eps))
    x16 = s.astype(np.float16)
    assert np.array_equal(got_x, x16.view(np.uint16))
    assert np.array_equal(got, (x16.astype(F32) * inv * w).astype(np.float16).view(np.uint16))


@pytest.mark.parametrize("heads", [4, 8, 12, 24, 32])
def test_rope_bits(ctx, heads):
    """Rows of +-1 with eps = 0 have unit RMS, so the normalised element is the gain, exactly."""
    tokens, theta = 1500, 1e6
    rng = np.random.default_rng(heads)
    sign = rng.choice(np.array([-1, 1], np.float16), (tokens, heads * 128))
    gain = (1 + 0.1 * rng.standard_normal(128)).astype(F32)
    bx, bw = ctx.upload(sign.view(np.uint16)), ctx.upload(gain)
    ctx.qk_norm_rope(bx.ptr, heads * 128, 0, heads, np.array([0, tokens], np.int32), weight_ptr=bw.ptr, eps=0.0,
                     theta=theta)
    ctx.synchronize()
    got = bx.read(np.uint16, (tokens, heads, 2, 8, 8))  # half, lane, element
    bx.free()
    bw.free()
    angle = np.arange(tokens, dtype=np.float64)[:, None] * theta ** (-np.arange(64, dtype=np.float64) / 64)
    cos, sin = (f(angle).astype(F32).reshape(tokens, 1, 1, 8, 8) for f in (np.cos, np.sin))
    n = sign.astype(F32).reshape(tokens, heads, 2, 8, 8) * gain.reshape(1, 1, 2, 8, 8)
    partner = np.stack([-n[:, :, 1], n[:, :, 0]], axis=2)
    cos_last = fma(n, np.broadcast_to(cos, n.shape), partner * sin)  # one rounding, then two, then the other order
    sin_last = fma(partner, np.broadcast_to(sin, n.shape), n * cos)
    once, twice = cos_last.astype(np.float16), cos_last.astype(F32).astype(np.float16)
    other = sin_last.astype(F32).astype(np.float16)
    expected = once.copy()
    expected[:, 0:4, ..., 1:7] = twice[:, 0:4, ..., 1:7]
    expected[:, 0:4, ..., 1:7:2] = other[:, 0:4, ..., 1:7:2]
    expected[:, 4:8, ..., 2:8] = twice[:, 4:8, ..., 2:8]
    expected[:, 4:8, ..., 2:8:2] = other[:, 4:8, ..., 2:8:2]
    differ = np.argwhere(got != expected.view(np.uint16))
    assert len(differ) == 0, (len(differ), differ[:4])
