"""The q8_0 window tile on the f32 matrix cores (k_window_mfma_q8_*) against the
scalar-ALU kernel over the same ring: both dequantize exactly and work in f32
throughout, so outputs agree to the f32 order of their sums (a score of 128
terms and 8 to 900 weights: 5e-6 of the output's spread) and the ring's bytes
are the same.  Edges: one query, ragged tiles, the fused write's 16-tile limit,
GQA 1 / 2 / 4, per-layer (split) and several-layer calls, wrapped segments."""
import numpy as np
import pytest
import torch

import vkv
from gpu_util import dev, layer_image, stream_ptr

pytestmark = pytest.mark.gpu


def both(head_dim, kv_heads, q_heads, layers, cap, call):
    outs, imgs = [], []
    for flags in (0, vkv.KERNEL_WINDOW_VALU):
        with vkv.Cache(n_streams=1, n_layers=layers, capacity=cap, n_kv_heads=kv_heads, head_dim=head_dim,
                       n_q_heads=q_heads, dtype=vkv.Q8_0, kernel_flags=flags) as c:
            out = call(c)
            torch.cuda.synchronize()
            outs.append(out.cpu().numpy())
            imgs.append([layer_image(c, w, 0, l).copy() for l in range(layers) for w in (0, 1)])
    for a, b in zip(*imgs):
        assert np.array_equal(a, b)
    return outs


def rows(seed, *shape):
    g = torch.Generator(device=dev()).manual_seed(seed)
    return torch.randn(*shape, device=dev(), generator=g)


@pytest.mark.parametrize("n", [1, 3, 17, 38, 64, 65, 199])
@pytest.mark.parametrize("pos0,layers", [(0, 1), (37, 2)])
def test_prefill(n, pos0, layers):
    kv, qd = 1024, 4096
    old = [rows(i, layers, max(pos0, 1), kv) for i in (1, 2)]
    q, k, v = (rows(i, layers, n, w) for i, w in ((3, qd), (4, kv), (5, kv)))

    def call(c):
        if pos0:
            c.append(0, 0, layers, [(0, pos0)], old[0].data_ptr(), old[1].data_ptr(), hip_stream=stream_ptr())
        ring = vkv.new_ring(512)
        ring.used = ring.next_absolute_position = pos0
        out = torch.full((layers, n, qd), float("nan"), device=dev())
        c.decoder_prefill(0, ring, 0, layers, n, q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                          128 ** -0.5, hip_stream=stream_ptr())
        return out

    a, b = both(128, 8, 32, layers, 512, call)
    assert np.isfinite(a).all() and np.abs(a - b).max() <= 5e-6 * max(1.0, np.abs(b).max())


@pytest.mark.parametrize("head_dim,kv_heads,q_heads,layers", [(64, 32, 32, 1), (64, 32, 32, 3), (64, 4, 8, 1),
                                                              (128, 2, 2, 1), (128, 3, 12, 2)])
@pytest.mark.parametrize("n,q0", [(1, 0), (4, 1297), (16, 2000), (37, 741), (128, 3000)])
def test_encoder_window(head_dim, kv_heads, q_heads, layers, n, q0):
    cap, win, kv = 878, 750, head_dim * kv_heads
    keep = min(q0, win)
    old = [rows(i, layers, max(keep, 1), kv) for i in (1, 2)]
    q, k, v = (rows(i, layers, n, w) for i, w in ((3, head_dim * q_heads), (4, kv), (5, kv)))

    def call(c):
        if keep:
            s, head = (q0 - keep) % cap, min(keep, cap - (q0 - keep) % cap)
            segs = [(s, head)] + ([(0, keep - head)] if keep > head else [])
            c.append(0, 0, layers, segs, old[0].data_ptr(), old[1].data_ptr(), hip_stream=stream_ptr())
        out = torch.full((layers, n, head_dim * q_heads), float("nan"), device=dev())
        c.enc_step(0, vkv.enc_plan(q0, n, cap, win), win, 0, layers, q.data_ptr(), k.data_ptr(), v.data_ptr(),
                   out.data_ptr(), head_dim ** -0.5, hip_stream=stream_ptr())
        return out

    a, b = both(head_dim, kv_heads, q_heads, layers, cap, call)
    assert np.isfinite(a).all() and np.abs(a - b).max() <= 5e-6 * max(1.0, np.abs(b).max())


@pytest.mark.parametrize("bad", [float("inf"), float("nan"), 3e38])
def test_rows_beyond_the_format_stay_with_the_queries_that_see_them(bad):
    """a V row whose scale overflows f16 reaches its own and later tokens only"""
    n, at = 40, 22
    q, k, v = (rows(i, 1, n, w) for i, w in ((3, 4096), (4, 1024), (5, 1024)))
    v[0, at] = bad

    def call(c):
        ring = vkv.new_ring(64)
        out = torch.zeros(1, n, 4096, device=dev())
        c.decoder_prefill(0, ring, 0, 1, n, q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                          128 ** -0.5, hip_stream=stream_ptr())
        return out

    a, b = both(128, 8, 32, 1, 64, call)
    assert np.isfinite(b[0, :at]).all() and np.array_equal(np.isfinite(a), np.isfinite(b))
    assert np.abs(a[0, :at] - b[0, :at]).max() <= 5e-6 * np.abs(b[0, :at]).max()


@pytest.mark.parametrize("bad", [float("inf"), float("nan"), 3e38])
@pytest.mark.parametrize("win,at", [(12, 17), (1, 16), (40, 0)])
def test_a_key_beyond_the_format_stays_with_the_queries_that_see_it(bad, win, at):
    """a K row whose scale overflows f16: the queries that mask it are as
    without it, those that see it (alone in its 16-key block or in the whole
    window too) are NaN, not zeros; in the unsplit and the split tile"""
    n = 40
    q, k, v = (rows(i, 1, n, w) for i, w in ((3, 4096), (4, 1024), (5, 1024)))
    k[0, at] = bad

    def prefill(c):
        out = torch.zeros(1, n, 4096, device=dev())
        c.decoder_prefill(0, vkv.new_ring(96), 0, 1, n, q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                          128 ** -0.5, hip_stream=stream_ptr())
        return out

    def window(width):
        def call(c):
            out = torch.zeros(1, n, width, device=dev())
            c.enc_step(0, vkv.enc_plan(0, n, 96, win), win, 0, 1, q.data_ptr(), k.data_ptr(), v.data_ptr(),
                       out.data_ptr(), 128 ** -0.5, hip_stream=stream_ptr())
            return out
        return call

    for shape, call, sees in (((128, 8, 32), prefill, range(at, n)),
                              ((128, 8, 32), window(4096), range(at, min(n, at + win))),
                              ((64, 16, 16), window(1024), range(at, min(n, at + win)))):
        a, b = both(*shape, 1, 96, call)
        clean = [i for i in range(n) if i not in sees]
        assert np.isfinite(b[0, clean]).all() and np.array_equal(np.isfinite(a), np.isfinite(b))
        if bad == bad:   # (a NaN row is stored as zeros: its largest magnitude is 0)
            assert np.isnan(a[0, list(sees)]).all()
        if clean:
            assert np.abs(a[0, clean] - b[0, clean]).max() <= 5e-6 * np.abs(b[0, clean]).max()
