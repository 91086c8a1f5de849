"""The many-row products (k_gemm_wide) at the edges of their tiles: every output
equals, bit for bit, the same input row's in calls of at most 16 rows (the
other kernel, held to the oracle in test_gpu_matmul.py), over weight types,
ragged rows and inputs, every tile shape of the launch rule (restated in form(),
so that a call meant for the wide kernel cannot fall back unseen), and each
epilogue but RoPE (test_gpu_decoder_prompt.py, test_gpu_encoder_chunk.py)."""
import numpy as np
import pytest
import torch

import vkv
from gpu_util import dev, stream_ptr
from kq_util import random_matrix


def form(dtypes, rows, n_in, P, swiglu=False):
    """launch_gemm_kq's choice for a call (wide_form): None or (column tiles, row tiles)"""
    up = lambda a, b: -(-a // b)
    q80, q4 = dtypes[0] == vkv.Q8_0, dtypes[0] == vkv.Q4_K
    t = sum(up(n, 16) for n in (rows[:1] if swiglu else rows))
    g2x2, g2x4 = up(t, 2) * up(P, 32), up(t, 4) * up(P, 32)
    g4x2, g4x4 = up(t, 2) * up(P, 64), up(t, 4) * up(P, 64)
    if P <= 16:
        return None
    if swiglu:
        four = g2x2 > (640 if q4 else 512) or (not q4 and g2x2 > 256 and g4x2 <= 256)
        need = 6144 if not q80 else 27648 if four and g4x2 > 256 else 24576
        return None if t * P < need else (4, 2) if four else (2, 2)
    if t < 128:
        wide = t * up(P, 16) >= (800 if n_in > 4096 else 560)
    else:
        wide = t * P >= (30720 if q80 else 10240 if P >= 96 else 16384)
    if not wide:
        return None
    if g2x2 > 1024 or (not q4 and g2x2 > 768 and g4x4 <= 256):
        return 4, 4
    return (2, 4) if not q80 and g2x2 > 256 and g2x4 <= 256 else (2, 2)


DTYPES = [vkv.Q4_K, vkv.Q6_K, vkv.Q8_0]
# (output rows, inputs, input rows) and each type's form: ragged rows and
# one-block K; 16-input remainders of 32- and 64-input tiles; odd row counts
# (scalar stores); more virtual waves than blocks, and several blocks each;
# both sides of 128 row tiles, the larger ones at K above 4096
Q4, Q6, Q8 = DTYPES
PLAIN = [((6151, 256, 97), {Q4: (2, 2), Q6: (4, 4), Q8: (4, 4)}),
         ((3072, 2304, 503), dict.fromkeys(DTYPES, (4, 4))),
         ((3072, 4096, 96), {Q4: (2, 4), Q6: (2, 4)}),
         ((4100, 1280, 65), {Q4: (2, 4), Q6: (2, 4)}),
         ((3073, 1280, 307), {Q4: (2, 2), Q6: (4, 4), Q8: (4, 4)}),
         ((3072, 5120, 163), dict.fromkeys(DTYPES, (2, 2))),
         ((1283, 2048, 131), dict.fromkeys(DTYPES, (2, 2))),
         ((1281, 4608, 145), dict.fromkeys(DTYPES, (2, 2))),
         ((1277, 512, 250), {Q4: (2, 4), Q6: (2, 4), Q8: (2, 2)}),
         ((8192, 512, 129), dict.fromkeys(DTYPES, (4, 4)))]
SWIGLU = [((9216, 768, 57), {Q4: (2, 2), Q6: (4, 2), Q8: (4, 2)}),
          ((5121, 1280, 21), {Q4: (2, 2), Q6: (2, 2)}),
          ((5120, 1280, 83), dict.fromkeys(DTYPES, (2, 2))),
          ((5121, 1536, 131), dict.fromkeys(DTYPES, (4, 2))),
          ((8200, 512, 131), dict.fromkeys(DTYPES, (4, 2))),
          ((9217, 256, 24), {Q4: (2, 2), Q6: (2, 2)})]


def cases(table):
    return [pytest.param(dt, *shape, f, id=f"{dt}-" + "-".join(map(str, shape)))
            for shape, forms in table for dt, f in forms.items()]


def test_the_shapes_reach_every_tile_form():
    seen = set()
    for table, swiglu in ((PLAIN, False), (SWIGLU, True)):
        for (n_rows, n_in, P), forms in table:
            for dt, f in forms.items():
                assert form([dt] * (1 + swiglu), [n_rows] * (1 + swiglu), n_in, P, swiglu) == f, (n_rows, n_in, P, dt)
                if n_in // 256 > (4 if swiglu else 8):   # several blocks in a virtual wave
                    seen.add((dt, f, swiglu))
    k = [(dt, f, False) for dt in DTYPES[:2] for f in ((2, 2), (2, 4), (4, 4))]
    q = [(vkv.Q8_0, f, False) for f in ((2, 2), (4, 4))]
    assert seen >= set(k + q + [(dt, f, True) for dt in DTYPES for f in ((2, 2), (4, 2))])


def workspace(n_cols, n_in):
    b = vkv.matmul_workspace(n_cols, n_in)
    t = torch.empty(b // 4 + 64, device=dev())
    return t, (t.data_ptr() + 255) & ~255, b


def by_16(call, P):
    for p in range(0, P, 16):
        call(p, min(16, P - p))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,n_rows,n_in,P,tile", cases(PLAIN))
@pytest.mark.parametrize("epilogue", ["plain", "residual", "gelu"])
def test_plain(dtype, n_rows, n_in, P, tile, epilogue):
    rng = np.random.default_rng(n_rows + n_in + P)
    w = torch.from_numpy(random_matrix(rng, dtype, n_rows, n_in, 0.05)).to(dev())
    g = torch.Generator(device=dev()).manual_seed(P)
    x = torch.randn(P, n_in, device=dev(), generator=g)
    add = torch.randn(P, n_rows, device=dev(), generator=g)
    bias = torch.randn(n_rows, device=dev(), generator=g)
    nw = torch.rand(n_in, device=dev(), generator=g) + 0.5
    ys = [torch.full((P, n_rows), float("nan"), device=dev()) for _ in range(2)]
    t, wp, wb = workspace(P, n_in)

    def call(y):
        def run(p, n):
            o = [w.data_ptr(), dtype, n_rows, y[p].data_ptr()]
            if epilogue != "plain":
                o += [add[p].data_ptr() if epilogue == "residual" else None, bias.data_ptr()]
            vkv.matmul(x[p].data_ptr(), n, n_in, [tuple(o)], wp, wb, norm_w_ptr=nw.data_ptr(),
                       epilogue=vkv.MV_GELU if epilogue == "gelu" else vkv.MV_STORE,
                       hip_stream=stream_ptr())
        return run

    call(ys[0])(0, P)
    by_16(call(ys[1]), P)
    torch.cuda.synchronize()
    assert torch.equal(ys[0], ys[1])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,n_rows,n_in,P,tile", cases(SWIGLU))
@pytest.mark.parametrize("biased", [False, True])
def test_swiglu(dtype, n_rows, n_in, P, tile, biased):
    rng = np.random.default_rng(n_rows + n_in + P)
    w = [torch.from_numpy(random_matrix(rng, dtype, n_rows, n_in, 0.05)).to(dev()) for _ in range(2)]
    g = torch.Generator(device=dev()).manual_seed(P)
    x = torch.randn(P, n_in, device=dev(), generator=g)
    bias = [torch.randn(n_rows, device=dev(), generator=g) for _ in range(2)]
    ys = [torch.full((P, n_rows), float("nan"), device=dev()) for _ in range(2)]
    t, wp, wb = workspace(P, n_in)

    def call(y):
        def run(p, n):
            b = [b.data_ptr() if biased else None for b in bias]
            vkv.matmul(x[p].data_ptr(), n, n_in,
                       [(w[0].data_ptr(), dtype, n_rows, y[p].data_ptr(), None, b[0]),
                        (w[1].data_ptr(), dtype, n_rows, None, None, b[1])], wp, wb,
                       epilogue=vkv.MV_SWIGLU, hip_stream=stream_ptr())
        return run

    call(ys[0])(0, P)
    by_16(call(ys[1]), P)
    torch.cuda.synchronize()
    assert torch.equal(ys[0], ys[1])


@pytest.mark.gpu
def test_several_matrices_and_an_unaligned_output():
    """Q/K/V of mixed types in one call, one output row-aligned to 4 bytes only"""
    rng = np.random.default_rng(5)
    mats, n_in, P = [(vkv.Q4_K, 2048), (vkv.Q6_K, 1036), (vkv.Q4_K, 1024)], 768, 101
    assert form([d for d, _ in mats], [n for _, n in mats], n_in, P)
    w = [torch.from_numpy(random_matrix(rng, dt, n, n_in, 0.05)).to(dev()) for dt, n in mats]
    x = torch.randn(P, n_in, device=dev())
    t, wp, wb = workspace(P, n_in)
    ys = [[torch.full((P * n + 1,), float("nan"), device=dev())[1:].view(P, n) for _, n in mats]
          for _ in range(2)]

    def call(y):
        def run(p, n):
            vkv.matmul(x[p].data_ptr(), n, n_in,
                       [(w[i].data_ptr(), dt, r, y[i][p].data_ptr()) for i, (dt, r) in enumerate(mats)],
                       wp, wb, hip_stream=stream_ptr())
        return run

    call(ys[0])(0, P)
    by_16(call(ys[1]), P)
    torch.cuda.synchronize()
    for a, b in zip(*ys):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [vkv.Q4_K, vkv.Q8_0])
def test_adapter_rows_in_rings(dtype):
    """176 adapter groups in one commit (input rows and outputs in rings, both
    across the wrap) against 16 at a time"""
    enc, dec, down, cap = 1280, 3072, 4, 1024
    assert form([dtype], [dec], enc * down, 176) and form([dtype], [dec], dec, 176)
    rng = np.random.default_rng(9)
    w0, w2 = (torch.from_numpy(random_matrix(rng, dtype, dec, k, 0.05)).to(dev()) for k in (enc * down, dec))
    ad = vkv.Adapter(w0.data_ptr(), w2.data_ptr(), dtype, dtype, enc, dec, down)
    frames = torch.randn(cap, enc, device=dev())
    src = vkv.RowRing(frames.data_ptr(), cap, enc)
    outs = []
    for step in (176, 16):
        emb = torch.full((224, dec), float("nan"), device=dev())
        ring = vkv.RowRing(emb.data_ptr(), 224, dec)
        wb = vkv.adapter_workspace(ad, step)
        ws = torch.empty(wb // 4 + 64, device=dev())
        for g in range(100, 276, step):
            vkv.adapter_commit(ad, src, ring, g, step, (ws.data_ptr() + 255) & ~255, wb,
                               hip_stream=stream_ptr())
        torch.cuda.synchronize()
        outs.append(emb.view(torch.int32))
    assert torch.equal(*outs)
