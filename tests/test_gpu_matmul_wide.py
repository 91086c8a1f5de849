"""The many-row products (k_gemm_wide) at the edges of their tiles: every output
equals, bit for bit, the same input row's in calls of at most 16 rows (the
other kernel, held to the oracle in test_gpu_matmul.py), over weight types,
ragged rows and inputs, every tile shape of the launch rule, and each epilogue."""
import numpy as np
import pytest
import torch

import vkv
from gpu_util import dev, stream_ptr
from kq_util import random_matrix

pytestmark = pytest.mark.gpu

# (output rows, inputs, input rows): 32 x 16-row tiles with ragged rows and
# one-block K; 16-input remainders of 32- and 64-input tiles; odd row counts
# (scalar stores); more virtual waves than blocks, and several blocks each
PLAIN = [(6151, 256, 97), (3072, 2304, 503), (3072, 4096, 96), (4100, 1280, 65), (1283, 2048, 131),
         (8192, 512, 129)]
SWIGLU = [(9216, 768, 57), (5121, 1280, 19), (8200, 512, 66), (9217, 256, 48)]
DTYPES = [vkv.Q4_K, vkv.Q6_K, vkv.Q8_0]


def workspace(n_cols, n_in):
    b = vkv.matmul_workspace(n_cols, n_in)
    t = torch.empty(b // 4 + 64, device=dev())
    return t, (t.data_ptr() + 255) & ~255, b


def by_16(call, P):
    for p in range(0, P, 16):
        call(p, min(16, P - p))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n_rows,n_in,P", PLAIN)
@pytest.mark.parametrize("epilogue", ["plain", "residual", "gelu"])
def test_plain(dtype, n_rows, n_in, P, epilogue):
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


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n_rows,n_in,P", SWIGLU)
@pytest.mark.parametrize("biased", [False, True])
def test_swiglu(dtype, n_rows, n_in, P, biased):
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


def test_several_matrices_and_an_unaligned_output():
    """Q/K/V of mixed types in one call, one output row-aligned to 4 bytes only"""
    rng = np.random.default_rng(5)
    mats, n_in, P = [(vkv.Q4_K, 2048), (vkv.Q6_K, 1036), (vkv.Q4_K, 1024)], 768, 101
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


@pytest.mark.parametrize("dtype", [vkv.Q4_K, vkv.Q8_0])
def test_adapter_rows_in_rings(dtype):
    """128 adapter groups in one commit (input rows and outputs in rings, the
    outputs across the wrap) against 16 at a time"""
    enc, dec, down, cap = 1280, 3072, 4, 512
    rng = np.random.default_rng(9)
    w0, w2 = (torch.from_numpy(random_matrix(rng, dtype, dec, k, 0.05)).to(dev()) for k in (enc * down, dec))
    ad = vkv.Adapter(w0.data_ptr(), w2.data_ptr(), dtype, dtype, enc, dec, down)
    frames = torch.randn(cap, enc, device=dev())
    src = vkv.RowRing(frames.data_ptr(), cap, enc)
    outs = []
    for step in (128, 16):
        emb = torch.full((160, dec), float("nan"), device=dev())
        ring = vkv.RowRing(emb.data_ptr(), 160, dec)
        wb = vkv.adapter_workspace(ad, step)
        ws = torch.empty(wb // 4 + 64, device=dev())
        for g in range(100, 228, step):
            vkv.adapter_commit(ad, src, ring, g, step, (ws.data_ptr() + 255) & ~255, wb,
                               hip_stream=stream_ptr())
        torch.cuda.synchronize()
        outs.append(emb.view(torch.int32))
    assert torch.equal(*outs)
