"""The short-prompt kernel of the fp16-activation linears (csrc/prefill_kg.hip) at the edges
of its work split: rows around its tiles, columns past N, fewer K steps than waves, K splits
that do not divide K, groups that straddle two waves' runs; against the oracle, and both tile
heights bit for bit (the K order depends on K and the splits alone)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import helpers as H

pytestmark = pytest.mark.gpu


def _both_tiles(monkeypatch, splits, run):
    out = []
    for bm in (32, 64):
        monkeypatch.setenv("QLIN_PREFILL_KG", f"{bm},{splits}")
        out.append(run())
        assert torch.equal(run(), out[-1])  # the arrival order of the splits must not matter
    assert torch.equal(*out)
    return out[0]


@pytest.mark.parametrize("M,N", [(17, 16), (33, 144), (64, 80), (65, 64)])
@pytest.mark.parametrize("K,splits", [(64, 1), (64, 3), (320, 1), (1088, 3), (1088, 8)])
def test_w8(monkeypatch, M, N, K, splits):
    from qwen35_amd.kernels import linear
    xp = H.act_f16(M, K + 8, seed=K + M)  # a row stride of its own
    w, s = H.w8(K, N, seed=N)
    res = torch.randn((M, N), generator=H.gen(7)).to(torch.float16)
    x = xp.cuda()[:, :K]
    wc, sc = w.cuda(), s.cuda()

    def run():
        o = res.cuda()
        return linear.linear_w8(x, wc, sc, o, residual=o)
    y = _both_tiles(monkeypatch, splits, run)
    H.assert_out_close(y, H.linear_w8_ref_cols(xp[:, :K].contiguous(), w, s, np.arange(N), residual=res))


@pytest.mark.parametrize("M,N", [(17, 16), (50, 208)])
@pytest.mark.parametrize("group,sdt,zeros", [(32, torch.float16, "random"), (64, torch.bfloat16, "none"),
                                             (128, torch.float32, "random"), (192, torch.float16, "none")])
@pytest.mark.parametrize("splits", [1, 3])
def test_w4(monkeypatch, M, N, group, sdt, zeros, splits):
    from qwen35_amd.kernels import linear
    K = 576 if group in (64, 192) else 640
    x = H.act_f16(M, K, seed=M)
    p, s, z = H.w4(K, N, seed=N, group=group, zeros=zeros)
    s = s.to(sdt)
    xc, pc, sc, zc = x.cuda(), p.cuda(), s.cuda(), None if z is None else z.cuda()

    def run():
        return linear.linear_w4(xc, pc, sc, torch.empty(M, N, dtype=torch.bfloat16, device="cuda"), w_zero=zc)
    y = _both_tiles(monkeypatch, splits, run)
    H.assert_out_close(y, H.linear_w4_ref_cols(x, p, s.float() if sdt == torch.bfloat16 else s, z, np.arange(N)))


def test_graph_replays():
    """The library's own choice with K splits under capture, replayed between eager calls."""
    from qwen35_amd.kernels import linear, qlin
    M, K, N = 48, 4096, 512
    x, (w, s) = H.act_f16(M, K, seed=1).cuda(), (t.cuda() for t in H.w8(K, N, seed=2))
    o = torch.empty(M, N, dtype=torch.float16, device="cuda")
    eager = linear.linear_w8(x, w, s, o).clone()
    g = torch.cuda.CUDAGraph()
    with qlin.capture(g):
        linear.linear_w8(x, w, s, o)
    for _ in range(3):
        o.zero_()
        g.replay()
        assert torch.equal(o, eager)
        assert torch.equal(linear.linear_w8(x, w, s, torch.empty_like(o)), eager)


@pytest.mark.parametrize("M,K,N", [(17, 512, 64), (129, 64, 400), (300, 1024, 1280)])
def test_wide_tile(monkeypatch, M, K, N):
    """The 128 x 384 tile of the large-tile kernel (QLIN_PREFILL_SHAPE=3): the bits of the
    256 x 256 tile (one K order), W8 with a residual and W4 with zeros in each scale dtype."""
    from qwen35_amd.kernels import linear
    x = H.act_f16(M, K, seed=M).cuda()
    w, s = (t.cuda() for t in H.w8(K, N, seed=N))
    p, s4, z = (t.cuda() for t in H.w4(K, N, seed=N, group=32, zeros="random"))
    res = torch.randn((M, N), generator=H.gen(9)).to(torch.float16).cuda()
    monkeypatch.setenv("QLIN_PREFILL", "tiled")
    outs = []
    for shape in (1, 3):
        monkeypatch.setenv("QLIN_PREFILL_SHAPE", str(shape))
        o = [linear.linear_w8(x, w, s, torch.empty_like(res), residual=res)]
        for dt in (torch.float16, torch.bfloat16, torch.float32):
            o.append(linear.linear_w4(x, p, s4.to(dt), torch.empty_like(res), w_zero=z))
        outs.append(o)
    assert all(torch.equal(a, b) for a, b in zip(*outs))
    H.assert_out_close(outs[1][0], H.linear_w8_ref_cols(x.cpu(), w.cpu(), s.cpu(), np.arange(N), residual=res.cpu()))
