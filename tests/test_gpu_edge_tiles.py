"""GPU parity of the edge kernel (csrc/edge.hip) at the edges of its work split: rows of
fewer than 8 columns, a last tile whose lanes overlap, K of fewer 64-wide blocks than the
workgroup has waves, 16 / 17 / 33 rows, groups of 32, and zeros above 15."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import helpers as H
from oracle import ref_cpu as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 7, 9, 127, 129, 250])
@pytest.mark.parametrize("M,K", [(1, 64), (16, 192), (17, 576), (33, 64)])
def test_w8_tiles(N, M, K):
    """In-place residual: a column is added once though two lanes may compute it."""
    from qwen35_amd.kernels import gemm
    a, as_ = H.engine_act(M, K, seed=3)
    b, bs = H.engine_w8(K, N, seed=4)
    out = (torch.randn(M, N) * 0.1).to(torch.bfloat16).cuda()
    ref = R.gemm_i8_ref(a.numpy(), as_.numpy(), b.numpy(), bs.numpy()) + out.float().cpu().numpy()
    gemm.gemm_i8(a.cuda(), as_.cuda(), b.cuda(), bs.cuda(), out, residual=out)
    H.assert_out_close(out, ref)


@pytest.mark.parametrize("sdt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("group,K", [(32, 64), (64, 576), (192, 576)])
@pytest.mark.parametrize("M,N", [(1, 5), (5, 131), (18, 1003)])
def test_w4_tiles(M, N, group, K, sdt):
    from qwen35_amd.kernels import w4
    a, as_ = H.engine_act(M, K, seed=5)
    gen = torch.Generator().manual_seed(6)
    p = torch.randint(0, 256, (K // 2, N), generator=gen, dtype=torch.uint8)
    s = (torch.rand((K // group, N), generator=gen) * 0.01 + 1e-3).to(sdt)
    z = torch.randint(0, 256, (K // group, N), generator=gen, dtype=torch.uint8)  # any byte is a zero point
    out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    w4.gemm_w4(a.cuda(), as_.cuda(), p.cuda(), s.cuda(), out, b_z=z.cuda())
    ref = R.gemm_w4_ref(a.numpy(), as_.numpy(), p.numpy(), s.float().numpy(), z.numpy())
    H.assert_out_close(out, ref)


def test_proj3_mixed_widths():
    """Projections below and above 8 columns in one call (two launches)."""
    from qwen35_amd.kernels import gemm
    M, K, ns = 20, 256, (130, 3, 65)
    a, as_ = H.engine_act(M, K, seed=7)
    ws = [H.engine_w8(K, n, seed=8 + n) for n in ns]
    out = torch.empty(M, sum(ns), dtype=torch.bfloat16, device="cuda")
    gemm.proj3(a.cuda(), as_.cuda(), *[t.cuda() for w in ws for t in w], out)
    ref = np.concatenate([R.gemm_i8_ref(a.numpy(), as_.numpy(), w.numpy(), s.numpy()) for w, s in ws], 1)
    H.assert_out_close(out, ref)
