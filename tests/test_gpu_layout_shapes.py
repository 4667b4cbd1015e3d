"""The load-time layout kernels (csrc/layout.hip) at the edges of their forms, bit for bit
against the oracle: strips past N and rows past the registers (requant), values at rounding
ties, odd word counts and off-grid sources (repacks)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import ref_cpu as R

pytestmark = pytest.mark.gpu


def _weights(K, N, seed):
    """Normal weights with exact ties of the W8 grid, an all-zero column and a huge one."""
    w = torch.randn(K, N, generator=torch.Generator().manual_seed(seed)) * 0.02
    w[0, 0] = 127.0  # scale exactly 1: the column's other values are on and beside ties
    w[1:, 0] = (torch.arange(K - 1) % 254 - 127).float() + 0.5
    w[2::3, 0] = torch.nextafter(w[2::3, 0], torch.tensor(0.0))
    w[:, 1] = 0.0
    w[:, 2] *= 1e36
    return w


@pytest.mark.parametrize("K,N", [(64, 4), (200, 20), (1030, 36), (2100, 516), (4130, 64), (300, 4100), (600, 8260),
                                 (65, 7), (8200, 20), (12300, 516)])
def test_requant_w8(K, N):
    from qwen35_amd.kernels import layout
    w = _weights(K, N, K + N)
    q, s = layout.requant_w8_row(w.cuda())
    rq, rs = R.requant_w8_row(w.numpy())
    assert np.array_equal(s.cpu().numpy(), rs)
    assert np.array_equal(q.cpu().numpy(), rq)


@pytest.mark.parametrize("group", [32, 64])
@pytest.mark.parametrize("K,N", [(64, 4), (128, 1030), (192, 2052), (64, 7)])
def test_requant_w4(K, N, group):
    from qwen35_amd.kernels import layout
    w = _weights(K, N, K + N + group)
    w[1:, 0] = (torch.arange(K - 1) % 14 - 7).float() + 0.5  # ties of the 4-bit grid
    w[0::group, 0] = 7.0
    p, s = layout.requant_w4_sym(w.cuda(), group)
    rp, rs = R.requant_w4_sym(w.numpy(), group)
    assert np.array_equal(s.cpu().view(torch.int16).numpy().view(np.uint16), rs)
    assert np.array_equal(p.cpu().numpy(), rp)


def _words(*shape, seed, off=0):
    """int32 words on the GPU, `off` words past an allocation's start."""
    t = torch.randint(-2 ** 31, 2 ** 31 - 1, shape, generator=torch.Generator().manual_seed(seed), dtype=torch.int32)
    flat = torch.empty(t.numel() + off, dtype=torch.int32, device="cuda")
    flat[off:].copy_(t.reshape(-1))
    return t.numpy().view(np.uint32), flat[off:].view(shape)


@pytest.mark.parametrize("K,N,off", [(2, 8, 0), (64, 24, 0), (66, 48, 0), (66, 48, 1), (300, 272, 0)])
def test_awq(K, N, off):
    from qwen35_amd.kernels import layout
    w, t = _words(K, N // 8, seed=K, off=off)
    pos = [0, 4, 1, 5, 2, 6, 3, 7]  # nibble of column 8c + j in word c
    nib = np.stack([(w >> (4 * p)) & 15 for p in pos], -1).reshape(K, N).astype(np.uint8)
    assert np.array_equal(layout.awq_w4_to_engine(t).cpu().numpy(), nib[0::2] | (nib[1::2] << 4))


@pytest.mark.parametrize("N,W,K,off", [(16, 1, 8, 0), (144, 3, 24, 0), (144, 5, 34, 0), (128, 36, 288, 0), (272, 36, 282, 0),
                                       (272, 36, 282, 1)])
def test_ct(N, W, K, off):
    from qwen35_amd.kernels import layout
    w, t = _words(N, W, seed=N + W, off=off)
    rows = np.ascontiguousarray(w).view(np.uint8).reshape(N, 4 * W)
    assert np.array_equal(layout.ct_w4_to_engine(t, K).cpu().numpy(), rows.T[: K // 2])
