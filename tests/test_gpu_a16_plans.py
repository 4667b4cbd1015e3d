"""The tile that the fp16-activation linears' plan picks by itself, at ragged sizes: 128x128
two to a CU (a grid of one to two rounds) and split in K, 128x384 and 256x256;
the plan printed must be the one a row names, and the results those of the oracle on
sampled columns."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wt,M,K,N,shape", [
    ("w8", 1001, 1024, 5008, "shape=0 splits=1 sk=0"), ("w4", 1001, 2048, 5008, "shape=0 splits=1 sk=0"),
    ("w8", 1300, 1024, 6128, "shape=3 splits=1 sk=0"), ("w4", 1300, 1024, 6128, "shape=3 splits=1 sk=0"),
    ("w8", 2040, 2048, 6128, "shape=1 splits=1 sk=0"), ("w8", 1300, 2048, 6128, "shape=3 splits=1 sk=0"),
    ("w8", 1010, 2048, 2032, "shape=2 splits=2 sk=0"), ("w4", 1010, 2048, 2032, "shape=2 splits=2 sk=0"),
])
def test_planned_tiles(monkeypatch, capfd, wt, M, K, N, shape):
    from qwen35_amd.kernels import linear
    x = H.act_f16(M, K, seed=M)
    cols = np.unique(np.concatenate([np.arange(8), np.arange(N - 8, N), np.arange(100, N, 509)]))
    out = torch.empty((M, N), dtype=torch.float16, device="cuda")
    monkeypatch.setenv("QLIN_PREFILL_VERBOSE", "1")
    if wt == "w8":
        w, s = H.w8(K, N, seed=N)
        linear.linear_w8(x.cuda(), w.cuda(), s.cuda(), out)
        ref = H.linear_w8_ref_cols(x, w, s, cols)
    else:
        p, s, z = H.w4(K, N, seed=N, group=128, zeros="random")
        linear.linear_w4(x.cuda(), p.cuda(), s.cuda(), out, w_zero=z.cuda())
        ref = H.linear_w4_ref_cols(x, p, s, z, cols)
    H.assert_out_close(out[:, cols], ref)
    assert f"tiled {shape}\n" in capfd.readouterr().err
