"""The tiled int8 kernel's tile shapes (csrc/prefill_i8_kernel.h): every tile gives the bits
of the 16-row tiles (one K order) at rows around each tile's height, an odd number of 64-wide
blocks, N a multiple of 64 only, and K splits; the 16-row tiles are held to the oracle."""
from __future__ import annotations

import pytest
import torch

import helpers as H
from oracle import ref_cpu as R

pytestmark = pytest.mark.gpu

TILES = {0: 128, 1: 64, 2: 96, 3: 128, 4: 160}  # QLIN_I8_TILE -> rows (tile 0: 128 columns, the others 64)


def _weights(wt, K, N, seed):
    if wt == "w8":
        b, s = H.engine_w8(K, N, seed)
        return b.cuda(), s.cuda(), None
    p, s, z = H.w4(K, N, seed, group=64, zeros="random" if wt == "w4z" else "none")
    return p.cuda(), s.to(torch.bfloat16).cuda(), z.cuda() if z is not None else None


def _families(monkeypatch, tile, splits, run):
    """run() on the 16-row tiles and on one tile of the tiled kernel."""
    monkeypatch.setenv("QLIN_ENGINE_SPLITS", str(splits))
    monkeypatch.setenv("QLIN_ENGINE_PREFILL", "skinny")
    rows = run()
    monkeypatch.setenv("QLIN_ENGINE_PREFILL", "tiled")
    monkeypatch.setenv("QLIN_I8_TILE", str(tile))
    return rows, run()


@pytest.mark.parametrize("splits,K", [(1, 320), (2, 768)])
@pytest.mark.parametrize("wt", ["w8", "w4", "w4z"])
@pytest.mark.parametrize("tile", TILES)
def test_gemm_tiles(monkeypatch, tile, wt, splits, K):
    from qwen35_amd.kernels import gemm
    N = 256 if tile == 0 else 192
    w, s, z = _weights(wt, K, N, 31)
    for M in (17, TILES[tile] - 1, TILES[tile] + 1, 2 * TILES[tile] + 33):
        a, as_ = H.engine_act(M, K, seed=32)
        res = torch.randn((M, N), generator=H.gen(33)).to(torch.bfloat16)

        def run():
            o = res.cuda()
            return gemm.gemm_i8(a.cuda(), as_.cuda(), w, s, o, residual=o, b_z=z)
        rows, tiled = _families(monkeypatch, tile, splits, run)
        assert torch.equal(rows, tiled)
    ref = R.gemm_i8_ref(a.numpy(), as_.numpy(), w.cpu().numpy(), s.float().cpu().numpy(),
                        b_z=None if z is None else z.cpu().numpy(), residual=res.float().numpy())
    H.assert_out_close(tiled, ref)


@pytest.mark.parametrize("splits,K", [(1, 320), (2, 768)])
@pytest.mark.parametrize("wt", ["w8", "w4", "w4z"])
@pytest.mark.parametrize("tile", [0, 1, 2])
def test_gate_up_tiles(monkeypatch, tile, wt, splits, K):
    """mlp_gate_up and mlp_gate_up_quant (the tiles that hold two weight sets)."""
    from qwen35_amd.kernels import gemm, w4
    N = 256 if tile == 0 else 192
    (wg, sg, zg), (wu, su, zu) = _weights(wt, K, N, 41), _weights(wt, K, N, 42)
    for M in (17, TILES[tile] + 1):
        a, as_ = (t.cuda() for t in H.engine_act(M, K, seed=43))

        def run():
            q = torch.empty(M, N, dtype=torch.int8, device="cuda")
            sc = torch.empty(M, N // 64, dtype=torch.float32, device="cuda")
            o = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
            gemm.mlp_gate_up_quant(a, as_, wg, sg, wu, su, q, sc, zg=zg, zu=zu)
            if wt == "w8":
                gemm.mlp_gate_up(a, as_, wg, sg, wu, su, o)
            else:
                w4.mlp_gate_up_w4(a, as_, wg, sg, wu, su, o, zg=zg, zu=zu)
            return q, sc, o
        rows, tiled = _families(monkeypatch, tile, splits, run)
        assert all(torch.equal(x, y) for x, y in zip(rows, tiled))


@pytest.mark.parametrize("wt", ["w8", "w4"])
def test_every_row_count_agrees_n64(wt):
    """N a multiple of 64 only, the library's own choice of tile: rows do not depend on M."""
    from qwen35_amd.kernels import gemm
    K, N = 1024, 8256
    w, s, z = _weights(wt, K, N, 51)
    a, as_ = (t.cuda() for t in H.engine_act(400, K, seed=52))
    outs = [gemm.gemm_i8(a[:M].contiguous(), as_[:M].contiguous(), w, s,
                         torch.empty(M, N, dtype=torch.bfloat16, device="cuda"), b_z=z) for M in (9, 17, 40, 130, 400)]
    for o in outs:
        assert torch.equal(o, outs[-1][: o.shape[0]])
