"""Codes at and beside rounding ties, groups that hold an infinity, and the producers'
sums over every team size.  The kernels multiply by 1 / scale and divide only near a
tie; the codes must stay those of a division (kernels/norm.py:15-25)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import ref_cpu as R

pytestmark = pytest.mark.gpu

PASS_GATE = 100.0  # sigmoid(100) is 1 in fp32, so gate_mul quantizes its first operand


def _run(a):
    from qwen35_amd.kernels import norm
    M, N = a.shape
    g = torch.full((M, 2 * N), PASS_GATE, dtype=a.dtype)
    q = torch.empty((M, N), dtype=torch.int8, device="cuda")
    s = torch.empty((M, N // 64), dtype=torch.float32, device="cuda")
    norm.gate_mul_quant(a.cuda(), g.cuda(), q, s, hd=64)
    return q.cpu().numpy(), s.cpu().numpy()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("amax", [127.0, 127.0 / 64, 126.0, 93.5, 3.0])
def test_codes_at_and_beside_ties(dtype, amax):
    """For amax = 127 * 2^e the scale is 2^e and (n + 1/2) * scale is a tie exactly; the
    others put the values' nearest neighbours just above and below one."""
    n = np.arange(-127, 127, dtype=np.float32)
    tie = (n + 0.5) * np.float32(np.float32(amax) / np.float32(127.0))
    t = torch.from_numpy(tie).to(dtype)
    step = torch.from_numpy((np.abs(tie) * 2.0 ** -8 + 1e-7).astype(np.float32))
    vals = torch.cat([t, (t.float() + step).to(dtype), (t.float() - step).to(dtype)])
    vals = vals[vals.float().abs() <= amax]
    rows = -(-len(vals) // 63)
    a = torch.zeros((rows, 64), dtype=dtype)
    flat = torch.zeros(rows * 63, dtype=dtype)
    flat[: len(vals)] = vals
    a[:, 1:] = flat.view(rows, 63)
    a[:, 0] = amax  # every group's scale is amax / 127
    rq, rs = R.quant_groups(a.float().numpy())
    gq, gs = _run(a)
    assert (gs.view(np.uint32) == rs.view(np.uint32)).all()
    assert (gq == rq).all(), np.argwhere(gq != rq)[0]


def test_groups_with_an_infinity_and_tiny_groups():
    a = torch.zeros((2, 192), dtype=torch.bfloat16)
    a[0, :64] = torch.linspace(-5, 5, 64).to(torch.bfloat16)
    a[0, 7] = float("inf")   # scale inf: every finite value's code is 0
    a[0, 64:128] = 1e-38     # scale 1e-8 (the floor): codes 0
    a[0, 128:] = 3.0e38      # the largest scale
    a[1] = torch.linspace(-1, 1, 192).to(torch.bfloat16)
    gq, gs = _run(a)
    assert np.isinf(gs[0, 0])
    assert (np.delete(gq[0, :64], 7) == 0).all()
    fin = a.clone()
    fin[0, :64] = 0
    rq, rs = R.quant_groups(fin.float().numpy())
    assert (gq[0, 64:] == rq[0, 64:]).all() and (gq[1] == rq[1]).all()
    assert (gs[0, 1:].view(np.uint32) == rs[0, 1:].view(np.uint32)).all()


@pytest.mark.parametrize("hd", [128, 256, 512])
def test_head_sums_of_every_team_size(hd):
    """Teams of 16, 32 and 64 lanes: the butterfly's order of adds decides the sums' bits."""
    from qwen35_amd.kernels import norm
    T, N = 5, 1024
    gen = torch.Generator().manual_seed(hd)
    v = torch.randn((T, N), generator=gen).to(torch.bfloat16)
    z = torch.randn((T, N), generator=gen).to(torch.bfloat16)
    w = torch.randn((hd,), generator=gen).to(torch.bfloat16)
    q = torch.empty((T, N), dtype=torch.int8, device="cuda")
    s = torch.empty((T, N // 64), dtype=torch.float32, device="cuda")
    norm.norm_gated_quant(v.cuda(), z.cuda(), w.cuda(), q, s)
    rq, rs = R.norm_gated_quant_ref(v.float().numpy(), z.float().numpy(), w.float().numpy())
    assert (q.cpu().numpy() == rq).all()
    assert (s.cpu().numpy().view(np.uint32) == rs.astype(np.float32).view(np.uint32)).all()


@pytest.mark.parametrize("M", [1, 3])
@pytest.mark.parametrize("K", [64, 576, 1984, 2048, 2112, 4096, 4160, 6144])
@pytest.mark.parametrize("dtype,wdt", [(torch.bfloat16, torch.float32), (torch.float16, torch.float16)])
def test_rmsnorm_row_lengths(M, K, dtype, wdt):
    """Rows of every form: parts of a wave, whole waves, one past them, the long rows."""
    from qwen35_amd.kernels import norm
    gen = torch.Generator().manual_seed(K + M)
    x = torch.randn((M, K + 8), generator=gen).to(dtype)[:, :K]
    w = torch.randn((K,), generator=gen).to(wdt)
    q = torch.empty((M, K), dtype=torch.int8, device="cuda")
    s = torch.empty((M, K // 64), dtype=torch.float32, device="cuda")
    xg = torch.empty((M, K + 8), dtype=dtype, device="cuda")[:, :K]
    xg.copy_(x)
    for one_plus in (True, False):
        norm.rmsnorm_quant(xg, w.cuda(), q, s, one_plus=one_plus)
        rq, rs = R.rmsnorm_quant_ref(x.float().numpy(), w.float().numpy(), one_plus=one_plus)
        assert (q.cpu().numpy() == rq).all()
        assert (s.cpu().numpy().view(np.uint32) == rs.astype(np.float32).view(np.uint32)).all()


@pytest.mark.parametrize("N,hd", [(64, 8), (192, 24), (192, 64), (2112, 2112), (4096, 256), (2560, 320)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gate_mul_head_sizes(N, hd, dtype):
    from qwen35_amd.kernels import norm
    gen = torch.Generator().manual_seed(N + hd)
    a = torch.randn((3, N), generator=gen).to(dtype)
    g = torch.randn((3, 2 * N + 8), generator=gen).to(dtype)
    q = torch.empty((3, N), dtype=torch.int8, device="cuda")
    s = torch.empty((3, N // 64), dtype=torch.float32, device="cuda")
    norm.gate_mul_quant(a.cuda(), g.cuda(), q, s, hd=hd)
    rq, rs = R.gate_mul_quant_ref(a.float().numpy(), g.float().numpy(), hd)
    assert (q.cpu().numpy() == rq).all()
    assert (s.cpu().numpy().view(np.uint32) == rs.astype(np.float32).view(np.uint32)).all()
