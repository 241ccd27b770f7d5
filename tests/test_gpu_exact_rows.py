"""EXACT mode's kernel (b1_exact_kernel: 1, 2 or 4 rows a work-group, scalar
activation loads, weights 4 blocks at a time; b1_exact_lds_kernel: 8 or 16)
against the oracle's scalar order, bit for bit.

Shapes: the five row counts on 256 CUs, row remainders, widths around the
256-column work-group, block counts around the groups of 4 (odd ones put the
packed rows on 2-byte boundaries), and rows at strides and offsets that leave
4-byte alignment only.  Values: N(0, 1), subnormals, signed zeros, and rows
whose sums reach infinity or NaN.
"""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [  # (m, k, n, rows a work-group on 256 CUs)
    (1, 32, 1, 1), (1, 3072, 257, 1), (3, 96, 255, 1), (5, 128, 513, 1), (7, 160, 300, 1),
    (65, 224, 1000, 2), (301, 64, 600, 2), (130, 256, 769, 2), (103, 416, 1024, 2), (201, 288, 3000, 2),
    (258, 1056, 1003, 2),
    # 4 rows: one quad of blocks and less, and K past 512, where lines are
    # touched ahead inside the loop, with 1 and 3 blocks after the last quad
    (1023, 192, 1500, 4), (130, 128, 5000, 4), (509, 672, 1500, 4), (1021, 608, 770, 4),
    (601, 96, 3600, 8), (1030, 288, 4090, 16),          # through LDS
]
NONFINITE = [(2, 96, 300, 1), (65, 224, 1000, 2), (258, 160, 3001, 2), (1021, 160, 770, 4), (601, 96, 3600, 8),
             (1030, 96, 4090, 16)]


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need the MI355X"
    return t


@pytest.fixture(scope="module")
def b1(torch):
    import bonsai_b1
    bonsai_b1.load()
    return bonsai_b1


@pytest.mark.parametrize("m,k,n,rows", SHAPES)
def test_bits(torch, b1, oracle, exact_plan, m, k, n, rows):
    from bonsai_b1 import synth
    assert exact_plan(m, n) == rows
    print(f"exact ({m},{k},{n})", flush=True)
    sys.stdout.flush()
    act = synth.activations(m, k, 31 * m + k)
    act[:, ::7] *= np.float32(1e-42)      # subnormal, and zero below the smallest
    act[:, 3::11] = np.float32(-0.0)
    raw = synth.packed_weights(n, k, n + 1)
    ref, _ = oracle.linear(act, raw, n, variant="scalar", nth=4)
    # rows one float past a 16-byte boundary, outputs in a wider matrix, the
    # packed weights on a 2-byte boundary
    lda = k + 1
    abuf = torch.zeros(m * lda + 1, device="cuda")
    a = abuf[1:].view(m, lda)[:, :k]
    a.copy_(torch.from_numpy(act))
    wbuf = torch.zeros(raw.size + 2, dtype=torch.uint8, device="cuda")
    wbuf[2:] = torch.from_numpy(raw.ravel()).cuda()
    out = torch.full((m, n + 3), 7.0, device="cuda")
    b1.linear(a, wbuf[2:], n, out=out[:, :n], mode="exact")
    nf = torch.zeros(1, dtype=torch.int32, device="cuda")
    y = b1.linear(torch.from_numpy(act).cuda(), torch.from_numpy(raw.ravel()).cuda(), n, mode="exact", nonfinite=nf)
    torch.cuda.synchronize()
    y = y.cpu().numpy()
    assert np.array_equal(y.view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(out[:, :n].cpu().numpy().view(np.uint32), ref.view(np.uint32))
    assert bool((out[:, n:] == 7.0).all()) and int(nf.item()) == 0


@pytest.mark.parametrize("m,k,n,rows", NONFINITE)
def test_nonfinite(torch, b1, oracle, exact_plan, m, k, n, rows):
    from bonsai_b1 import synth
    assert exact_plan(m, n) == rows
    print(f"exact non-finite ({m},{k},{n})", flush=True)
    act = synth.activations(m, k, 5)
    act[0, 9] = np.inf
    act[m - 1, k - 1] = np.nan
    act[m // 2, :] *= np.float32(3e38) / np.abs(act[m // 2]).max()
    raw = synth.packed_weights(n, k, 6)
    ref, _ = oracle.linear(act, raw, n, variant="scalar", nth=4)
    nf = torch.zeros(1, dtype=torch.int32, device="cuda")
    y = b1.linear(torch.from_numpy(act).cuda(), torch.from_numpy(raw.ravel()).cuda(), n, mode="exact", nonfinite=nf)
    torch.cuda.synchronize()
    y = y.cpu().numpy()
    bad = ~np.isfinite(ref)
    assert np.array_equal(np.isnan(y), np.isnan(ref)) and int(nf.item()) == int(bad.sum())
    assert np.array_equal(y[~np.isnan(ref)], ref[~np.isnan(ref)])
