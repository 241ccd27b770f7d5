"""The GEMM that converts fp32 activations tile by tile (b1_gemm_fused_kernel,
in_dim % 384 != 0 or no workspace) at every tile its launcher picks on 256 CUs,
with row and column remainders.

Bar for rows within the fp16 range: against the float64 product of the
fp16-rounded activations, per element |y - ref| <= 2 K 2^-24 sum_k |a_k w_k|,
the bound of an fp32 sum of K products in any order (twice, for products added
pairwise inside an MFMA step).  Rows holding an |a| >= 65520 or an infinity:
EXACT mode's bits; NaN rows: NaN; the non-finite counter counts what is stored.
"""
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [  # (m, k, n, tile on 256 CUs)
    (17, 64, 1, "32x64"), (33, 448, 65, "32x64"), (77, 2048, 5504, "32x64"), (300, 320, 1027, "32x64"),
    (1000, 256, 5500, "64x128"), (640, 128, 4097, "64x128"), (1024, 64, 8193, "64x128"),
    (1000, 192, 8100, "64x256"), (2049, 64, 8192, "64x256"),
    (2000, 448, 8100, "128x512"), (2305, 896, 12300, "128x512"),
]


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


@pytest.mark.parametrize("m,k,n,tile", SHAPES)
def test_tiles(torch, b1, unpack, fused_plan, m, k, n, tile):
    from bonsai_b1 import synth
    assert fused_plan(m, k, n) == tile
    print(f"fused gemm ({m},{k},{n})", flush=True)
    a = synth.device_activations(m, k, 51)
    w = synth.device_packed_weights(n, k, 52)
    buf = torch.full((m, n + 3), 7.0, device="cuda")
    b1.linear(a, w, n, out=buf[:, :n], mode="gemm")
    torch.cuda.synchronize()
    y = buf[:, :n].clone()
    assert bool((buf[:, n:] == 7.0).all())
    h, wd = a.half().double(), unpack(w, n, k)
    ref, mag = h @ wd.t(), h.abs() @ wd.abs().t()
    assert float(((y.double() - ref).abs() / (2.0 * k * 2.0 ** -24 * mag)).max()) <= 1.0
    # rows beyond the fp16 range, first, last and at a tile's edge
    big = sorted({0, min(30, m - 1), m // 2, m - 1})
    a[big[0], k - 1] = 65520.0
    for r in big[1:]:
        a[r] *= 1.0e6
    a[m - 1, 1] = float("inf")
    a[m - 2, 2] = float("nan")
    nf = torch.zeros(1, dtype=torch.int32, device="cuda")
    z = b1.linear(a, w, n, mode="gemm", nonfinite=nf)
    e = b1.linear(a, w, n, mode="exact")
    torch.cuda.synchronize()
    keep = torch.ones(m, dtype=torch.bool, device="cuda")
    keep[big + [m - 2]] = False
    assert torch.equal(z[keep], y[keep])
    assert torch.equal(z[big], e[big])
    assert bool(torch.isnan(z[m - 2]).all())
    assert int(nf.item()) == int((~torch.isfinite(z)).sum())


@pytest.mark.parametrize("m,k,n", [(17, 64, 1), (77, 2048, 130), (33, 448, 65), (640, 128, 4097), (1000, 192, 8100),
                                   (2000, 448, 8100)])
@pytest.mark.parametrize("step", [1, 3])
def test_many_rows_beyond_fp16(torch, b1, m, k, n, step):
    """Every row, or every third one, beyond the fp16 range: whole groups of 4
    flagged rows a wave, the remainders of a tile's flagged rows and of its
    columns, at every tile; EXACT mode's bits in those rows, the others
    unchanged."""
    from bonsai_b1 import synth
    print(f"fused gemm, rows beyond fp16 ({m},{k},{n}) step {step}", flush=True)
    a = synth.device_activations(m, k, 53)
    w = synth.device_packed_weights(n, k, 54)
    y = b1.linear(a, w, n, mode="gemm")
    big = torch.arange(0, m, step, device="cuda")
    a[big] *= 1.0e6
    nf = torch.zeros(1, dtype=torch.int32, device="cuda")
    buf = torch.full((m, n + 3), 7.0, device="cuda")
    b1.linear(a, w, n, out=buf[:, :n], mode="gemm", nonfinite=nf)
    e = b1.linear(a, w, n, mode="exact")
    torch.cuda.synchronize()
    keep = torch.ones(m, dtype=torch.bool, device="cuda")
    keep[big] = False
    assert torch.equal(buf[big, :n], e[big])
    assert torch.equal(buf[keep, :n], y[keep])
    assert bool((buf[:, n:] == 7.0).all()) and int(nf.item()) == 0
