"""The small-batch kernel at 9 to 16 tokens (b1_gemv3_kernel<16, false>): fp32
rows read 64 bytes a quad of lanes and put into fragments through LDS.

Shapes: every token count's edges, K of one block group, one pass and several,
a width of one row and with a remainder.  Bar for tokens within the fp16
range: against the float64 product of the fp16-rounded activations, per
element |y - ref| <= 2 K 2^-24 sum_k |a_k w_k|, the bound of an fp32 sum of K
products in any order (twice, for products added pairwise inside an MFMA
step).  Tokens holding an |a| >= 65520: EXACT mode's bits; others unchanged.
"""
import pytest

pytestmark = pytest.mark.gpu


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


@pytest.mark.parametrize("m,k,n", [(9, 256, 1), (10, 1024, 300), (12, 3072, 9216), (13, 3328, 97), (15, 9216, 600),
                                   (16, 3072, 4100), (16, 512, 17)])
def test_rows(torch, b1, unpack, m, k, n):
    from bonsai_b1 import synth
    print(f"small batch ({m},{k},{n})", flush=True)
    a = torch.zeros((m, k + 4), device="cuda")[:, :k]      # rows apart
    a.copy_(synth.device_activations(m, k, 71))
    w = synth.device_packed_weights(n, k, 72)
    y = b1.linear(a, w, n, mode="gemv")
    h, wd = a.half().double(), unpack(w, n, k)
    ref, mag = h @ wd.t(), h.abs() @ wd.abs().t()
    torch.cuda.synchronize()
    assert float(((y.double() - ref).abs() / (2.0 * k * 2.0 ** -24 * mag)).max()) <= 1.0
    big = [0, m // 2, m - 1]
    a[0, k - 1] = -65520.0
    a[m // 2] *= 1.0e6
    a[m - 1, 17] = 3.0e38
    nf = torch.zeros(1, dtype=torch.int32, device="cuda")
    z = b1.linear(a, w, n, mode="gemv", nonfinite=nf)
    e = b1.linear(a, w, n, mode="exact")
    torch.cuda.synchronize()
    keep = [t for t in range(m) if t not in big]
    assert torch.equal(z[keep], y[keep])
    assert torch.equal(z[big], e[big])
    assert int(nf.item()) == int((~torch.isfinite(z)).sum())
