"""The K-range tile GEMM (b1_tile_gemm_kernel): the packed GEMM of shapes
with few output tiles, whose work-groups split K into 1, 2, 4 or 8 contiguous
ranges and add the partial tiles in LDS.

Shapes: every number of ranges and tile height on 256 CUs, row counts at and
around the 32- and 64-row tile edges, widths one column past or short of a
tile, K whose ranges are of unequal length or whose ends cut off weight groups
of 2 and 4 pairs, and one weight row.

Bars:
  plain     : against the float64 product of the fp16-rounded activations,
              per element |y - ref| <= 2 K 2^-24 sum_k |a_k w_k|, the bound
              of an fp32 sum of K products in any order (twice, for products
              added pairwise inside an MFMA step).
  epilogues : gate-residual bit for bit residual + gate * y in fp32 on the
              plain call's y; SwiGLU and GELU packed outputs bit for bit the
              separate producers' packing of that y.
"""
import sys

import pytest

pytestmark = pytest.mark.gpu

# (m, k, n), by K ranges on 256 CUs
RANGES = {
    8: [(17, 3072, 48), (32, 3072, 3071), (33, 3072, 97), (64, 3456, 1000), (65, 15360, 193), (256, 3072, 3072),
        (33, 3456, 300)],
    4: [(31, 1920, 18433), (129, 2688, 9000), (512, 1536, 3072), (500, 2688, 3071)],
    2: [(63, 768, 577), (200, 1152, 640), (1024, 1536, 3072), (300, 3072, 9216), (777, 1920, 3000),
        (1024, 8064, 3072)],
    1: [(19, 384, 1), (63, 384, 1500), (130, 768, 30000), (1000, 1152, 9217), (400, 384, 9217), (1100, 1152, 9000)],
}
SHAPES = [s for r in RANGES.values() for s in r]
# (m, k, n, epilogue, split, kernel on 256 CUs): every tile, plain and packed
PLANS = [(17, 3072, 48, "plain", 0, "k8 32x48"), (256, 3072, 3072, "plain", 0, "k8 64x48"),
         (129, 2688, 9000, "plain", 0, "k4 32x96"), (512, 1536, 3072, "plain", 0, "k4 64x96"),
         (200, 1152, 640, "plain", 0, "k2 64x96"), (63, 384, 1500, "plain", 0, "k1 32x192"),
         (130, 768, 30000, "plain", 0, "k1 64x192"), (1000, 1152, 9217, "plain", 0, "k1 128x192"),
         (64, 3456, 960, "packed_swiglu", 0, "k8 32x64"), (256, 3072, 3072, "packed_swiglu", 0, "k8 64x64"),
         (512, 1536, 3072, "packed_swiglu", 0, "k4 64x128"), (200, 1152, 640, "packed_swiglu", 0, "k2 64x128"),
         (1024, 1536, 3072, "packed_swiglu", 0, "k2 64x192"), (63, 384, 1472, "packed_swiglu", 0, "k1 32x192")]


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


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


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_plain(torch, b1, unpack, m, k, n):
    from bonsai_b1 import synth
    say(f"k-range gemm ({m},{k},{n})")
    a = synth.device_activations(m, k, 401)
    w = synth.device_packed_weights(n, k, 402)
    out = torch.full((m, n + 5), 7.0, device="cuda")
    b1.linear(a, w, n, out=out[:, :n], mode="gemm")            # odd row stride: scalar stores
    nf = torch.zeros(1, dtype=torch.int32, device="cuda")
    y = b1.linear(a, w, n, mode="gemm", nonfinite=nf)
    torch.cuda.synchronize()
    assert torch.equal(out[:, :n], y) and bool((out[:, n:] == 7.0).all())
    assert int(nf.item()) == 0
    h = a.half().double()
    wd = unpack(w, n, k)
    ref, mag = h @ wd.t(), h.abs() @ wd.abs().t()
    over = ((y.double() - ref).abs() / (2.0 * k * 2.0 ** -24 * mag)).max()
    say(f"  largest error / bound {float(over):.3e}")
    assert float(over) <= 1.0
    # rows beyond the fp16 range and non-finite rows, in the sum's own place
    if m > 17:
        a[m - 1] *= 1.0e6
        a[3, k - 1] = float("inf")
        z = b1.linear(a, w, n, mode="gemm", nonfinite=nf)
        torch.cuda.synchronize()
        assert int(nf.item()) == n and not bool(torch.isfinite(z[3]).any())
        keep = [i for i in range(m - 1) if i != 3]
        assert torch.equal(z[keep], y[keep])
        last = (a[m - 1].double() @ wd.t())
        assert float((z[m - 1].double() - last).norm() / last.norm()) < 1e-3   # fp16 rounding: 2^-11 a term


@pytest.mark.parametrize("m,k,n", [s for s in SHAPES if s[2] > 64])
def test_epilogues(torch, b1, m, k, n):
    from bonsai_b1 import synth
    n = n // 64 * 64
    say(f"k-range epilogues ({m},{k},{n})")
    a = synth.device_activations(m, k, 403)
    w = synth.device_packed_weights(n, k, 404)
    p = b1.pack_act_f16(a)
    y = b1.linear_packed_f16_epi(p, w, k, n, m, "none")
    gate = synth.device_activations(1, n, 405)[0]
    for pad in (0, 3):
        res = synth.device_activations(m, n + pad, 406)[:, :n]
        got = b1.linear_packed_f16_epi(p, w, k, n, m, "gate_residual", gate=gate, residual=res)
        torch.cuda.synchronize()
        assert torch.equal(got, res + gate * y)
    glu = b1.swiglu_pack_f16(y)
    f32 = b1.linear_packed_f16_epi(p, w, k, n, m, "swiglu")
    assert torch.equal(b1.pack_act_f16(f32), glu)
    split = n // 128 * 64
    for act, producer in (("none", b1.pack_act_f16), ("gelu_tanh", b1.gelu_tanh_pack_f16),
                          ("swiglu", b1.swiglu_pack_f16)):
        for sp in {0, split}:
            out, packed = b1.linear_packed_f16_to_packed(p, w, k, n, m, sp, act)
            want = producer(y[:, sp:].contiguous())
            torch.cuda.synchronize()
            assert torch.equal(packed[:want.numel()], want), (act, sp)
            if sp:
                assert torch.equal(out[:, :sp], y[:, :sp]), (act, sp)
