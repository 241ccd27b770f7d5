"""Which bits a packed GEMM gives: those of its number of K ranges, whatever
kernel runs.

With one range the 128 x 512, 144 x 384, 128 x 384 and K-range tile kernels add
every output's products in the same order, so that the entry points, the
epilogues, the batch's concatenated q/k/v GEMM and calls over some of the rows
agree bit for bit although their shapes take different kernels.  The number of
ranges follows the shape (batch, in_dim, out_dim): a call over few of the rows
may add 2, 4 or 8 ranges, the same values up to the order of the fp32 sums.
"""
import pytest

pytestmark = pytest.mark.gpu

K, N = 3072, 9216
ROWS = {"144x384": 4608, "128x384": 4096, "128x512": 3584, "128x512+64": 4240, "k1 32x192": 400, "k1 64x192": 900,
        "k1 128x192": 2431}


def say(msg):
    print(msg, flush=True)


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


@pytest.mark.parametrize("values", ["normal", "wide"])
def test_kernels_agree(torch, b1, gemm_plan, values):
    """The first rows of one input through every kernel: N(0, 1), and
    magnitudes from 2^-14 to 2^13 with rows beyond the fp16 range (row
    scales)."""
    from bonsai_b1 import synth
    say(f"one range, every kernel, {values}")
    a = synth.device_activations(4608, K, 501)
    if values == "wide":
        a *= torch.exp2(torch.randint(-14, 14, a.shape, device="cuda").float())
        a[3] *= 1.0e4
        a[390] *= 1.0e5
    w = synth.device_packed_weights(N, K, 502)
    want = None
    for name, m in ROWS.items():
        assert gemm_plan(m, K, N) == name
        packed, scale = b1.pack_act_f16_scaled(a[:m])
        y = b1.linear_packed_f16_scaled(packed, scale, w, K, N, m)
        torch.cuda.synchronize()
        assert values == "normal" or bool((scale != 1.0).any())
        if want is None:
            want = y
        assert torch.equal(y, want[:m]), name


@pytest.mark.parametrize("split", [0, 448])
def test_packed_swiglu_at_any_split(torch, b1, gemm_plan, split):
    """Packed SwiGLU columns from a split point inside a 384-column tile run
    the 128 x 512 kernel where the plain linear runs 144 x 384 tiles: the same
    bits as that linear and the separate producer."""
    from bonsai_b1 import synth
    m, n = 4608, N
    say(f"packed SwiGLU split {split}")
    assert gemm_plan(m, K, n) == "144x384"
    assert gemm_plan(m, K, n, "packed_swiglu", split) == ("128x512" if split % 384 else "144x384")
    p = b1.pack_act_f16(synth.device_activations(m, K, 503))
    w = synth.device_packed_weights(n, K, 504)
    y = b1.linear_packed_f16(p, w, K, n, m)
    out, packed = b1.linear_packed_f16_to_packed(p, w, K, n, m, split, "swiglu")
    want = b1.swiglu_pack_f16(y[:, split:].contiguous())
    torch.cuda.synchronize()
    assert torch.equal(packed[:want.numel()], want)
    assert split == 0 or torch.equal(out[:, :split], y[:, :split])


@pytest.mark.parametrize("m,k,n", [(1664, 1152, 3072), (4096, 1152, 1024), (4608, 3072, 1152)])
def test_qkv_as_one_gemm(torch, b1, gemm_plan, m, k, n):
    """q, k and v over adjacent rows of one buffer into adjacent columns: one
    GEMM, of another kernel than each alone, with the bits of each alone."""
    from bonsai_b1 import synth
    say(f"q/k/v ({m},{k},{n})")
    assert gemm_plan(m, k, n) != gemm_plan(m, k, 3 * n)
    x = synth.device_activations(m, k, 505)
    parts = [synth.device_packed_weights(n, k, 506 + i) for i in range(3)]
    cat = torch.cat([p.reshape(-1) for p in parts])
    step = n * (k // 32 * 6)
    qkv = torch.empty((m, 3 * n), device="cuda")
    b1.linear_batch([(x, b1.device_weights(cat[i * step:(i + 1) * step], k, n), qkv[:, i * n:(i + 1) * n])
                     for i in range(3)])
    refs = [b1.linear(x, p, n) for p in parts]
    torch.cuda.synchronize()
    for i, r in enumerate(refs):
        assert torch.equal(qkv[:, i * n:(i + 1) * n], r), i


@pytest.mark.parametrize("rows", [416, 384, 17])
def test_rows_of_a_call(torch, b1, gemm_plan, unpack, rows):
    """A call over the first rows of another, through the plain and the
    epilogue entries: bit for bit where both sum one range, else the order of
    the sum apart (each within 2 K 2^-24 sum |a w| of the exact product), and
    the epilogues always over the bits of their own shape's plain call."""
    from bonsai_b1 import synth
    m, ranges = 1024, gemm_plan(rows, K, N)[:2]
    say(f"first {rows} of {m} rows, {ranges}")
    assert gemm_plan(m, K, N).startswith("k1 ") and (ranges == "k1") == (rows == 416)
    p = b1.pack_act_f16(synth.device_activations(m, K, 507))
    w = synth.device_packed_weights(N, K, 508)
    gate, res = synth.device_activations(1, N, 509)[0], synth.device_activations(m, N, 510)
    part = p[:rows * K * 2]
    whole, y = b1.linear_packed_f16(p, w, K, N, m), b1.linear_packed_f16(part, w, K, N, rows)
    g = b1.linear_packed_f16_epi(part, w, K, N, rows, "gate_residual", gate=gate, residual=res[:rows])
    torch.cuda.synchronize()
    assert torch.equal(g, res[:rows] + gate * y)
    if ranges == "k1":
        assert torch.equal(y, whole[:rows])
    else:
        a = synth.device_activations(m, K, 507)[:rows].half().double().abs()
        mag = a @ unpack(w, N, K).abs().t().contiguous()
        assert float(((y.double() - whole[:rows].double()).abs() / (4.0 * K * 2.0 ** -24 * mag)).max()) <= 1.0
