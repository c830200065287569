"""k_attn_short -- the fast decode step's attention at short contexts (a head per workgroup, f32 sums) -- against float64 arithmetic on the
same f16 inputs, and the step that uses it against the exact chain."""
import numpy as np
import pytest

from crabml_amd import synth

pytestmark = pytest.mark.gpu
EXACT = 4194304  # CRABML_HIP_LLAMA_EXACT_ATTENTION


def attend(dev, q, k, v, n_heads, n_kv, hd, seq, cap):
    """the kernel on a cache whose rows past `seq` are NaN; float64 on the rows that count"""
    kc, vc = (np.full((n_kv, cap, hd), np.nan, np.float16) for _ in range(2))
    kc[:, :seq], vc[:, :seq] = k, v
    got, _ = dev.debug_short_attention(q, kc.view(np.uint16).reshape(-1), vc.view(np.uint16).reshape(-1), n_heads, n_kv, hd, seq, cap)
    q16 = q.astype(np.float16).astype(np.float64).reshape(n_heads, hd)
    ref = np.zeros((n_heads, hd))
    with np.errstate(invalid="ignore", over="ignore"):
        for h in range(n_heads):
            s = k[h // (n_heads // n_kv)].astype(np.float64) @ q16[h]
            p = np.exp(s - s.max())
            ref[h] = (p / p.sum()) @ v[h // (n_heads // n_kv)].astype(np.float64)
    return got.reshape(n_heads, hd), ref


# a row of 8 / 16 / 32 lanes, full and with dead lanes; positions at the edges of a wave's request, of the speculative 64 and of a round
@pytest.mark.parametrize("n_heads,n_kv,hd", [(6, 6, 8), (4, 2, 40), (6, 6, 48), (8, 1, 64), (6, 2, 96), (32, 8, 128), (4, 4, 136), (4, 1, 256)])
@pytest.mark.parametrize("spread", [1.0, 8.0])
def test_against_float64(ca, n_heads, n_kv, hd, spread):
    dev = ca.HipTensorDevice(0)
    rng = np.random.default_rng(hd)
    for seq in (1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 31, 33, 63, 64, 65, 127, 128, 129, 191, 192, 193, 511, 700):
        for cap in (seq, seq + 200):
            q = (rng.standard_normal(n_heads * hd) * spread / np.sqrt(hd)).astype(np.float32)
            k, v = (rng.standard_normal((n_kv, seq, hd)).astype(np.float16) for _ in range(2))
            got, ref = attend(dev, q, k, v, n_heads, n_kv, hd, seq, cap)
            # exp's argument carries the score's f32 error, hd roundings of |score| <= 32: 2e-5 of the largest output, as for the long kernels
            assert np.max(np.abs(got - ref)) <= 2e-5 * np.max(np.abs(ref)), (seq, cap)


@pytest.mark.parametrize("hd", [48, 128])
def test_infinities_and_nan(ca, hd):
    """a score of -inf has weight zero wherever it lies, +inf and NaN scores make the head NaN, an infinite v stays in its column"""
    dev = ca.HipTensorDevice(0)
    rng = np.random.default_rng(5)
    for seq, at in ((3, 0), (40, 33), (130, 129), (300, 64)):
        q = np.abs(rng.standard_normal(hd)).astype(np.float32)
        k, v = (rng.standard_normal((1, seq, hd)).astype(np.float16) for _ in range(2))
        k[0, at, 3] = -np.inf
        got, ref = attend(dev, q, k, v, 1, 1, hd, seq, seq + 8)
        assert np.max(np.abs(got - ref)) <= 2e-5 * np.max(np.abs(ref)), seq
        v[0, at ^ 1, 5] = np.inf
        got, ref = attend(dev, q, k, v, 1, 1, hd, seq, seq + 8)
        assert np.isposinf(got[0, 5]) and np.isfinite(np.delete(got[0], 5)).all(), seq
        for bad in (np.inf, np.nan):
            k[0, at, 3] = bad
            assert np.isnan(attend(dev, q, k, v, 1, 1, hd, seq, seq + 8)[0]).all(), (seq, bad)


@pytest.mark.parametrize("n_heads,n_kv,hd", [(3, 1, 32), (8, 2, 64), (5, 5, 96), (32, 8, 128), (2, 1, 160), (4, 1, 256)])
@pytest.mark.parametrize("qtype,name", [(synth.Q8_0, "Q8_0"), (synth.Q8_1, "Q8_1")])
def test_its_quantizer_is_the_quantizer(ca, n_heads, n_kv, hd, qtype, name):
    """what the kernel leaves for wo (Q8_0; Q8_1 under Q4_1 layers) is what the stand-alone quantizer makes of its f32 row, bit for bit -- blocks of
    zeros, of one large element, with infinities and NaN among them"""
    dev = ca.HipTensorDevice(0)
    rng = np.random.default_rng(hd + qtype)
    for seq in (1, 77):
        q = rng.standard_normal(n_heads * hd).astype(np.float32)
        k, v = (rng.standard_normal((n_kv, seq, hd)).astype(np.float16) for _ in range(2))
        v[0, :, 0:32] = 0
        if hd >= 64:
            v[-1, :, 32:64], v[-1, :, 40] = 1e-3, 6e4
        if hd >= 96:
            v[0, seq - 1, 70] = np.inf
        if hd >= 128:
            v[-1, 0, 127] = np.nan
        out, blocks = dev.debug_short_attention(q, k.view(np.uint16).reshape(-1), v.view(np.uint16).reshape(-1), n_heads, n_kv, hd, seq, seq, qtype=qtype)
        raw = ca.HipTensor.new(out, [out.size], dev).debug_quantize(getattr(ca.GGMLType, name)).reshape(out.size // 32, -1)
        blocks = blocks.reshape(-1, 34)
        assert np.array_equal(blocks[:, :32], raw[:, -32:].view(np.int8)), seq
        assert np.array_equal(blocks[:, 32], raw[:, :2].copy().view(np.uint16)[:, 0]), seq
        want = raw[:, -32:].view(np.int8).astype(np.int32).sum(axis=1) if name == "Q8_0" else raw[:, 2:4].copy().view(np.uint16)[:, 0]
        assert np.array_equal(blocks[:, 33], want), seq


def test_q4_1_steps_on_the_short_kernel_equal_the_segment_path(ca):
    """Q4_1 layers from 96 cached positions: the five-kernel step, whose attention quantizes its own row to Q8_1, against the segments with the
    quantizer in a launch of its own, bit for bit up to k_attn_flash's first positions"""
    dev = ca.HipTensorDevice(0)
    conf, w = synth.to_hip(synth.build_model(synth.SHAPES["tiny-hd128"], synth.Q4_1, seed=62), dev)
    five = ca.HipLlamaRunner(conf, w, dev, 460, True)
    segs = ca.HipLlamaRunner(conf, w, dev, 460, True, extra_flags=512)  # CRABML_HIP_LLAMA_Q4_1_SEGMENTS
    assert [five.debug_graphs(i)[0] for i in (94, 95, 446, 447)] == [0, 3, 3, 2]
    for i, t in enumerate(int(x) for x in np.random.default_rng(9).integers(0, 1000, size=450)):
        if 90 <= i < 130 or i >= 440:
            a, b = five.forward(t, i), segs.forward(t, i)
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), i
        else:
            five.forward_async(t, i), segs.forward_async(t, i)


@pytest.mark.parametrize("fmt", ["Q8_0", "F16", "Q4_K"])
def test_step_across_the_switches(ca, fmt):
    """positions 0 .. 529: k_attn_short from the start (Q8_0) or from 96 (the others) up to 448, k_attn_flash behind -- graph and eager agree
    bit for bit, and stay as close to the exact chain as k_attn_flash is required to"""
    model = synth.build_model(synth.SHAPES["tiny-hd128"], synth.TYPE_BY_NAME[fmt], seed=78)
    dev = ca.HipTensorDevice(0)
    conf, w = synth.to_hip(model, dev)
    a, e, x = ca.HipLlamaRunner(conf, w, dev, 533, True), ca.HipLlamaRunner(conf, w, dev, 533, True, False), ca.HipLlamaRunner(conf, w, dev, 533, True, extra_flags=EXACT)
    check = {0, 94, 95, 96, 97, 128, 446, 447, 448, 510, 511, 512, 529}
    assert [a.debug_graphs(i)[0] for i in (94, 95, 446, 447)] == [0, 0 if fmt == "Q8_0" else 3, 0 if fmt == "Q8_0" else 3, 2]
    errs = []
    for i in range(530):
        t = (5 * i + 2) % 1000
        if i not in check:
            for r in (a, e, x):
                r.forward_async(t, i)
            continue
        got, eager, exact = a.forward(t, i).copy(), e.forward(t, i).copy(), x.forward(t, i).copy()
        assert np.array_equal(got.view(np.uint32), eager.view(np.uint32)), i
        if fmt != "Q8_0" and i < 95:
            assert np.array_equal(got.view(np.uint32), exact.view(np.uint32)), i
        errs.append(np.max(np.abs(got - exact)) / np.max(np.abs(exact)))
    assert max(errs) <= 7.5e-2, errs  # (the widest of the long kernels' bounds, helpers.FAST_TOL: a flipped level of the quantized row)


@pytest.mark.parametrize("fmt", ["Q4_0", "Q8_0"])
@pytest.mark.parametrize("asked", ["exact norm", "norms apart", "mixed layers"])
def test_steps_that_keep_the_norms_order_keep_the_attentions(ca, fmt, asked):
    """below 96 cached positions a Q4_0 / Q8_0 step leaves the reference's f16 chain only together with its norms' order: with the norm's
    division kept in its launch, with norms as launches of their own, and over files whose layers mix formats, EXACT_ATTENTION changes no bit"""
    model = synth.build_model(synth.SHAPES["tiny-gqa"], synth.TYPE_BY_NAME[fmt], seed=31)
    if asked == "mixed layers":
        t = model.tensors["blk.0.attn_v.weight"]
        t.typ = synth.Q8_0 if fmt == "Q4_0" else synth.Q4_0
        t.data = synth.random_blocks(np.random.default_rng(1), t.shape[0] * t.shape[1], t.typ)
    kw, flags = dict(norm_epilogue=asked != "norms apart"), 8388608 if asked == "exact norm" else 0  # CRABML_HIP_LLAMA_EXACT_NORM
    dev = ca.HipTensorDevice(0)
    conf, w = synth.to_hip(model, dev)
    a = ca.HipLlamaRunner(conf, w, dev, 128, True, extra_flags=flags, **kw)
    b = ca.HipLlamaRunner(conf, w, dev, 128, True, extra_flags=flags + EXACT, **kw)
    for i in range(95):
        la, lb = a.forward((7 * i + 3) % 1000, i), b.forward((7 * i + 3) % 1000, i)
        assert np.array_equal(la.view(np.uint32), lb.view(np.uint32)), i


@pytest.mark.parametrize("fmt", ["Q4_0", "Q4_K", "F16"])
@pytest.mark.parametrize("shape,seq,long_from", [("tiny-hd128", 64, 0), ("tiny-hd128", 300, 0), ("tiny-hd128", 513, 0), ("tiny-hd128", 1000, 0),
                                                 ("tiny-hd128", 1000, 1), ("tiny-hd128", 400, 500), ("15m", 600, 0)])
def test_a_context_captures_the_steps_that_its_positions_run(ca, fmt, shape, seq, long_from):
    """one graph for every attention form between the first and the last cache position, and none that nothing replays"""
    if fmt == "Q4_K" and shape == "15m":
        pytest.skip("width 288 is not whole super-blocks")
    dev = ca.HipTensorDevice(0)
    conf, w = synth.to_hip(synth.build_model(synth.SHAPES[shape], synth.TYPE_BY_NAME[fmt], seed=2), dev)
    r = ca.HipLlamaRunner(conf, w, dev, seq, True, attn_long_from=long_from)
    assert sorted({r.debug_graphs(p)[0] for p in range(seq)}) == r.debug_graphs(0)[1]
