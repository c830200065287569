"""The two ends of a decode step: sampler, advance, embedding, first norm and its quantizer in one launch behind the classifier, and several steps in
one graph -- against steps that are given their tokens one at a time, eager ones among them, bit for bit."""
import numpy as np
import pytest

from crabml_amd import synth
from crabml_amd import synth_bifazen as sb
from crabml_amd import synth_hybrid as sh

pytestmark = pytest.mark.gpu


def greedy_by_hand(ca, r, token, pos, n):
    ids = []
    for i in range(n):
        token = ca.sample_argmax(r.forward(token, pos + i))
        ids.append(token)
    return ids


# (4352: more than four elements a thread; 288: rows that end inside a wave; Q5_K, F32: launches per operation)
WIDE = synth.ModelShape("wide", 4352, 512, 1, 34, 2, 600, 64, 1e-5, None)


@pytest.mark.parametrize("fmt,shape", [("Q4_0", "tiny-hd128"), ("Q8_0", "15m"), ("Q4_1", "tiny-hd128"), ("Q4_K", "tiny-hd128"), ("Q4_K", "tiny-gqa"), ("F16", "15m"),
                                       ("Q5_K", "tiny-gqa"), ("F32", "tiny-gqa"), ("Q6_K", "tiny-gqa"), ("Q4_0", WIDE), ("Q4_K", WIDE), ("F16", WIDE)])
@pytest.mark.parametrize("strict", [False, True])
@pytest.mark.parametrize("now", [False, True])
def test_greedy_runs_equal_single_steps(ca, monkeypatch, fmt, shape, strict, now):
    if now:  # several steps a graph from the first run on
        monkeypatch.setenv("CRABML_HIP_TEST_HOOKS", "1")
        monkeypatch.setenv("CRABML_HIP_GRAPH_STEPS", "1")
    dev = ca.HipTensorDevice(0, strict_order=strict)
    model = synth.build_model(shape if isinstance(shape, synth.ModelShape) else synth.SHAPES[shape], synth.TYPE_BY_NAME[fmt], seed=21)
    conf, w = synth.to_hip(model, dev)
    long = fmt in ("Q4_0", "Q8_0") and not isinstance(shape, synth.ModelShape) and not strict
    seq = 600 if long else 60
    a, b, e = ca.HipLlamaRunner(conf, w, dev, seq, True), ca.HipLlamaRunner(conf, w, dev, seq, True), ca.HipLlamaRunner(conf, w, dev, seq, True, False)
    pos, token = 0, 3
    for n in (1, 7, 8, 9, 17) + ((400, 100) if long else ()):  # (400, 100: runs over the switches of the attention)
        ids = a.decode_greedy(token, n)
        assert ids == greedy_by_hand(ca, b, token, pos, n), n
        assert ids == e.decode_greedy(token, n), n
        pos, token = pos + n, ids[-1]
    la, lb, le = a.forward(token, pos), b.forward(token, pos), e.forward(token, pos)
    assert np.array_equal(la.view(np.uint32), lb.view(np.uint32)) and np.array_equal(la.view(np.uint32), le.view(np.uint32))


NILIVIK = sh.config(84, 131, [sh.layer(3, 1, 36, 44, 50, 2, 28, 36, 40)], loop={"start": 0, "stop": 1, "times": 2})
NILIVIK_WIDE = sh.config(4104, 67, [sh.layer(1, 1, 8, 8, 16, 1, 8, 8, 16)])  # (more than four columns a thread, the last ones in part)
BIFAZEN = sb.config(200, 131, [sb.latent(2, 12, 4, 12, 20, 30, 40), sb.attention(2, 1, 8, 8, 9, 40)], streams=3)


@pytest.mark.parametrize("config,tensors", [(NILIVIK, sh.random_tensors), (BIFAZEN, sb.random_tensors)])
@pytest.mark.parametrize("rows", [1, 3])
def test_runs_capture_several_steps_a_graph_as_they_go(ca, hdev, tmp_path, config, tensors, rows):
    """runs of all lengths capture graphs of eight, four and two steps behind their first ones: the same tokens before, during and behind that"""
    folder = sh.write_model(config, tensors(config, 7), str(tmp_path / "m"))
    g, e = ca.load_model(folder, hdev, seq_len=300), ca.load_model(folder, hdev, seq_len=300, use_graph=False)
    seqs = [[r.open() for _ in range(rows)] for r in (g, e)]
    ids = list(range(1, rows + 1))
    for n in (1, 3, 9, 30, 9, 60, 17, 7, 100, 12):
        a, b = g.decode_batch(seqs[0], ids, n), e.decode_batch(seqs[1], ids, n)
        assert list(a) == list(b), n
        ids = list(a[-rows:])
    last = [r.step([(s, [t], [0]) for s, t in zip(q, ids)]) for r, q in zip((g, e), seqs)]
    assert np.array_equal(last[0].view(np.uint32), last[1].view(np.uint32))


@pytest.mark.parametrize("now", [False, True])
@pytest.mark.parametrize("config,tensors", [(NILIVIK, sh.random_tensors), (NILIVIK_WIDE, sh.random_tensors), (BIFAZEN, sb.random_tensors)])
@pytest.mark.parametrize("f32", [False, True])
def test_greedy_batches_equal_single_steps(ca, hdev, tmp_path, monkeypatch, config, tensors, f32, now):
    if now:  # several steps a graph from the first run on
        monkeypatch.setenv("CRABML_HIP_TEST_HOOKS", "1")
        monkeypatch.setenv("CRABML_HIP_GRAPH_STEPS", "1")
    folder = sh.write_model(config, tensors(config, 5), str(tmp_path / "m"))
    g, e, h = (ca.load_model(folder, hdev, seq_len=64, f32=f32, **kw) for kw in ({}, {"use_graph": False}, {}))
    for rows in (1, 2, 3, 16):
        seqs = [[r.open() for _ in range(rows)] for r in (g, e, h)]
        ids = [(7 * i + rows) % 60 for i in range(rows)]
        for n in (1, 8, 17, 9, 25):
            a, b = g.decode_batch(seqs[0], ids, n), e.decode_batch(seqs[1], ids, n)
            assert list(a) == list(b), (rows, n)
            for k in range(n):
                ids = [ca.sample_argmax(x) for x in h.step([(s, [t], [0]) for s, t in zip(seqs[2], ids)])]
                assert ids == list(a[k * rows:(k + 1) * rows]), (rows, n, k)
        last = [r.step([(s, [t], [0]) for s, t in zip(q, ids)]) for r, q in zip((g, e, h), seqs)]
        for x in last[1:]:
            assert np.array_equal(last[0].view(np.uint32), x.view(np.uint32)), rows
        for r, q in zip((g, e, h), seqs):
            for s in q:
                r.close(s)


@pytest.mark.parametrize("config,tensors", [(NILIVIK, sh.random_tensors), (BIFAZEN, sb.random_tensors)])
@pytest.mark.parametrize("f32", [False, True])
def test_weights_past_the_caches_are_the_same_weights(ca, hdev, tmp_path, monkeypatch, config, tensors, f32):
    """models too large for the caches read their weights with loads of another kind: the same logits from the same model either way"""
    folder = sh.write_model(config, tensors(config, 6), str(tmp_path / "m"))
    kept = ca.load_model(folder, hdev, seq_len=64, f32=f32)
    monkeypatch.setenv("CRABML_HIP_TEST_HOOKS", "1")
    monkeypatch.setenv("CRABML_HIP_STREAM_WEIGHTS", "1")
    past = ca.load_model(folder, hdev, seq_len=64, f32=f32)
    for rows in (1, 2, 3, 8, 16):
        a, b = [kept.open() for _ in range(rows)], [past.open() for _ in range(rows)]
        for i in range(6):
            ids = [(11 * i + 5 * k) % 60 for k in range(rows)]
            x, y = (r.step([(s, [t], [0]) for s, t in zip(q, ids)]) for r, q in ((kept, a), (past, b)))
            assert np.array_equal(x.view(np.uint32), y.view(np.uint32)), (rows, i)
        for r, q in ((kept, a), (past, b)):
            for s in q:
                r.close(s)


@pytest.mark.parametrize("fmt,shape", [("Q4_0", "tiny-hd128"), ("Q8_0", "15m"), ("Q4_K", "tiny-hd128"), ("F16", "15m"), ("Q6_K", "tiny-gqa")])
def test_a_step_by_itself_has_one_front(ca, fmt, shape):
    """a program that samples on the host pays for no embedding and first norm but its own step's (in these formats the only launch that counts as one)"""
    dev = ca.HipTensorDevice(0)
    conf, w = synth.to_hip(synth.build_model(synth.SHAPES[shape], synth.TYPE_BY_NAME[fmt], seed=22), dev)
    r = ca.HipLlamaRunner(conf, w, dev, 60, True, False)
    r.forward(3, 0)
    dev.prof_enable(True)
    for i in range(3):
        r.forward(5 + i, 1 + i)
        assert sum(x["launches"] for x in dev.prof_read() if x["stage"] == 6) == 1, i
    r.decode_greedy(9, 4)
    assert sum(x["launches"] for x in dev.prof_read() if x["stage"] == 6) == 4
    dev.prof_enable(False)


@pytest.mark.parametrize("fmt,shape", [("Q8_0", "15m"), ("Q4_K", "tiny-hd128")])
def test_a_runner_captures_several_steps_as_it_runs(ca, fmt, shape):
    """none when it is made, the sizes that a run has use for behind its first steps, and the same tokens before, during and behind that"""
    dev = ca.HipTensorDevice(0)
    conf, w = synth.to_hip(synth.build_model(synth.SHAPES[shape], synth.TYPE_BY_NAME[fmt], seed=23), dev)
    a, e = ca.HipLlamaRunner(conf, w, dev, 400, True), ca.HipLlamaRunner(conf, w, dev, 400, True, False)
    assert [a.debug_graph_steps(p) for p in (0, 100, 399)] == [(8, 0)] * 3 and e.debug_graph_steps(0) == (1, 0)
    token = 3
    for n, captured in ((1, 0), (3, 0), (7, 2), (8, 2), (6, 6), (194, 7), (20, 7)):  # (bits: eight steps, four, two)
        ids = a.decode_greedy(token, n)
        assert ids == e.decode_greedy(token, n), n
        token = ids[-1]
        assert a.debug_graph_steps(0)[1] == captured and e.debug_graph_steps(0)[1] == 0, n
    x, y = a.forward(token, 239), e.forward(token, 239)
    assert np.array_equal(x.view(np.uint32), y.view(np.uint32))


@pytest.mark.parametrize("strict,layers,steps", [(False, 32, 2), (True, 32, 1), (False, 24, 3), (True, 24, 3)])
def test_deep_models_chain_few_steps(ca, strict, layers, steps):
    """steps of 5 launches a layer and some, up to 384 launches a graph; no pairs on the strict device"""
    dev = ca.HipTensorDevice(0, strict_order=strict)
    shape = synth.ModelShape("deep", 256, 512, layers, 2, 2, 300, 64, 1e-5, None)
    conf, w = synth.to_hip(synth.build_model(shape, synth.Q4_0, seed=24), dev)
    a, e = ca.HipLlamaRunner(conf, w, dev, 60, True), ca.HipLlamaRunner(conf, w, dev, 60, True, False)
    assert a.debug_graph_steps(0) == (steps, 0)
    assert a.decode_greedy(3, 25) == e.decode_greedy(3, 25)
    assert a.debug_graph_steps(0)[1] == (1 if steps > 1 else 0)
