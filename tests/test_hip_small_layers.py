"""A small model's decode step with all its layers in one launch, against the step of five launches a layer, bit for bit."""
import ctypes
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from crabml_amd import synth

pytestmark = pytest.mark.gpu
FIVE = 134217728  # CRABML_HIP_LLAMA_NO_SMALL_LAYERS


# the smallest; heads of eight columns, as many as there are workgroups; heads that fill part of their lanes; the widest rows of each kind, with one key head
# and with as many as fit; workgroups without rows of wo or without rows of gate and up
@pytest.mark.parametrize("dim,hidden,layers,heads,kv_heads", [(32, 32, 1, 1, 1), (256, 96, 2, 32, 8), (288, 768, 3, 6, 6), (896, 1024, 2, 14, 1), (512, 1024, 3, 8, 4),
                                                              (64, 992, 2, 2, 1), (320, 64, 5, 5, 5)])
@pytest.mark.parametrize("fmt", ["Q8_0", "Q4_0"])
def test_one_launch_equals_five_a_layer(ca, fmt, dim, hidden, layers, heads, kv_heads):
    dev = ca.HipTensorDevice(0)
    shape = synth.ModelShape("small", dim, hidden, layers, heads, kv_heads, 300, 160, 1e-5, None)
    conf, w = synth.to_hip(synth.build_model(shape, synth.TYPE_BY_NAME[fmt], seed=31), dev)
    seq = 150  # (past the first 64 positions, and to the last)
    one, eager, five = (ca.HipLlamaRunner(conf, w, dev, seq, True, g, extra_flags=f) for g, f in ((True, 0), (False, 0), (True, FIVE)))
    wgs = max((dim + 2 * (dim // heads * kv_heads) + 31) // 32, hidden // 32, heads)
    assert (one.debug_small_layers(), eager.debug_small_layers(), five.debug_small_layers()) == (wgs, wgs, 0)
    pos, token = 0, 3
    for n in (1, 5, 58, 2, 70):
        ids = one.decode_greedy(token, n)
        assert ids == five.decode_greedy(token, n) == eager.decode_greedy(token, n), (pos, n)
        pos, token = pos + n, ids[-1]
    while pos < seq:
        x, y, z = one.forward(token, pos), five.forward(token, pos), eager.forward(token, pos)
        assert np.isfinite(x).all() and np.array_equal(x.view(np.uint32), y.view(np.uint32)) and np.array_equal(x.view(np.uint32), z.view(np.uint32)), pos
        pos, token = pos + 1, (token * 7 + pos) % 300
    # a prompt behind it, and steps behind the prompt
    prompt = [(5 * i + 1) % 300 for i in range(40)]
    one.reset()
    five.reset()
    x, y = one.prefill(prompt), five.prefill(prompt)
    assert np.array_equal(np.asarray(x).view(np.uint32), np.asarray(y).view(np.uint32))
    assert one.decode_greedy(9, 30) == five.decode_greedy(9, 30)


# several passes of 128 over a head's cached rows, to the end of the cache (heads of 48) and across the position from which the step's attention is k_attn_flash
# (heads of 64: 57344 / 64 = 896 cached)
@pytest.mark.parametrize("dim,heads,seq,until", [(288, 6, 640, 640), (512, 8, 912, 895)])
@pytest.mark.parametrize("fmt", ["Q8_0", "Q4_0"])
def test_one_launch_equals_five_a_layer_at_every_position(ca, fmt, dim, heads, seq, until):
    dev = ca.HipTensorDevice(0)
    shape = synth.ModelShape("small", dim, 768, 2, heads, heads // 2, 300, seq, 1e-5, None)
    conf, w = synth.to_hip(synth.build_model(shape, synth.TYPE_BY_NAME[fmt], seed=34), dev)
    one, five = (ca.HipLlamaRunner(conf, w, dev, seq, True, extra_flags=f) for f in (0, FIVE))
    assert one.debug_small_layers() > 0 and five.debug_small_layers() == 0
    assert [one.debug_graphs(p)[0] == 0 for p in (0, until - 1, min(until, seq - 1))] == [True, True, until == seq]
    pos, token = 0, 3
    for n in (190, 3, 127, 3, 125, 3, until - 467):
        assert one.decode_greedy(token, n) == (ids := five.decode_greedy(token, n)), (pos, n)
        pos, token = pos + n, ids[-1]
        x, y = one.forward(token, pos), five.forward(token, pos)
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32)), pos
        pos += 1
    while pos < seq:
        x, y = one.forward(token, pos), five.forward(token, pos)
        assert np.isfinite(x).all() and np.array_equal(x.view(np.uint32), y.view(np.uint32)), pos
        pos, token = pos + 1, (token * 7 + pos) % 300
    for layer in range(2):
        for v in (False, True):
            assert np.array_equal(one.debug_kv(layer, v, True), five.debug_kv(layer, v, True))


@pytest.mark.parametrize("fmt,out", [("Q8_0", "Q6_K"), ("Q4_0", "Q6_K"), ("Q4_0", "F16"), ("Q8_0", "Q4_1")])
def test_a_classifier_of_another_type_reads_the_row_behind_the_one_launch(ca, fmt, out):
    dev = ca.HipTensorDevice(0)
    shape = synth.ModelShape("small", 256, 512, 3, 4, 2, 300, 60, 1e-5, None)
    conf, w = synth.to_hip(synth.build_model(shape, synth.TYPE_BY_NAME[fmt], seed=35, output_type=synth.TYPE_BY_NAME[out]), dev)
    one, five = (ca.HipLlamaRunner(conf, w, dev, 60, True, extra_flags=f) for f in (0, FIVE))
    assert one.debug_small_layers() > 0 and five.debug_small_layers() == 0
    assert one.decode_greedy(3, 40) == five.decode_greedy(3, 40)
    for pos in range(40, 60):
        x, y = one.forward(pos, pos), five.forward(pos, pos)
        assert np.isfinite(x).all() and np.array_equal(x.view(np.uint32), y.view(np.uint32)), pos


def test_contexts_past_the_reserved_workgroups(ca):
    """more contexts than half of the CUs hold, each on a stream of its own and all of them under way at once"""
    shape = synth.ModelShape("small", 288, 768, 2, 6, 6, 300, 160, 1e-5, None)
    model, runners = synth.build_model(shape, synth.Q8_0, seed=32), []
    for i in range(8):
        dev = ca.HipTensorDevice(0)
        runners.append(ca.HipLlamaRunner(*synth.to_hip(model, dev), dev, 100, True))
    assert [r.debug_small_layers() for r in runners] == [27] * 4 + [0] * 4
    dev = ca.HipTensorDevice(0)
    want = ca.HipLlamaRunner(*synth.to_hip(model, dev), dev, 100, True, extra_flags=FIVE).decode_greedy(3, 90)
    with ThreadPoolExecutor(8) as pool:
        ids = list(pool.map(lambda r: r.decode_greedy(3, 90), runners))
    assert all(x == want for x in ids)
    assert [r.debug_small_layers() for r in runners] == [27] * 4 + [0] * 4  # (all of them met)


@pytest.mark.parametrize("graph", [True, False])
def test_workgroups_that_do_not_meet(ca, monkeypatch, graph):
    """one poll instead of a million: no gather is met.  The call that finds out is made again in launches per layer, and the context stays with them; steps
    that nobody has looked at cannot be made again: an error until the context is reset"""
    shape = synth.ModelShape("small", 288, 768, 3, 6, 6, 300, 160, 1e-5, None)
    model = synth.build_model(shape, synth.Q8_0, seed=33)
    dev = ca.HipTensorDevice(0)
    conf, w = synth.to_hip(model, dev)
    five = ca.HipLlamaRunner(conf, w, dev, 100, True, graph, extra_flags=FIVE)
    ids = five.decode_greedy(3, 40)
    logits = five.forward(ids[-1], 40).view(np.uint32)
    monkeypatch.setenv("CRABML_HIP_TEST_HOOKS", "1")
    monkeypatch.setenv("CRABML_HIP_SMALL_POLLS", "1")
    by_steps, by_run, unseen, prompt = (ca.HipLlamaRunner(conf, w, dev, 100, True, graph) for _ in range(4))
    assert [r.debug_small_layers() for r in (by_steps, by_run, unseen, prompt)] == [27] * 4
    token = 3
    for pos in range(40):
        x = by_steps.forward(token, pos)
        token = int(ca.sample_argmax(x))
        assert token == ids[pos]
    assert np.array_equal(by_steps.forward(ids[-1], 40).view(np.uint32), logits)
    assert by_run.decode_greedy(3, 40) == ids and np.array_equal(by_run.forward(ids[-1], 40).view(np.uint32), logits)
    unseen.forward_async(3, 0)
    for call in (lambda: unseen.forward(ids[0], 1), lambda: unseen.forward(ids[0], 2), lambda: unseen.decode_greedy(ids[0], 2), lambda: unseen.prefill([1, 2])):
        with pytest.raises(ca.CrabmlError, match="not to be used"):
            call()
    unseen.reset()
    assert unseen.decode_greedy(3, 40) == ids
    prompt.forward_async(3, 0)
    with pytest.raises(ca.CrabmlError, match="not to be used"):
        prompt.prefill([1, 2, 3])
    assert [r.debug_small_layers() for r in (by_steps, by_run, unseen, prompt)] == [0] * 4
    # what they had reserved is there again
    monkeypatch.delenv("CRABML_HIP_SMALL_POLLS")
    more = [ca.HipLlamaRunner(conf, w, dev, 100, True, graph) for _ in range(4)]
    assert [r.debug_small_layers() for r in more] == [27] * 4
    assert all(r.decode_greedy(3, 40) == ids for r in more)


def test_the_computed_exp_is_the_table(ca):
    """the step's exp against the device's table, every f16"""
    lib = ctypes.CDLL(ca.LIB_PATH)
    dev = ca.HipTensorDevice(0)
    got, table = np.zeros(65536, np.uint16), np.zeros(65536, np.uint16)
    assert lib.crabml_hip_debug_exp_of_f16(ctypes.c_void_p(dev.raw_handle()), got.ctypes.data_as(ctypes.c_void_p), table.ctypes.data_as(ctypes.c_void_p)) == 0
    nan = (table & 0x7fff) > 0x7c00
    assert np.array_equal(got[~nan], table[~nan]) and np.all((got[nan] & 0x7fff) > 0x7c00)
