"""Head widths that are not whole quant blocks: wo's launch quantizes the attention row itself (fast device, Q4_0 / Q8_0)."""
import numpy as np
import pytest

from crabml_amd import synth
from oracle import oracle as o
from tests.helpers import FAST_TOL, to_oracle

pytestmark = pytest.mark.gpu
SPLIT_ALWAYS = 16  # CRABML_HIP_LLAMA_SPLIT_CHUNKS_ALWAYS: two workgroups per 32-row chunk also for short rows


@pytest.mark.parametrize("fmt", ["Q4_0", "Q8_0"])
@pytest.mark.parametrize("dim,hidden,heads,kv", [(96, 64, 2, 1), (288, 768, 6, 6), (1280, 96, 16, 4)])  # heads of 48, 48 and 80
@pytest.mark.parametrize("split", [False, True])
def test_decode_against_the_oracle(ca, fmt, dim, hidden, heads, kv, split):
    shape = synth.ModelShape("odd", dim, hidden, 2, heads, kv, 512, 32)
    model = synth.build_model(shape, synth.TYPE_BY_NAME[fmt], seed=3)
    odev = o.OracleDevice(thread_num=2)
    oconf, ow = to_oracle(model, odev)
    want = o.OracleLlamaRunner(oconf, ow, odev, 32, True)
    dev = ca.HipTensorDevice(0)
    conf, w = synth.to_hip(model, dev)
    got = ca.HipLlamaRunner(conf, w, dev, 32, True, extra_flags=SPLIT_ALWAYS if split else 0)
    errs = []
    for i, t in enumerate([1, 77, 300, 5, 6, 7]):
        a, b = got.forward(t, i), want.forward([t], i)
        errs.append(np.max(np.abs(a - b)) / np.max(np.abs(b)))
    assert max(errs) <= FAST_TOL[fmt][1], errs


@pytest.mark.parametrize("fmt", ["Q4_0", "Q8_0"])
@pytest.mark.parametrize("dim,hidden,heads,kv", [(96, 64, 2, 1), (288, 768, 6, 6), (1280, 96, 16, 4)])
@pytest.mark.parametrize("split", [False, True])
def test_the_bits_of_the_quantizers_own_launch(ca, monkeypatch, fmt, dim, hidden, heads, kv, split):
    shape = synth.ModelShape("odd", dim, hidden, 2, heads, kv, 512, 64)
    dev = ca.HipTensorDevice(0)
    conf, w = synth.to_hip(synth.build_model(shape, synth.TYPE_BY_NAME[fmt], seed=4), dev)
    a = ca.HipLlamaRunner(conf, w, dev, 64, True, extra_flags=SPLIT_ALWAYS if split else 0)
    monkeypatch.setenv("CRABML_HIP_TEST_HOOKS", "1")
    monkeypatch.setenv("CRABML_HIP_ATTN_ROW_APART", "1")  # (read when a context is made)
    b = ca.HipLlamaRunner(conf, w, dev, 64, True, extra_flags=SPLIT_ALWAYS if split else 0)
    for i in range(40):
        assert np.array_equal(a.forward((7 * i + 1) % 512, i).view(np.uint32), b.forward((7 * i + 1) % 512, i).view(np.uint32)), i
