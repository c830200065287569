"""The decode step's mixers at the edges of their workgroups -- head widths of every class, heads that do not divide into a workgroup's, cached
rows around a wave's request, a round, what one workgroup keeps to itself and what the others share -- on one-layer models against the oracles."""
import numpy as np
import pytest

from crabml_amd import synth_bifazen as sb
from crabml_amd import synth_hybrid as sh
from tests import bifazen_oracle as bo
from tests import hybrid_oracle as ho

pytestmark = pytest.mark.gpu
# relative to the logits' rms: f32 sums in another order; bf16 rows, the wider of the two designs' whole-model bounds
TOL = {True: 2e-5, False: 2.5e-2}


def chunked(heads, kv, dim, vdim):
    # (three linear heads of one slice or two: an odd number of them, two to a workgroup)
    return sh.config(64, 50, [sh.layer(heads, kv, dim, vdim, 400, 3, 8, 40, None)], embed_scale=8.0), sh.random_tensors, ho


def windowed(heads, kv, dim, vdim):
    return sb.config(64, 50, [sb.attention(heads, kv, dim, vdim, 290, None)], streams=1), sb.random_tensors, bo


@pytest.mark.parametrize("heads,kv,dim,vdim", [(5, 1, 24, 64), (2, 2, 128, 72), (6, 1, 200, 256)])
@pytest.mark.parametrize("design", [chunked, windowed])
@pytest.mark.parametrize("f32", [True, False])
def test_decoded_rows(ca, hdev, tmp_path, design, heads, kv, dim, vdim, f32):
    config, tensors, oracle = design(heads, kv, dim, vdim)
    bits = tensors(config, 7)
    r = ca.load_model(sh.write_model(config, bits, str(tmp_path)), hdev, seq_len=420, f32=f32)
    toks = [int(x) for x in np.random.default_rng(dim).integers(0, 50, 405)]
    want = np.asarray(oracle.forward(config, {k: sh.from_bf16(v) for k, v in bits.items()}, toks), np.float64)
    # decoded from position p on, for rows p + 1, ..: 1-9, 31-34, 63-66, 127-130 and 255-258 (one workgroup, then shares of 64 rows: from 65 to 257, by
    # width and format), the ring's and the chunk's turn
    for p, n in ((0, 9), (30, 4), (62, 4), (126, 4), (254, 4), (288, 5), (382, 4), (398, 5)):
        s = r.open()
        if p:
            r.step([(s, toks[:p], [])])
        got = np.asarray([r.step([(s, [x], [0])])[0] for x in toks[p:p + n]], np.float64)
        r.close(s)
        d = got - want[p:p + n]
        assert np.max(np.sqrt((d * d).mean(axis=-1))) <= TOL[f32] * np.sqrt((want * want).mean()), p


# as many shares of the rows as 256 CUs give 16 sequences: one, two and four, of unequal lengths
@pytest.mark.parametrize("heads,kv,dim,vdim", [(16, 16, 8, 16), (8, 8, 136, 24), (16, 4, 72, 128)])
@pytest.mark.parametrize("design", [chunked, windowed])
@pytest.mark.parametrize("f32", [True, False])
def test_sixteen_sequences_of_unequal_lengths(ca, hdev, tmp_path, design, heads, kv, dim, vdim, f32):
    config, tensors, oracle = design(heads, kv, dim, vdim)
    bits = tensors(config, 8)
    r = ca.load_model(sh.write_model(config, bits, str(tmp_path)), hdev, seq_len=420, f32=f32)
    toks = [int(x) for x in np.random.default_rng(vdim).integers(0, 50, 404)]
    want = np.asarray(oracle.forward(config, {k: sh.from_bf16(v) for k, v in bits.items()}, toks), np.float64)
    lengths = [0, 1, 62, 64, 100, 126, 127, 128, 190, 192, 254, 256, 287, 320, 383, 399]
    seqs = [r.open() for _ in lengths]
    for s, n in zip(seqs, lengths):
        if n:
            r.step([(s, toks[:n], [])])
    for t in range(4):
        got = np.asarray(r.step([(s, [toks[n + t]], [0]) for s, n in zip(seqs, lengths)]), np.float64)
        d = got - want[[n + t for n in lengths]]
        assert np.max(np.sqrt((d * d).mean(axis=-1))) <= TOL[f32] * np.sqrt((want * want).mean()), t
    for s in seqs:
        r.close(s)
