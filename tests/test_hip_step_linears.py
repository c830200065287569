"""The matrix-core linears of a decode step (3 to 16 sequences) at sizes that reach every form of them -- 32 weight rows a workgroup, sixteen
waves, rows and pieces of k that do not divide -- on one-layer models of both designs against the plain implementations."""
import numpy as np
import pytest

from crabml_amd import synth_bifazen as sb
from crabml_amd import synth_hybrid as sh
from tests import bifazen_oracle as bo
from tests import hybrid_oracle as ho

pytestmark = pytest.mark.gpu


def nilivik(width, ff, vocab):
    return sh.config(width, vocab, [sh.layer(4, 2, 24, 40, 100, 3, 16, 24, ff)]), sh.random_tensors, ho


def bifazen(width, ff, vocab):
    return sb.config(width, vocab, [sb.latent(4, 16, 6, 24, 40, 50, ff), sb.attention(4, 2, 24, 40, 50, ff)], streams=3), sb.random_tensors, bo


# width, ff, vocab: everything on 16 rows and eight waves; sixteen waves in front of the residual; 32 rows (the vocabulary, Bifazen's gate | up)
@pytest.mark.parametrize("width,ff,vocab", [(72, 90, 50), (2090, 4104, 60), (328, 8200, 16401)])
@pytest.mark.parametrize("design", [nilivik, bifazen])
@pytest.mark.parametrize("f32", [False, True])
def test_batched_steps(ca, hdev, tmp_path, design, width, ff, vocab, f32):
    config, tensors, oracle = design(width, ff, vocab)
    bits = tensors(config, 11, pool=1 << 20)
    r = ca.load_model(sh.write_model(config, bits, str(tmp_path)), hdev, seq_len=16, f32=f32)
    floats = {k: sh.from_bf16(v) for k, v in bits.items()}
    rng = np.random.default_rng(width)
    toks = rng.integers(0, vocab, (16, 3))
    want = [oracle.forward(config, floats, t) for t in toks[:3]]
    for batch in (1, 3, 6, 16, 2):  # (f32: one, two and four groups of rows; the forms for few rows in between: they share the step's buffers)
        seqs = [r.open() for _ in range(batch)]
        got = np.array([r.step([(s, [int(toks[i, t])], [0]) for i, s in enumerate(seqs)]) for t in range(3)])  # [step, sequence, vocab]
        for s in seqs:
            r.close(s)
        for i in range(min(batch, 3)):
            d = got[:, i] - want[i]
            # the bounds of the designs' own tests
            assert np.sqrt((d * d).mean(axis=1)).max() <= (2e-5 if f32 else 2.5e-2) * np.sqrt((want[i] ** 2).mean()), (batch, i)


# the classifier in one round of workgroups of 32, 48 and 64 rows, a tile and four rows past each line (of few columns: eight waves with a piece of k each or none; of
# 2090: eight or sixteen with several, of 2048: sixteen with two), in rounds of 32 and 48 (either side of one and a half of those a CU, of two of them with long rows, rows
# of 8 KB); two workgroups to a k of 3104 and 3072 columns with a tile that 72 and 2048 rows do not fill and fill
@pytest.mark.parametrize("width,ff,vocab", [(72, 3100, 4100), (72, 90, 8196), (72, 90, 12292), (72, 90, 16388), (2090, 90, 4100), (2090, 90, 8196), (2090, 90, 12292), (2048, 3072, 50),
                                            (2048, 90, 4100), (72, 90, 18434), (2090, 90, 24580), (4096, 90, 16388)])
def test_one_round_of_workgroups(ca, hdev, tmp_path, width, ff, vocab):
    config, tensors, oracle = nilivik(width, ff, vocab)
    bits = tensors(config, 12, pool=1 << 20)
    r = ca.load_model(sh.write_model(config, bits, str(tmp_path)), hdev, seq_len=16)
    toks = np.random.default_rng(vocab + ff).integers(0, vocab, (16, 3))
    want = oracle.forward(config, {k: sh.from_bf16(v) for k, v in bits.items()}, toks[0])
    seen = []
    for batch in (3, 8, 9, 16):
        seqs = [r.open() for _ in range(batch)]
        got = np.array([r.step([(s, [int(toks[i, t])], [0]) for i, s in enumerate(seqs)])[0] for t in range(3)])
        for s in seqs:
            r.close(s)
        d = got - want
        assert np.sqrt((d * d).mean(axis=1)).max() <= 2.5e-2 * np.sqrt((want ** 2).mean()), batch  # (the design's own bound)
        seen.append(got)
    assert all(np.array_equal(s, seen[0]) for s in seen)  # (bit for bit: a sequence's logits do not depend on how many share its step)


# k shared by two workgroups (nine rows and more) behind every input and in front of every output that takes it, and by the halves of one (up to eight): the output
# projection with 68 and 64 pieces of the linear branch's square sum, without any, into the residual and into streams; normed linears of 3104 columns (194 pieces of the
# square sum) in front of xIELU, GELU * up and the classifier
@pytest.mark.parametrize("design,oracle,config", [
    (sh, ho, sh.config(200, 50, [sh.layer(8, 1, 16, 128, 24, 17, 16, 128, 90)] * 2)),
    (sh, ho, sh.config(84, 50, [sh.layer(16, 4, 16, 128, 24, 16, 16, 128, 90)] * 2)),
    (sh, ho, sh.config(3104, 50, [sh.layer(4, 2, 24, 40, 100, 3, 16, 24, 90)])),
    (sb, bo, sb.config(3104, 50, [sb.latent(4, 16, 6, 24, 40, 50, 90), sb.attention(4, 2, 24, 40, 50, 90)], streams=3)),
    (sb, bo, sb.config(84, 90, [sb.latent(18, 16, 8, 200, 40, 70, 90), sb.attention(16, 2, 16, 200, 24, 90)], streams=2))])
def test_shared_k_gives_the_bits_of_few_rows(ca, hdev, tmp_path, design, oracle, config):
    bits = design.random_tensors(config, 13, pool=1 << 20)
    r = ca.load_model(sh.write_model(config, bits, str(tmp_path)), hdev, seq_len=16)
    toks = np.random.default_rng(config["width"]).integers(0, config["vocab"], (16, 10))
    floats = {k: sh.from_bf16(v) for k, v in bits.items()}
    want = np.array([oracle.forward(config, floats, t) for t in toks[:3]])
    seen = []
    for batch in (3, 8, 9, 16):
        seqs = [r.open() for _ in range(batch)]
        got = np.array([r.step([(s, [int(toks[i, t])], [0]) for i, s in enumerate(seqs)])[:3] for t in range(10)]).transpose(1, 0, 2)  # [sequence, step, vocab]
        for s in seqs:
            r.close(s)
        d = got - want
        assert np.sqrt((d * d).mean(axis=2)).max() <= 2.5e-2 * np.sqrt((want ** 2).mean()), batch  # (the designs' own bound)
        seen.append(got)
    for other in seen[1:]:
        assert np.array_equal(other.view(np.uint32), seen[0].view(np.uint32))


# columns: those of the steps in flight, one octet more; one staged segment of one row, of two, of eight (8192, 4096, 1024 elements), and one octet more
@pytest.mark.parametrize("m,k", [(70, 2048), (70, 2056), (515, 4096), (33, 4104), (66, 8200), (17, 1032), (16389, 2056)])
def test_row_kernels_over_long_rows(ca, hdev, m, k):
    rng = np.random.default_rng(k + m)
    bits = sh.to_bf16(rng.standard_normal((m, k)).astype(np.float32))
    w = sh.from_bf16(bits).astype(np.float64)
    t = ca.HipTensor.from_cpu(bits.view(np.uint8).reshape(-1), [m, k], ca.GGMLType.BF16, hdev)
    for b in (1, 2, 3, 5, 8, 9, 16):
        x = rng.standard_normal((b, k)).astype(np.float32)
        got = t.matmul_vec(ca.HipTensor.new(x.reshape(-1), [b, k], hdev)).export().reshape(b, m)
        # (f32 sums of k products, k / 64 of them in a lane's chain: 2 + k / 64 roundings of 2^-24 each at the most, of the products' absolute values)
        bound = (2 + k / 64) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T)
        assert (np.abs(got - x.astype(np.float64) @ w.T) <= bound).all(), b


# one and two rows, either side of every line of the forms: 512, 1024, 2048 and 4096 columns; 1024, 4096, 8192 and 16384 rows of weights
@pytest.mark.parametrize("k", [8, 512, 520, 1024, 1032, 2040, 2048, 2056, 4096, 4104])
@pytest.mark.parametrize("m", [3, 1024, 1025, 4097, 8193, 16384])
def test_row_forms(ca, hdev, m, k):
    rng = np.random.default_rng(k + m)
    bits = sh.to_bf16(rng.standard_normal((m, k)).astype(np.float32))
    w = sh.from_bf16(bits)
    t = ca.HipTensor.from_cpu(bits.view(np.uint8).reshape(-1), [m, k], ca.GGMLType.BF16, hdev)
    x = rng.standard_normal((2, k)).astype(np.float32)
    # (as above, the sums of the reference in 32 bits as well: k more roundings at the most)
    bound = (2 + k / 64 + k) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T)
    for b in (1, 2):
        got = t.matmul_vec(ca.HipTensor.new(x[:b].reshape(-1), [b, k], hdev)).export().reshape(b, m)
        assert (np.abs(got - x[:b] @ w.T) <= bound[:b]).all(), b


# one and two rows of both designs, the norm's gain one number or a vector: classifiers from 16384 rows on of more than 1024 and of more than 4096 columns, of more than 2048
# rows; gate | up of 2048 rows and a pair more, of few columns and many; residuals behind more than 4096 columns, of 2048 rows and more, and behind 8192
@pytest.mark.parametrize("width,ff,vocab", [(1032, 90, 16388), (2048, 90, 16384), (4104, 90, 16384), (2056, 1024, 2049), (2056, 1026, 2048), (328, 1024, 50), (328, 1026, 50),
                                            (2056, 4104, 50), (2048, 4104, 50), (2056, 8192, 50)])
@pytest.mark.parametrize("design", [nilivik, bifazen])
def test_one_and_two_rows(ca, hdev, tmp_path, design, width, ff, vocab):
    config, tensors, oracle = design(width, ff, vocab)
    bits = tensors(config, 14, pool=1 << 20)
    r = ca.load_model(sh.write_model(config, bits, str(tmp_path)), hdev, seq_len=16)
    floats = {k: sh.from_bf16(v) for k, v in bits.items()}
    toks = np.random.default_rng(width + ff).integers(0, vocab, (2, 3))
    want = np.array([oracle.forward(config, floats, t) for t in toks])
    for batch in (1, 2):
        seqs = [r.open() for _ in range(batch)]
        got = np.array([r.step([(s, [int(toks[i, t])], [0]) for i, s in enumerate(seqs)]) for t in range(3)]).transpose(1, 0, 2)
        for s in seqs:
            r.close(s)
        d = got - want[:batch]
        assert np.sqrt((d * d).mean(axis=2)).max() <= 2.5e-2 * np.sqrt((want ** 2).mean()), batch  # (the designs' own bound)
