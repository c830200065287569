"""F16 weights on the fast device: the row kernels (one row of the rhs; up to 32768 results of several) and the matrix-core GEMM (past that, and
the prompt pass from two rows on), against float64 on the rhs as the reference rounds it (f16, buf_f16.rs:83-97)."""
import numpy as np
import pytest

from crabml_amd import synth
from tests.helpers import FAST_TOL, GEMV_REL

pytestmark = pytest.mark.gpu

# (m, k, rows): one row; ragged m and rows; a tail of k shorter than a step of 64; k that is not whole 16-byte pieces; every tile height;
# results on either side of the GEMM's first
SHAPES = [(1, 8, 1), (5, 72, 1), (16385, 520, 1), (2050, 4104, 1), (33, 70, 1), (33, 70, 3), (1, 8, 2), (130, 72, 33), (128, 64, 2), (257, 328, 129),
          (300, 512, 256), (96, 4096, 300), (1027, 136, 65), (2048, 2048, 31), (16384, 64, 2),
          (16385, 72, 2), (1100, 200, 33), (4097, 8, 9), (10923, 136, 3)]


@pytest.mark.parametrize("m,k,rows", SHAPES)
def test_matmul_vec_f16(ca, hdev, m, k, rows):
    rng = np.random.default_rng(m * 31 + k * 7 + rows)
    w = rng.standard_normal((m, k)).astype(np.float16)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    t = ca.HipTensor.from_cpu(w.view(np.uint8).reshape(-1), [m, k], ca.GGMLType.F16, hdev)
    got = t.matmul_vec(ca.HipTensor.new(x.reshape(-1), [rows, k], hdev)).export().reshape(rows, m)
    wd, xd = w.astype(np.float64), x.astype(np.float16).astype(np.float64)
    assert np.all(np.abs(got - xd @ wd.T) <= GEMV_REL * (np.abs(xd) @ np.abs(wd).T))


@pytest.mark.parametrize("m", [37, 1037])  # row kernels, matrix cores
def test_matmul_vec_f16_infinite_and_nan_rows_stay_apart(ca, hdev, m):
    """a row of the rhs that holds an infinity or a NaN changes that row's results only; so do the weights' rows"""
    rng = np.random.default_rng(3)
    w, x = rng.standard_normal((m, 72)).astype(np.float16), rng.standard_normal((35, 72)).astype(np.float32)
    w[m - 1, 71], x[34, 71], x[5, 0] = np.inf, np.nan, np.inf
    t = ca.HipTensor.from_cpu(w.view(np.uint8).reshape(-1), [m, 72], ca.GGMLType.F16, hdev)
    got = t.matmul_vec(ca.HipTensor.new(x.reshape(-1), [35, 72], hdev)).export().reshape(35, m)
    rows = [r for r in range(35) if r not in (5, 34)]
    assert np.isfinite(got[rows][:, :m - 1]).all() and np.isinf(got[rows][:, m - 1]).all()
    assert np.isnan(got[34]).all() and not np.isfinite(got[5]).any()


@pytest.mark.parametrize("m,k,rows", [(1, 8, 3), (77, 768, 15), (4096, 512, 8), (16384, 136, 2), (127, 4104, 258)])
def test_rows_of_few_results_equal_single_calls(ca, hdev, m, k, rows):
    """up to 32768 results the row kernels take all rows of the rhs in one launch (258: two of them): the bits of a call per row"""
    rng = np.random.default_rng(m + rows)
    w, x = rng.standard_normal((m, k)).astype(np.float16), rng.standard_normal((rows, k)).astype(np.float32)
    t = ca.HipTensor.from_cpu(w.view(np.uint8).reshape(-1), [m, k], ca.GGMLType.F16, hdev)
    got = t.matmul_vec(ca.HipTensor.new(x.reshape(-1), [rows, k], hdev)).export().reshape(rows, m)
    for r in sorted({0, 1, rows // 2, rows - 1}):
        assert np.array_equal(got[r].view(np.uint32), t.matmul_vec(ca.HipTensor.new(x[r], [k], hdev)).export().view(np.uint32)), r


@pytest.mark.parametrize("rows", [2, 65, 203])
def test_prompt_pass_equals_the_token_loop(ca, rows):
    """one prompt pass (k of its GEMMs cut into pieces at this width) against the same tokens one by one"""
    shape = synth.ModelShape("f16", 2048, 2304, 1, 16, 4, 1000, 256)
    dev = ca.HipTensorDevice(0)
    conf, w = synth.to_hip(synth.build_model(shape, synth.F16, seed=4), dev)
    toks = [(13 * i + 5) % 1000 for i in range(rows)]
    a, b = ca.HipLlamaRunner(conf, w, dev, 256, True), ca.HipLlamaRunner(conf, w, dev, 256, True)
    want = [b.forward(t, i) for i, t in enumerate(toks)][-1]
    for _ in range(2):  # (the pieces' counters are left at zero)
        got = a.prefill(toks)
        assert np.max(np.abs(got - want)) <= FAST_TOL["F16"][1] * np.max(np.abs(want))
        a.reset()


# dim, hidden, heads, kv heads, vocab: rows shorter than a wave's step; ragged rows everywhere; rows past the 4096 elements that two pieces a
# thread hold; classifiers on either side of the row count that gives a wave four rows
@pytest.mark.parametrize("dim,hidden,heads,kv,vocab", [(96, 32, 3, 1, 50), (352, 544, 4, 2, 4097), (4160, 4128, 32, 8, 77), (512, 4128, 8, 8, 50)])
@pytest.mark.parametrize("kv_f16", [True, False])
def test_decode_step_against_the_scalar_order(ca, dim, hidden, heads, kv, vocab, kv_f16):
    """the fast step against the strict device (the reference's sums, its own launches) on the same tokens; the graph replays itself"""
    shape = synth.ModelShape("f16", dim, hidden, 2, heads, kv, vocab, 128, 1e-5, dim // heads // 2 * 2)
    model = synth.build_model(shape, synth.F16, seed=5)
    logits = []
    for strict in (True, False):
        dev = ca.HipTensorDevice(0, False, 0, strict)
        conf, w = synth.to_hip(model, dev)
        r = ca.HipLlamaRunner(conf, w, dev, 128, kv_f16)
        logits.append(np.array([r.forward((7 * i + 3) % vocab, i) for i in range(12)]))
        if not strict:
            r.reset()
            first = r.forward(3 % vocab, 0)
            assert np.array_equal(first, logits[1][0])  # (a replay leaves nothing behind that changes the next one)
    # 2-norms; two orders of a sum flip roundings to f16 (every rhs, cached rows, the exponential's levels), each 2^-11 of an element: up to
    # 1.2e-3 over these models where the fast device takes one launch per op, four such steps allowed
    err = np.linalg.norm(logits[1] - logits[0], axis=1) / np.linalg.norm(logits[0], axis=1)
    assert np.max(err) <= 4 * 2.0 ** -11, err


# either side of 512, 1024, 2048 and 4096 columns; classifiers either side of sixteen rows a CU, of rows of 4096 columns and of others; ffn_down of up to 1024 long rows
@pytest.mark.parametrize("dim,hidden,heads,kv,vocab", [(544, 512, 4, 4, 4095), (1024, 1056, 8, 2, 4096), (1056, 4096, 8, 4, 70), (512, 1024, 8, 2, 16400), (2080, 544, 20, 4, 4100),
                                                       (2560, 512, 20, 4, 4095), (3584, 544, 28, 4, 4100), (1024, 4096, 8, 2, 70), (4096, 512, 32, 8, 4100), (5120, 512, 40, 8, 4100)])
def test_decode_step_forms_against_the_scalar_order(ca, dim, hidden, heads, kv, vocab):
    test_decode_step_against_the_scalar_order(ca, dim, hidden, heads, kv, vocab, True)
