"""matmul_vec on several rows of the rhs in one launch of the row kernels: bit for bit what a call per row gives, for every format, on both
devices.  (From 16 rows on the fast device has matrix-core kernels for some formats: those counts are left to the formats without one.)"""
import numpy as np
import pytest

from crabml_amd import synth
from tests.test_hip_gemv import HT

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["Q4_0", "Q8_0", "Q4_1", "Q5_0", "Q5_1", "Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K", "Q8_K", "F32", "F16"])
@pytest.mark.parametrize("strict", [False, True])
# rows of the matrix: less than a tile, tiles that do not divide by the eight XCDs, two rows a wave; rows of the rhs: past one launch's share
@pytest.mark.parametrize("m,k,rows", [(1, 256, 2), (77, 768, 15), (8210, 512, 5), (9, 256, 259)])
def test_rows_equal_single_calls(ca, fmt, strict, m, k, rows):
    if rows > 15 and not strict and fmt in ("Q4_0", "Q8_0", "Q4_1", "Q4_K", "Q6_K", "Q8_K"):
        rows = 15
    if fmt == "F16":
        k += 0 if strict else 2  # (fast: rows of whole 16-byte pieces are in test_hip_f16.py, past 32768 results on the matrix cores)
    rng = np.random.default_rng(m + rows)
    typ = synth.TYPE_BY_NAME[fmt]
    dev = ca.HipTensorDevice(0, False, 0, strict)
    w = ca.HipTensor.from_cpu(synth.random_blocks(rng, m * k, typ), [m, k], getattr(ca.GGMLType, HT[fmt]), dev)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    got = w.matmul_vec(ca.HipTensor.new(x.reshape(-1), [rows, k], dev)).export().reshape(rows, m)
    picks = sorted({0, 1, rows // 2, rows - 1})
    for r in picks:
        one = w.matmul_vec(ca.HipTensor.new(x[r], [k], dev)).export()
        assert np.array_equal(got[r].view(np.uint32), one.view(np.uint32)), r


@pytest.mark.parametrize("fmt,strict,m,k", [("F32", False, 262146, 8), ("Q8_0", True, 524304, 32)])
def test_more_threads_than_a_launch_holds(ca, fmt, strict, m, k):
    """256 rows of the rhs on matrices whose launch would have 2^32 threads: several launches (of too large a one only a part runs)"""
    rows = 257
    rng = np.random.default_rng(9)
    dev = ca.HipTensorDevice(0, False, 0, strict)
    w = ca.HipTensor.from_cpu(synth.random_blocks(rng, m * k, synth.TYPE_BY_NAME[fmt]), [m, k], getattr(ca.GGMLType, HT[fmt]), dev)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    got = w.matmul_vec(ca.HipTensor.new(x.reshape(-1), [rows, k], dev)).export().reshape(rows, m)
    for r in (0, 127, 254, 255, 256):
        one = w.matmul_vec(ca.HipTensor.new(x[r], [k], dev)).export()
        assert np.array_equal(got[r].view(np.uint32), one.view(np.uint32)), r


@pytest.mark.parametrize("fmt", ["F32", "F16", "Q5_K"])
# tiles of 64 rows against 256 CUs' room for 1024: seven rows of the rhs a launch and a remainder, one a launch
@pytest.mark.parametrize("m,rows", [(8210, 16), (65600, 3)])
def test_lane_per_row_kernel_over_several_launches(ca, fmt, m, rows):
    """the strict device's lane-per-row kernel takes no more rows of the rhs at once than the CUs hold lines for"""
    rng = np.random.default_rng(m)
    dev = ca.HipTensorDevice(0, False, 0, True)
    w = ca.HipTensor.from_cpu(synth.random_blocks(rng, m * 256, synth.TYPE_BY_NAME[fmt]), [m, 256], getattr(ca.GGMLType, HT[fmt]), dev)
    x = rng.standard_normal((rows, 256)).astype(np.float32)
    got = w.matmul_vec(ca.HipTensor.new(x.reshape(-1), [rows, 256], dev)).export().reshape(rows, m)
    for r in range(rows):
        one = w.matmul_vec(ca.HipTensor.new(x[r], [256], dev)).export()
        assert np.array_equal(got[r].view(np.uint32), one.view(np.uint32)), r


# rows of the rhs: one, two and four of the kernel's tiles, their remainders, several workgroups; rows of the matrix: less than a tile, remainders, tiles that do
# and do not divide by the eight XCDs; super-blocks: fewer than are on their way at once, a remainder, many
@pytest.mark.parametrize("m,k,rows", [(1, 256, 4), (15, 768, 16), (130, 1280, 17), (100, 512, 32), (256, 1024, 33), (77, 2304, 64), (129, 256, 65), (48, 14336, 130)])
@pytest.mark.parametrize("levels", ["random", "largest"])
def test_strict_q4_k_on_the_matrix_cores(ca, m, k, rows, levels):
    """several rows against one row at a time (the row kernels, which the oracle covers); `largest`: every level 15, scale and minimum 63, quant -128 or 127"""
    rng = np.random.default_rng(m + rows)
    dev = ca.HipTensorDevice(0, False, 0, True)
    raw = synth.random_blocks(rng, m * k, synth.TYPE_BY_NAME["Q4_K"])
    x = rng.standard_normal((rows, k)).astype(np.float32)
    if levels == "largest":
        raw = raw.copy()
        raw.reshape(-1, 144)[:, 4:] = 255
        x = np.where(rng.random((rows, 1)) < 0.5, 1.0, np.where(rng.random((rows, k)) < 0.5, -1.0, 0.99)).astype(np.float32)
    w = ca.HipTensor.from_cpu(raw, [m, k], ca.GGMLType.Q4K, dev)
    got = w.matmul_vec(ca.HipTensor.new(x.reshape(-1), [rows, k], dev)).export().reshape(rows, m)
    for r in range(rows):
        one = w.matmul_vec(ca.HipTensor.new(x[r], [k], dev)).export()
        assert np.array_equal(got[r].view(np.uint32), one.view(np.uint32)), r


@pytest.mark.parametrize("k", [256, 2304])
def test_strict_q4_k_rows_of_large_matrices(ca, k):
    """from 32768 rows of the matrix on a wave takes four of them, below two: the same bits"""
    m, rng, dev = 32773, np.random.default_rng(k), ca.HipTensorDevice(0, False, 0, True)
    raw = synth.random_blocks(rng, m * k, synth.TYPE_BY_NAME["Q4_K"])
    x = ca.HipTensor.new(rng.standard_normal(k).astype(np.float32), [k], dev)
    got = ca.HipTensor.from_cpu(raw, [m, k], ca.GGMLType.Q4K, dev).matmul_vec(x).export()
    size = raw.size // m
    for first, n in ((0, 77), (16384, 64), (m - 77, 77)):
        part = raw.reshape(-1)[first * size:(first + n) * size].copy()
        want = ca.HipTensor.from_cpu(part, [n, k], ca.GGMLType.Q4K, dev).matmul_vec(x).export()
        assert np.array_equal(got[first:first + n].view(np.uint32), want.view(np.uint32)), first
