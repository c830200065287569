"""Rules of the launches that the host decides by arithmetic alone (CPU): what they give over the sizes that they are asked about."""
import ctypes

import pytest

import crabml_amd

lib = ctypes.CDLL(crabml_amd.LIB_PATH)


def rhs_rows(m):
    rows = ctypes.c_size_t()
    assert lib.crabml_hip_debug_rhs_rows(ctypes.c_size_t(m), ctypes.byref(rows)) == 0
    return rows.value


# rows of the matrix a workgroup takes, its threads: f32 / f16 / bf16 rows, quantized rows (one or two a wave), the strict device's
@pytest.mark.parametrize("per_wg,threads", [(4, 256), (8, 256), (16, 256), (2, 128), (4, 128), (64, 64)])
def test_several_rhs_rows_stay_one_legal_launch(per_wg, threads):
    for m in [1, 7, 4096, 128256, 262080, 262141, 262144, 262146, 524287, 524304, 1 << 20, 12345678, 1 << 25, (1 << 26) - 64]:
        rows = rhs_rows(m)
        tiles = -(-m // per_wg)
        tiles = -(-tiles // 8) * 8 if rows > 1 else tiles
        assert 1 <= rows <= 256 and tiles * rows * threads < 1 << 32, (m, rows)
    assert rhs_rows(128256) == 256 and rhs_rows(262144) == 255  # (no fewer than fit)


@pytest.mark.parametrize("n_cu", [1, 80, 256])
def test_shares_of_cached_rows(n_cu):
    """the hybrid step's attention: no more workgroups than CUs beside one per (sequence, kv head, head block), no share without 64 rows to take"""
    for per in (1, 2, 3, 16, 48, 255, 256, 257, 4096):
        for rows in (1, 63, 64, 65, 700, 2048, 100000):
            n = ctypes.c_int32()
            assert lib.crabml_hip_debug_mix_shares(n_cu, per, rows, ctypes.byref(n)) == 0
            assert 1 <= n.value <= -(-rows // 64) and n.value * per <= max(n_cu, per)
            assert n.value == -(-rows // 64) or (n.value + 1) * per > n_cu  # (no fewer than fit)


@pytest.mark.parametrize("row_bytes,row_bytes2", [(4096, 0), (4096, 256), (2304, 144), (16384, 0), (32768, 2048)])
def test_weights_touched_ahead_fit_the_l2s(row_bytes, row_bytes2):
    """a matrix that the L2s hold (32 MB) is touched ahead whole, a larger one not at all"""
    for rows in (2, 8, 16, 32):
        for m in (32, 2048, 4096, 7264, 8192, 32768, 1 << 20):
            n = ctypes.c_size_t()
            assert lib.crabml_hip_debug_prefetch(m & 1, ctypes.c_size_t(1 << 30), m, rows, ctypes.c_size_t(row_bytes), ctypes.c_size_t(row_bytes2), ctypes.byref(n)) == 0
            all_of_it = m * (row_bytes + row_bytes2)
            assert n.value == (all_of_it if all_of_it <= 32 << 20 else 0), (m, rows, n.value)


@pytest.mark.parametrize("hybrid,gigabytes,touched", [(0, 1.3, True), (0, 2.3, True), (0, 3.34, True), (0, 4.22, False), (0, 6.1, False), (1, 0.65, True), (1, 1.2, True),
                                                      (1, 2.2, False), (1, 4.2, False)])
def test_weights_are_touched_ahead_where_that_won(hybrid, gigabytes, touched):
    """sizes of models at which a step was timed with and without"""
    n = ctypes.c_size_t()
    assert lib.crabml_hip_debug_prefetch(hybrid, ctypes.c_size_t(int(gigabytes * 1e9)), 4096, 32, ctypes.c_size_t(2048), ctypes.c_size_t(256), ctypes.byref(n)) == 0
    assert (n.value > 0) == touched


def test_rows_of_the_residual_linears():
    """k_gemv_res_nq: a chunk of 32 rows or half of one; k_gemv_res_ord: four waves of two rows; k_gemv_res: two waves of one"""
    for args, want in {(1, 0, 1): 32, (1, 1, 1): 32, (1, 0, 2): 16, (1, 1, 2): 16, (0, 1, 1): 8, (0, 1, 2): 8, (0, 0, 1): 2, (0, 0, 2): 2}.items():
        rows = ctypes.c_int32()
        assert lib.crabml_hip_debug_residual_rows(*args, ctypes.byref(rows)) == 0
        assert rows.value == want, args


def test_rows_of_a_steps_linears():
    """bf16 rows (behind no norm, or where there are no more than sixteen weight rows a CU): eight weight rows a workgroup for up to eight of them where sixteen leave half of the CUs idle and the rows are long, thirty-two from 16384 on; f32
    rows never eight.  What the mixer touches ahead of w_o is cut by the same rule."""
    for (bf16, n, k, nb), want in {(1, 2048, 8192, 3): 8, (1, 2048, 2048, 8): 8, (1, 2048, 2048, 9): 16, (1, 2049, 8192, 4): 16, (1, 2048, 2047, 4): 16, (1, 72, 4096, 4): 8,
                                   (0, 2048, 8192, 4): 16, (0, 16384, 2048, 4): 32, (1, 16384, 2048, 4): 32, (1, 16383, 2048, 16): 16}.items():
        rows = ctypes.c_int32()
        assert lib.crabml_hip_debug_step_linear_rows(bf16, n, k, nb, 256, ctypes.byref(rows)) == 0
        assert rows.value == want, (bf16, n, k, nb)


def graph_steps(nodes, seq_len, left=0, made=0, have=0):
    top, place = ctypes.c_int32(), ctypes.c_int32()
    assert lib.crabml_hip_debug_graph_steps(ctypes.c_size_t(nodes), ctypes.c_size_t(seq_len), ctypes.c_size_t(left), ctypes.c_size_t(made), have, ctypes.byref(top),
                                            ctypes.byref(place)) == 0
    return top.value, place.value


def test_graphs_of_several_steps_are_bounded():
    for nodes in (1, 14, 23, 31, 44, 63, 123, 161, 192, 193, 243, 1000):
        for seq_len in (1, 2, 3, 15, 16, 400, 8192):
            n = graph_steps(nodes, seq_len)[0]
            assert 1 <= n <= 8 and (n == 1 or (n * nodes <= 384 and 2 * n <= seq_len)), (nodes, seq_len)
    assert graph_steps(23, 8192)[0] == 8 and graph_steps(123, 8192)[0] == 3 and graph_steps(193, 8192)[0] == 1


@pytest.mark.parametrize("nodes", [23, 50, 63, 90, 123, 180, 250])
def test_a_run_captures_behind_its_own_steps(nodes):
    """a capture (at most 2 us a launch) only while steps of the same run keep the GPU busy (4 us a launch), none that the run does not use, and the same run
    once more goes through graphs from its first step on"""
    top = graph_steps(nodes, 8192)[0]
    for n in range(1, 120):
        have, made, launches = 0, 0, 0
        while made < n:
            place = graph_steps(nodes, 8192, n - made, made, have)[1]
            size = 1 if place < 0 else top >> place
            assert size <= n - made and (place < 0 or size >= 2)
            if place >= 0 and not have >> place & 1:
                assert 4 * made >= 2 * size and (place == 0 or n - made < 2 * size), (n, made, size)
                have |= 1 << place
            made += size
            launches += 1
        assert made == n
        if top > 1 and n >= 2 * top:
            assert have & 1 and launches <= top // 2 + 1 + n // top + 3, (n, launches)
        made = 0
        while made < n:
            place = graph_steps(nodes, 8192, n - made, made, have)[1]
            if made == 0 and have:
                assert place >= 0, n
            have |= 1 << place if place >= 0 else 0
            made += 1 if place < 0 else top >> place


@pytest.mark.parametrize("dtype,rows,k,b,narrow_us,wide_us", [
    (2, (256, 0, 0), 256, 300, 5.9, 7.8), (2, (256, 64, 64), 256, 128, 6.0, 7.7), (2, (768, 768, 0), 256, 300, 6.4, 8.4), (2, (1536, 0, 0), 1536, 128, 10.1, 11.9),
    (2, (3072, 0, 0), 3072, 65, 10.4, 13.5), (2, (3072, 0, 0), 3072, 300, 24.2, 13.6), (2, (1280, 320, 320), 1280, 300, 13.4, 11.4), (2, (3072, 0, 0), 8192, 300, 47.3, 27.1),
    (2, (4096, 1024, 1024), 4096, 128, 26.9, 20.3), (3, (1536, 0, 0), 1536, 128, 9.8, 12.2), (3, (1536, 384, 384), 1536, 1000, 31.7, 14.3), (8, (1536, 0, 0), 4096, 300, 21.3, 13.3),
    (8, (4096, 0, 0), 4096, 1000, 56.7, 39.6), (12, (256, 64, 64), 256, 65, 4.3, 7.2), (12, (1280, 0, 0), 3584, 65, 11.5, 16.4), (12, (1536, 0, 0), 1536, 300, 7.0, 12.8),
    (12, (4096, 0, 0), 11008, 65, 50.6, 22.6), (12, (2048, 512, 512), 2048, 700, 34.1, 17.1), (14, (1280, 0, 0), 3584, 65, 17.4, 21.5), (14, (1536, 384, 384), 1536, 65, 12.6, 15.9),
    (14, (1536, 384, 384), 1536, 1000, 33.6, 17.6), (14, (3072, 0, 0), 8192, 65, 22.5, 15.6)])
def test_prompt_gemm_runs_the_faster_kernel(dtype, rows, k, b, narrow_us, wide_us):
    """launches that were timed with both"""
    wide, size = ctypes.c_int32(), ctypes.c_size_t
    assert lib.crabml_hip_debug_prompt_gemm(dtype, size(rows[0]), size(rows[1]), size(rows[2]), size(k), size(b), 256, size(2048 * max(sum(rows), 4096)), 1, ctypes.byref(wide)) == 0
    assert wide.value == (wide_us < narrow_us)


@pytest.mark.parametrize("hidden,rows,waves", [
    (14336, 300, 4), (14336, 384, 4), (14336, 640, 4), (11008, 450, 4), (8192, 700, 4), (8192, 200, 4), (8640, 200, 4), (8640, 512, 4), (7680, 896, 4),
    (14336, 130, 8), (14336, 256, 8), (14336, 512, 8), (14336, 768, 8), (14336, 1024, 8), (8192, 300, 8), (8640, 300, 8), (8640, 850, 8), (16384, 200, 8)])
def test_gate_up_takes_eight_waves_where_they_won(hidden, rows, waves):
    """sizes at which both were timed"""
    n = ctypes.c_int32()
    assert lib.crabml_hip_debug_gateup_waves(ctypes.c_size_t(hidden), ctypes.c_size_t(rows), 256, ctypes.byref(n)) == 0
    assert n.value == waves


@pytest.mark.parametrize("k", [256, 512, 2816, 4096, 14336])
@pytest.mark.parametrize("rows", [(4096, 0, 0), (4096, 1024, 1024), (1088, 1088, 0), (300, 0, 0)])
def test_prompt_gemm_tiles_cover_k(rows, k):
    """every plan of the wide prompt GEMM: pieces of whole super-blocks, none of them empty where they meet in memory, partial outputs inside the scratch, no
    pieces in memory for gate | up, Q6_K without the tile its registers do not hold"""
    out = (ctypes.c_int32 * 4)()
    size = ctypes.c_size_t
    for dtype in (2, 14):
        for b in (65, 96, 97, 128, 203, 513, 1024, 3000):
            for ws in (0, 1 << 22, 1 << 26):
                for pair in (0, 1) if rows[1] == rows[0] else (0,):
                    assert lib.crabml_hip_debug_wide_tile(dtype, size(rows[0]), size(rows[1]), size(rows[2]), size(k), size(b), pair, 256, size(ws), out) == 0
                    f, t, groups, pieces = out
                    assert (f, t, groups) in [(4, 8, 1), (4, 6, 1), (2, 8, 1), (2, 6, 1), (2, 8, 2), (2, 6, 2)]
                    assert dtype != 14 or (f, t) != (4, 8)
                    assert not pair or pieces == 1
                    chunks = k // 128
                    per = (-(-chunks // (groups * pieces)) + 1) // 2 * 2
                    assert pieces == 1 or (per * (groups * pieces - 1) < chunks and (pieces - 1) * sum(rows) * b <= ws)
