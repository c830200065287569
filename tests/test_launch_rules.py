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
