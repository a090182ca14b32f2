"""The memory a case is admitted with is that of the layout it is created with,
on both sides of the row padding's limits (400 000 points, rows of 314)."""
import ctypes as C

import pytest

import astr_amd as A
from astr_amd import serve as S

# (configuration, points, row pitch, fields): 72 x 73 x 75 points are 394 200, 74 x 73 x 75 are 405 150
CASES = [(A.tgv_config(32), 33 * 33, 48, 37), (A.tgv_config(71, 72, 74), 73 * 75, 80, 37),
         (A.tgv_config(73, 72, 74), 73 * 75, 80, 37), (A.tgv_config(128), 129 * 129, 136, 37),
         (A.tgv_config(313, 40, 40), 41 * 41, 320, 37), (A.tgv_config(320, 40, 40), 41 * 41, 336, 37),
         (A.vortex_config(64), 65, 80, 37), (A.main_config(128), 129 * 129, 136, 42)]


@pytest.mark.parametrize("cfg,rows,pitch,fields", CASES)
def test_case_bytes_of_the_layout(cfg, rows, pitch, fields):
    stride = (pitch * rows + 1 + 63) // 64 * 64
    want = fields * stride * 8
    got = A.case_field_bytes(cfg)
    # the main path's halo sources: at most ten rows of five fields per boundary line
    assert got == want if fields == 37 else want <= got <= want + 2 * 8 * 50 * 2 * (129 + 129)
    assert S.case_bytes(cfg) == got + 64 * 1024


@pytest.mark.gpu
@pytest.mark.parametrize("cfg,rows,pitch,fields", CASES)
def test_case_bytes_of_a_created_case(cfg, rows, pitch, fields):
    f, lay = A.Flow(cfg), A.Layout()
    assert A.lib().astr_hip_field_info(f.h, C.byref(lay)) == 0
    assert lay.pitch == pitch
    if fields == 37:
        assert A.case_field_bytes(cfg) == fields * lay.field_stride * 8
