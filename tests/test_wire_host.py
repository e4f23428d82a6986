"""How a wire call is launched (bz_kv_wire_launch_shape), without a GPU: every vector has a lane, and no launch has more
work-items than 32 bits count."""
import ctypes as C

import pytest

from blitz_scale_amd import _lib
from blitz_scale_amd._lib import BZ_BF16, BZ_E4M3, BZ_ERR_UNSUPPORTED, BZ_F16

GIB = 1 << 30


def launch_shape(pages, layers, kv_heads, page_size, head_dim, dtype, wire):
    lib, kv = _lib.load(), _lib.BzPagedKV()
    kv.num_kv_heads, kv.page_size, kv.head_dim, kv.kv_dtype = kv_heads, page_size, head_dim, dtype
    lib.bz_paged_kv_set_layout(kv, _lib.BZ_LAYOUT_HND)
    per, wgs = C.c_uint32(), C.c_uint32()
    rc = lib.bz_kv_wire_launch_shape(pages, layers, C.byref(kv), wire, C.byref(per), C.byref(wgs))
    return rc, per.value, wgs.value, pages * layers * kv.stride_page // 8


@pytest.mark.parametrize("dtype,wire,gib", [(BZ_BF16, BZ_BF16, 256), (BZ_F16, BZ_E4M3, 256), (BZ_E4M3, BZ_E4M3, 128)])
@pytest.mark.parametrize("part", [0.0001, 0.2499, 0.25, 0.2501, 0.4999, 0.5, 0.5001, 0.9999])
def test_every_size_that_four_vectors_per_lane_can_cover_is_launched(dtype, wire, gib, part):
    page_bytes = 2 * 8 * 16 * 128 * (1 if dtype == BZ_E4M3 else 2)
    rc, per, wgs, vecs = launch_shape(int(gib * GIB * part) // (32 * page_bytes), 32, 8, 16, 128, dtype, wire)
    assert rc == 0 and per in (1, 2, 4)
    assert wgs * 256 < 2 ** 32 and (wgs - 1) * 256 * per < vecs <= wgs * 256 * per


@pytest.mark.parametrize("dtype,gib", [(BZ_BF16, 256), (BZ_E4M3, 128)])
def test_more_work_items_than_a_launch_has_are_refused(dtype, gib):
    page_bytes = 2 * 8 * 16 * 128 * (1 if dtype == BZ_E4M3 else 2)
    assert launch_shape(gib * GIB // (32 * page_bytes), 32, 8, 16, 128, dtype, BZ_E4M3)[0] == BZ_ERR_UNSUPPORTED
    assert launch_shape(0, 32, 8, 16, 128, dtype, BZ_E4M3)[2] == 0


def test_chunks_that_are_no_whole_number_of_workgroups_take_the_general_form():
    assert launch_shape(10, 2, 3, 4, 8, BZ_F16, BZ_F16)[1:3] == (4, 1)  # 24 vectors per chunk
    assert launch_shape(10, 2, 3, 16, 64, BZ_BF16, BZ_E4M3)[1] == 4     # 768: no multiple of 512
    assert launch_shape(10, 2, 4, 16, 64, BZ_BF16, BZ_E4M3)[1] == 2


@pytest.mark.parametrize("dtype,wire,per", [(BZ_BF16, BZ_BF16, 1), (BZ_F16, BZ_F16, 1), (BZ_F16, BZ_E4M3, 2), (BZ_E4M3, BZ_E4M3, 2)])
def test_a_lane_moves_16_bytes_of_the_narrower_side(dtype, wire, per):
    assert launch_shape(1000, 32, 8, 16, 128, dtype, wire)[:2] == (0, per)
