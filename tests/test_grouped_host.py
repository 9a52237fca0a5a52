"""What a grouped plan refuses (checked before any device call)."""
import ctypes

import pytest


@pytest.mark.parametrize('bn', [-1, 1, 32, 63, 96, 100, 384])
def test_tile_widths_refused(bn):
    from electrolites_amd import _lib, batch
    items, plan, work = (batch.JKItem * 1)(), ctypes.c_void_p(), ctypes.c_size_t()
    with pytest.raises(Exception, match='not in'):
        _lib.call('mdf_grouped_plan_create', ctypes.cast(items, ctypes.c_void_p), 0, 1, 1, 0, bn, 0,
                  ctypes.byref(plan), ctypes.byref(work))
