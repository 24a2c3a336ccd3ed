import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line(
        "markers", "gpu: needs an MI355X (runs the HIP library)")


@pytest.fixture(params=["resident", "launched"])
def pcg_form(request):
    """The PCG of small and middle levels in one launch (the default), and with
    the t-marching launches that larger levels take."""
    import ctypes as C
    from ofblend_amd import _lib
    from ofblend_amd import manta as M
    from ofblend_amd.abi import FLOF_STENCIL_AUTO, FLOF_STENCIL_TMARCH
    L, ctx = _lib.lib(), M.context()

    def counts():
        a, b = C.c_int64(), C.c_int64()
        assert L.flof_ctx_resident_counts(ctx, C.byref(a), C.byref(b)) == 0
        return a.value, b.value

    before = counts()
    launched = request.param == "launched"
    assert L.flof_ctx_set_stencil(ctx, FLOF_STENCIL_TMARCH if launched else FLOF_STENCIL_AUTO) == 0
    try:
        yield request.param
    finally:
        assert L.flof_ctx_set_stencil(ctx, FLOF_STENCIL_AUTO) == 0
    now = counts()
    assert now[1] == before[1] and (now[0] == before[0]) == launched
