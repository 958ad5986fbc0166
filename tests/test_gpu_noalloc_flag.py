"""fx_rhs_noalloc's connectivity check: the result of an invalid call does not stay for later ones,
whichever layouts of the shared scratch array lie between them."""
import ctypes as C

import numpy as np
import pytest

from fluxo_amd import native as NT
from test_zzz_no_alloc import DeviceProblem, _case, _hip

pytestmark = pytest.mark.gpu


def test_invalid_call_then_valid_calls():
    hip, L = _hip(), NT.lib()
    for kinds in (("ns_tgv", "euler_nfvse"), ("euler_nfvse", "ns_tgv")):
        for kind in kinds:
            m, U, opts = _case(kind)
            cfg = NT.make_config(int(m["N"]), int(m["nElems"]), int(m["nSides"]), **opts)
            bad = dict(m)
            s2e = np.array(m["SideToElem"], dtype=np.int32, copy=True)
            s2e.reshape(-1)[-5] = 0  # the last side's master element
            bad["SideToElem"] = s2e
            for mesh, want in ((m, 0), (bad, -1), (m, 0)):
                dp = DeviceProblem(hip, mesh, U)
                try:
                    rc = L.fx_rhs_noalloc(C.byref(cfg), C.byref(dp.mesh), dp.U, dp.Ut, None)
                    assert hip.hipDeviceSynchronize() == 0
                finally:
                    dp.free()
                assert rc == want, L.fx_last_error().decode()
