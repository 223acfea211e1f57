"""cs_upload_state / cs_download_state through pinned staging
slots (down from 24 MiB, up from 64 MiB) and below them: every owned word comes back
as it went in, whole arrays come back the same from both sizes of call, and a
download of some of the arrays leaves the others alone."""
import ctypes

import numpy as np
import pytest

import cubesphere_amd as cs

pytestmark = pytest.mark.gpu


# not staged; staged down only, with ragged last chunks; both ways, more chunks than slots
@pytest.mark.parametrize("N,NR", [(16, 3), (45, 21), (96, 33)])
def test_state_round_trip(N, NR):
    cfg = cs.make_config(N, NR, 3, cs.RECON_WENO5, cs.RS_HLLD, cs.EMF_LLF, cs.FP64, 2)
    st = cs.init_problem(cfg, 2, seed=3)
    rng = np.random.default_rng(N)
    Ui, ei = st.interior()
    Ui[...] = rng.uniform(1.0, 2.0, Ui.shape)
    ei[...] = rng.uniform(1.0, 2.0, ei.shape)
    staged = sum(a.nbytes for a in st.arrays()) >= 24 << 20
    assert staged == (N > 16)
    h = cs.CubeSphere(cfg)
    try:
        h.upload(st)
        a, b = h.download(), h.download()
        Ua, ea = a.interior()
        assert np.array_equal(Ua, Ui) and np.array_equal(ea, ei)
        # faces off the panel edges are the caller's (the two copies of each
        # panel-edge face take their mean)
        g = cfg.nghost
        for got, sent in zip(a.views()[2:], st.views()[2:]):
            cut = (slice(None), slice(g + 1, g + NR), slice(g + 1, g + N), slice(g + 1, g + N))
            assert np.array_equal(got[cut], sent[cut])
        for x, y in zip(a.arrays(), b.arrays()):
            assert np.array_equal(x, y)
        # some arrays only: NULL arrays are left out
        U = np.full_like(a.U, np.nan)
        Bz = np.full_like(a.Bz, np.nan)
        p = lambda v: None if v is None else v.ctypes.data_as(ctypes.c_void_p)
        assert cs.lib().cs_download_state(h.h, p(U), None, None, None, p(Bz)) == 0
        assert np.array_equal(U, a.U) and np.array_equal(Bz, a.Bz)
    finally:
        h.close()
