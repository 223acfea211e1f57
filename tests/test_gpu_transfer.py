"""cs_upload_state / cs_download_state through pinned staging
slots (down from 24 MiB, up from 64 MiB) and below them: every owned word comes back
as it went in, whole arrays come back the same from both sizes of call, and a
download of some of the arrays leaves the others alone."""
import ctypes
import threading

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


def test_transfers_of_two_handles_at_once():
    """Two handles on two threads (the calls release the interpreter), both
    past the thresholds of both directions: each has its own slots while its
    transfer runs, and a third handle made later takes the slots that they left.
    Every array comes back as a download of its own handle alone gives it."""
    cfg = cs.make_config(96, 33, 3, cs.RECON_WENO5, cs.RS_HLLD, cs.EMF_LLF, cs.FP64, 2)
    st = [cs.init_problem(cfg, 2, seed=q) for q in range(3)]
    for q, s in enumerate(st):
        s.interior()[0][...] *= 1.0 + 0.1 * q
    hs = [cs.CubeSphere(cfg) for _ in range(2)]
    got = [[], []]

    def work(q):
        for _ in range(4):
            hs[q].upload(st[q])
            got[q].append(hs[q].download())

    try:
        th = [threading.Thread(target=work, args=(q,)) for q in range(2)]
        for t in th:
            t.start()
        for t in th:
            t.join()
        hs.append(cs.CubeSphere(cfg))
        hs[2].upload(st[2])
        got.append([hs[2].download()])
        for q, h in enumerate(hs):
            assert len(got[q]) == (1 if q == 2 else 4)
            alone = h.download()
            assert np.array_equal(alone.interior()[0], st[q].interior()[0])
            for g in got[q]:
                for x, y in zip(g.arrays(), alone.arrays()):
                    assert np.array_equal(x, y)
    finally:
        for h in hs:
            h.close()


def test_pinned_arrays_round_trip():
    """Arrays that the caller has pinned are copied directly, pageable ones of
    the same call through the slots: the same words either way."""
    torch = pytest.importorskip("torch")
    cfg = cs.make_config(96, 33, 3, cs.RECON_WENO5, cs.RS_HLLD, cs.EMF_LLF, cs.FP64, 2)
    st = cs.init_problem(cfg, 2, seed=5)
    h = cs.CubeSphere(cfg)
    try:
        h.upload(st)
        want = h.download()
        for pinned in ((0,), (1, 2, 3, 4), (0, 1, 2, 3, 4)):
            src, dst = [], []
            for q, a in enumerate(st.arrays()):
                mk = lambda: torch.zeros(a.size, dtype=torch.float64, pin_memory=q in pinned).numpy()
                src.append(mk())
                dst.append(mk())
                src[q][:] = a.ravel()
            p = lambda arrs: [v.ctypes.data_as(ctypes.c_void_p) for v in arrs]
            assert cs.lib().cs_upload_state(h.h, *p(src)) == 0
            assert cs.lib().cs_download_state(h.h, *p(dst)) == 0
            for x, y in zip(dst, want.arrays()):
                assert np.array_equal(x, y.ravel())
    finally:
        h.close()
