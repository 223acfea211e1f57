"""Surface steps on both sides of the sizes at which a face or zone gets two
lanes instead of one: 32768 x- and y-faces (2 * 6 * (N + 2) * (N + 1), between
N = 50 and 51) and 32768 zones (6 * N * N, between N = 73 and 74).

Both forms do the same arithmetic up to FMA contraction, so the CPU oracle
bounds them as it does every stage: 1e-10 relative L1 after three steps."""
import numpy as np
import pytest

import cubesphere_amd as cs
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _steps(cfg, st, dt0):
    dev = cs.CubeSphere(cfg)
    try:
        dev.upload(st)
        dev.dt = dt0
        dev.advance(3, use_graph=True)
        return dev.download()
    finally:
        dev.close()


@pytest.mark.parametrize("recon", [cs.RECON_WENO5, cs.RECON_PCM])
@pytest.mark.parametrize("n", [7, 50, 51, 73, 74])
def test_lane_pairs_match_oracle(n, recon):
    print(f"lane pairs n={n} recon={recon}", flush=True)
    cfg = cs.make_config(n, 1, 3, recon, cs.RS_HLL if n % 2 else cs.RS_HLLD, cs.EMF_LLF, cs.FP64, 3)
    st = cs.init_problem(cfg, 2, seed=9)
    G = orc.Grid(cfg)
    dt0 = G.cfl(st, 0.0)
    ref = st.copy()
    G.advance(ref, 3, dt0)
    dev = cs.CubeSphere(cfg)
    dev.upload(st)
    dev.dt = dt0
    dev.advance(3, use_graph=True)
    got = dev.download()
    dev.close()
    (Ug, eg), (Uo, eo) = got.interior(), ref.interior()
    assert np.abs(Ug - Uo).sum() < 1e-10 * np.abs(Uo).sum()
    assert np.abs(eg - eo).sum() < 1e-10 * np.abs(eo).sum()


@pytest.mark.parametrize("n", [50, 51, 73, 74])
def test_lane_pairs_in_a_rotating_frame_match_oracle(n):
    """The same sizes in a rotating frame, whose source both lanes of a zone
    would add."""
    print(f"lane pairs rotating n={n}", flush=True)
    cfg = cs.make_config(n, 1, 3, cs.RECON_WENO5, cs.RS_HLLD, cs.EMF_LLF, cs.FP64, 3, omega=(0.1, -0.2, 0.7))
    st = cs.init_problem(cfg, 1, seed=3)
    G = orc.Grid(cfg)
    dt0 = G.cfl(st, 0.0)
    ref = st.copy()
    G.advance(ref, 3, dt0)
    (Ug, eg), (Uo, eo) = _steps(cfg, st, dt0).interior(), ref.interior()
    assert np.abs(Ug - Uo).sum() < 1e-10 * np.abs(Uo).sum()
    assert np.abs(eg - eo).sum() < 1e-10 * np.abs(eo).sum()


@pytest.mark.parametrize("n", [50, 51, 73, 74])
def test_lane_pairs_mixed_close_to_fp64(n):
    """The mixed form on both sides of the lines: FP32 reconstruction and
    Riemann solves round every flux to 6e-8 of its terms, so three steps of the
    blast, whose state moves by less than its own size in them, stay within
    1e-6 relative L1 of FP64."""
    print(f"lane pairs mixed n={n}", flush=True)
    out = []
    for prec in (cs.FP64, cs.MIXED):
        cfg = cs.make_config(n, 1, 3, cs.RECON_WENO5, cs.RS_HLLD, cs.EMF_LLF, prec, 3, omega=(0.1, -0.2, 0.7))
        st = cs.init_problem(cfg, 2, seed=3)
        out.append(_steps(cfg, st, 2e-4).interior()[0])
    assert np.abs(out[1] - out[0]).sum() < 1e-6 * np.abs(out[0]).sum()
    assert not np.array_equal(out[0], out[1])
