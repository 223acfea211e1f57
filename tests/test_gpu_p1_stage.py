"""GPU parity of the P1 stage of a shell (recon CS_RECON_P1ADP: the
reference's LIMIT_ALL_SLOPES_P1 with its positivity limiter and the ADP
constrained least squares, face fluxes at the face centres with HLLD or HLL,
MAKE_EDGE_EFIELDS_P1, the arc-length constrained transport, CLEANUP_AFTER_UPDATE
and EVALUATE_TIMESTEP, over all six sectors in one graph per step) against the
oracle's sequence of the same routines (oracle.p1s_step_oracle), whose
pieces are bit-exact with the reference's routines built from source.

Cases named for the benchmark configurations they shrink:
  C2: 6x16^2 surface between conducting walls, HLLD, SSP-RK3, magnetised blast;
  C5: 6x8^2x3 shell r in [1, 1.5], HLLD, IMEX-SSP2(2,2,2) with the radial
      gravity implicit, hydrostatic state with density noise (radial ghost
      layers by PAD_BOUNDARY_R, outflow at both ends, and, in a second case,
      by ADD_BOUNDARY with the problem's own state);
  plus the reference's own combination (HLL, Heun RK2) on a shell, a
  6x8^2x20 shell whose columns the face kernels march in one-level chunks,
  and a blast with log-normal noise so the
  positivity limiter removes slopes and its loop-order replay runs on the
  device.

Tolerance: the device evaluates the separable form of the face geometry (a
few ulps from the oracle's per-face quadrature), lets the compiler fuse
multiply-adds and solves the constrained least squares with six unknowns
eliminated in the zone's own frame, so after two steps every conserved variable agrees with
the oracle to 1e-9 relative L1 over the owned zones (and the owned face B
to 1e-9 of its largest magnitude); the next time step to 1e-9."""
import ctypes

import numpy as np
import pytest

import cubesphere_amd as cs
from oracle import oracle as orc
from test_gpu_p1 import later_neighbours

pytestmark = pytest.mark.gpu


def _cfg(name):
    if name == "C2_surface16_hlld_rk3":
        return cs.make_config(16, 1, 4, cs.RECON_P1ADP, cs.RS_HLLD, cs.EMF_LLF, cs.FP64, 3), 2, 0.0
    if name == "C5_shell8x3_hlld_imex":
        return (cs.make_config(8, 3, 4, cs.RECON_P1ADP, cs.RS_HLLD, cs.EMF_LLF, cs.FP64, 2, cs.RBC_PAD,
                               cs.RMESH_UNIFORM, 1.0, 1.5, grav=1.0, imex=1), 3, 0.0)
    if name == "shell8x3_hll_rk2":
        return (cs.make_config(8, 3, 4, cs.RECON_P1ADP, cs.RS_HLL, cs.EMF_LLF, cs.FP64, 2, cs.RBC_PAD,
                               cs.RMESH_UNIFORM, 1.0, 1.3), 2, 0.0)
    if name == "shell8x3_problem_boundary":
        return (cs.make_config(8, 3, 4, cs.RECON_P1ADP, cs.RS_HLLD, cs.EMF_LLF, cs.FP64, 2, cs.RBC_PROBLEM,
                               cs.RMESH_UNIFORM, 1.0, 1.5, grav=1.0, imex=1, bc_problem=103), 103, 0.0)
    if name == "shell8x20_hlld_imex":
        return (cs.make_config(8, 20, 4, cs.RECON_P1ADP, cs.RS_HLLD, cs.EMF_LLF, cs.FP64, 2, cs.RBC_PAD,
                               cs.RMESH_UNIFORM, 1.0, 2.0, grav=1.0, imex=1), 3, 0.0)
    if name == "surface12_blast_noise":
        return cs.make_config(12, 1, 4, cs.RECON_P1ADP, cs.RS_HLLD, cs.EMF_LLF, cs.FP64, 3), 2, 1.5
    raise ValueError(name)


CASES = ["C2_surface16_hlld_rk3", "C5_shell8x3_hlld_imex", "shell8x3_hll_rk2", "shell8x3_problem_boundary",
         "shell8x20_hlld_imex", "surface12_blast_noise"]


def _state(cfg, prob, noise, seed=11):
    if prob >= 100:  # a problem of PROBLEM_GENERATOR_U_A on the quadrature geometry
        st = cs.init_problem(cfg, 0, seed=seed)
        st.U[:], st.ent[:], st.Bx[:], st.By[:], st.Bz[:] = orc.init_problem_p1(cfg, prob, seed=seed)
        return st
    st = cs.init_problem(cfg, prob, seed=seed)
    if noise > 0.0:
        rng = np.random.default_rng(seed)
        U = st.U.reshape(6, 8, -1)
        f = np.exp(noise * rng.normal(size=U[:, 0].shape))
        for c in range(8):
            if c in (0, 1, 2, 3):
                U[:, c] *= f
        U[:, 4] *= np.exp(noise * rng.normal(size=U[:, 4].shape))
        st.ent *= np.exp(noise * rng.normal(size=st.ent.shape))
    return st


def _owned_faces(cfg, q):
    N, NR, g = cfg.ntp, cfg.nr, cfg.nghost
    nf, nfr = N + 2 * g + 1, NR + 2 * g + 1
    m = np.zeros((nfr, nf, nf), bool)
    i0, j0, k0 = (0 if q == 0 else 1), (0 if q == 1 else 1), (0 if q == 2 else 1)
    m[k0 + g:NR + 1 + g, j0 + g:N + 1 + g, i0 + g:N + 1 + g] = True
    return m.ravel()


def _compare(cfg, got, ref, tol):
    Ug, eg = got.interior()
    Uo, eo = ref.interior()
    worst = 0.0
    for c in range(8):
        den = np.abs(Uo[:, c]).sum()
        if den > 0:
            worst = max(worst, float(np.abs(Ug[:, c] - Uo[:, c]).sum() / den))
    worst = max(worst, float(np.abs(eg - eo).sum() / max(np.abs(eo).sum(), 1e-300)))
    for q, (bg, bo) in enumerate(zip(got.arrays()[2:], ref.arrays()[2:])):
        m = np.tile(_owned_faces(cfg, q), 6)
        scale = max(np.abs(bo[m]).max(), 1e-300)
        worst = max(worst, float(np.abs(bg[m] - bo[m]).max() / scale))
    assert worst < tol, worst
    return worst


def _divb(cfg, geo, st, bscale):
    """per owned zone, the sum of the six face fluxes A B over V^(2/3) bscale,
    on the oracle's quadrature geometry"""
    N, NR, g = cfg.ntp, cfg.nr, cfg.nghost
    gd = orc.geometry_dims(cfg)
    nz, nf = N + 2 * g, N + 2 * g + 1
    Bx, By, Bz = (b.reshape(6, NR + 2 * g + 1, nf, nf) for b in st.arrays()[2:])
    xa = geo["xf"]["area"].reshape(6, NR + 2 * g, nz, nf)
    ya = geo["yf"]["area"].reshape(6, NR + 2 * g, nf, nz)
    za = geo["zf"]["area"].reshape(6, NR + 2 * g + 1, nz, nz)
    vol = geo["v_vol"].reshape(6, NR + 2 * g, nz, nz)
    out = []
    k, j, i = np.meshgrid(np.arange(1, NR + 1), np.arange(1, N + 1), np.arange(1, N + 1), indexing="ij")
    for s in range(6):
        d = (xa[s, k - 1 + g, j - 1 + g, i + g] * Bx[s, k + g, j + g, i + g] -
             xa[s, k - 1 + g, j - 1 + g, i - 1 + g] * Bx[s, k + g, j + g, i - 1 + g] +
             ya[s, k - 1 + g, j + g, i - 1 + g] * By[s, k + g, j + g, i + g] -
             ya[s, k - 1 + g, j - 1 + g, i - 1 + g] * By[s, k + g, j - 1 + g, i + g] +
             za[s, k + g, j - 1 + g, i - 1 + g] * Bz[s, k + g, j + g, i + g] -
             za[s, k - 1 + g, j - 1 + g, i - 1 + g] * Bz[s, k - 1 + g, j + g, i + g])
        scale = vol[s, k - 1 + g, j - 1 + g, i - 1 + g] ** (2.0 / 3.0) * bscale
        out.append(d / scale)
    return np.array(out)


@pytest.mark.parametrize("name", CASES)
def test_p1_stage_matches_oracle(name):
    cfg, prob, noise = _cfg(name)
    st0 = _state(cfg, prob, noise)
    G = orc.Grid(cfg)
    As = orc.p1s_patches(cfg)
    geo = orc.quad_geometry(cfg)
    ref = st0.copy()
    dt0 = 2e-3 if cfg.nr > 1 else 1e-3
    print(f"case {name}: oracle steps", flush=True)
    dts = [dt0]
    for _ in range(2):
        dts.append(orc.p1s_step_oracle(G, cfg, As, ref, dts[-1]))
    print(f"case {name}: device steps", flush=True)
    h = cs.CubeSphere(cfg)
    try:
        h.upload(st0)
        up = h.download()
        h.dt = dt0
        h.advance(1)
        dt1 = h.dt
        assert abs(dt1 - dts[1]) <= 1e-9 * dts[1], (dt1, dts[1])
        h.dt = dts[1]
        h.advance(1)
        got = h.download()
        dt2 = h.dt
    finally:
        h.close()
    w = _compare(cfg, got, ref, 1e-9)
    assert abs(dt2 - dts[2]) <= 1e-9 * dts[2], (dt2, dts[2])
    # one fixed field scale (the largest owned face B of the input): ghost
    # faces, which the exchange rewrites, do not enter
    bscale = max(np.abs(b[np.tile(_owned_faces(cfg, q), 6)]).max() for q, b in enumerate(up.arrays()[2:]))
    d0, d1 = _divb(cfg, geo, up, bscale), _divb(cfg, geo, got, bscale)
    change = float(np.abs(d1 - d0).max())
    print(f"case {name}: rel L1 {w:.2e}, div B {np.abs(d0).max():.2e}, its change over two steps {change:.2e}")
    # constrained transport: each zone's discrete divergence changes only by rounding
    assert change < 1e-12


def test_p1_stage_march_chunks():
    """A shell with enough blocks of columns that the face kernels march two
    levels per workgroup, the last chunk of one level (48^2 x 41: 192 blocks of
    15 x 7 columns, 45 levels of k_flux and 49 of k_face_pts): one step
    against the oracle.  The smaller shells of this file march one level each."""
    cfg = cs.make_config(48, 41, 4, cs.RECON_P1ADP, cs.RS_HLLD, cs.EMF_LLF, cs.FP64, 2, cs.RBC_PAD, cs.RMESH_UNIFORM,
                         1.0, 1.5)
    st0 = _state(cfg, 3, 0.0)
    ref = st0.copy()
    print("march chunks: oracle step", flush=True)
    dt1 = orc.p1s_step_oracle(orc.Grid(cfg), cfg, orc.p1s_patches(cfg), ref, 1e-3)
    print("march chunks: device step", flush=True)
    h = cs.CubeSphere(cfg)
    try:
        h.upload(st0)
        h.dt = 1e-3
        h.advance(1)
        got = h.download()
        assert abs(h.dt - dt1) <= 1e-9 * dt1
    finally:
        h.close()
    _compare(cfg, got, ref, 1e-9)


@pytest.mark.parametrize("name", ["shell8x20_hlld_imex", "C2_surface16_hlld_rk3", "shell20x9"])
def test_p1_stage_march_lengths(name):
    """The face kernels' marches at the lengths that large shells take (up to
    eight levels a workgroup in k_face_pts and four or sixteen in k_flux) with
    ragged last chunks, on small ones: two steps equal bit for bit those of
    one-level marches, which test_p1_stage_matches_oracle compares with the
    oracle."""
    if name == "shell20x9":  # several blocks of columns in both directions
        cfg, prob = cs.make_config(20, 9, 4, cs.RECON_P1ADP, cs.RS_HLLD, cs.EMF_LLF, cs.FP64, 2, cs.RBC_PAD,
                                   cs.RMESH_UNIFORM, 1.0, 1.5), 2
    else:
        cfg, prob, _ = _cfg(name)
    st0 = _state(cfg, prob, 0.0)
    want = None
    for pts, flux in ((1, 1), (2, 2), (3, 3), (5, 4), (8, 7), (16, 16)):
        h = cs.CubeSphere(cfg)
        try:
            assert cs.lib().cs_p1_set_march(h.h, pts, flux) == 0
            h.upload(st0)
            h.dt = 1e-3
            h.advance(2)
            got = h.download(), h.dt
        finally:
            h.close()
        if want is None:
            want = got
        for a, b in zip(got[0].arrays(), want[0].arrays()):
            assert np.array_equal(a, b), (pts, flux)
        assert got[1] == want[1]


def test_p1_stage_long_replay_list():
    """The positivity replay with more zones on its list than its 512
    workgroups take in groups of 64 (a lane then redoes all fields of its
    zone): one step on a shell whose noise removes the slopes of a tenth of the
    zones, against the oracle."""
    cfg = cs.make_config(24, 20, 4, cs.RECON_P1ADP, cs.RS_HLLD, cs.EMF_LLF, cs.FP64, 2, cs.RBC_PAD, cs.RMESH_UNIFORM,
                         1.0, 1.5)
    st0 = _state(cfg, 2, 1.5)
    ref = st0.copy()
    print("long replay list: oracle step", flush=True)
    As = orc.p1s_patches(cfg)
    dt1 = orc.p1s_step_oracle(orc.Grid(cfg), cfg, As, ref, 2e-5)
    print("long replay list: device step", flush=True)
    h = cs.CubeSphere(cfg)
    try:
        h.upload(st0)
        h.dt = 2e-5
        h.advance(1)
        got = h.download()
        assert abs(h.dt - dt1) <= 1e-9 * dt1
    finally:
        h.close()
    _compare(cfg, got, ref, 1e-9)
    gone = np.array([A["ent"].reshape(4, 28, 32, 32)[0] == 0.0 for A in As])  # the last stage's removed zones
    assert later_neighbours(gone) > 512 * 64


def test_p1_stage_graph_equals_eager():
    cfg, prob, noise = _cfg("surface12_blast_noise")
    st0 = _state(cfg, prob, noise)
    out = []
    for graph in (True, False):
        h = cs.CubeSphere(cfg)
        try:
            h.upload(st0)
            h.dt = 1e-3
            h.advance(3, use_graph=graph)
            out.append((h.download(), h.dt))
        finally:
            h.close()
    for a, b in zip(out[0][0].arrays(), out[1][0].arrays()):
        assert np.array_equal(a, b)
    assert out[0][1] == out[1][1]


def test_p1_stage_surface_conserves_mass():
    """Closed shell between conducting walls: mass to rounding after 5 steps."""
    cfg, prob, noise = _cfg("C2_surface16_hlld_rk3")
    st0 = _state(cfg, prob, noise)
    geo = orc.quad_geometry(cfg)
    N, NR, g = cfg.ntp, cfg.nr, cfg.nghost
    vol = geo["v_vol"].reshape(6, NR + 2 * g, N + 2 * g, N + 2 * g)[:, g:g + NR, g:g + N, g:g + N]
    h = cs.CubeSphere(cfg)
    try:
        h.upload(st0)
        h.dt = 1e-3
        h.advance(5)
        got = h.download()
    finally:
        h.close()
    m0 = (st0.interior()[0][:, 0] * vol).sum()
    m1 = (got.interior()[0][:, 0] * vol).sum()
    assert abs(m1 / m0 - 1.0) < 1e-13
