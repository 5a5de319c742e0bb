"""Hand-written adjoint (render + spot kernel + structure factor) against the
FP64 torch reference gradients of oracle/diffsims_grad.py (GPU).

The reference is pinned to central finite differences of the NumPy oracle in
tests/test_grad_oracle.py; here the GPU's FP32 loss and gradients are compared
with it on the same seeded inputs and the same frozen structure.
Tolerances: loss within 1e-5 relative; each gradient group (orientation,
reciprocal basis, positions, B) within 5e-5 of that group's largest |component|
(FP32 pixel sums and FP32 atomics over patterns).
"""

import numpy as np
import pytest
import torch

from oracle import diffsims_grad as G
from oracle import diffsims_oracle as O
from tests import parity as P
from tests.test_grad_oracle import mono_problem

pytestmark = pytest.mark.gpu

TOL_LOSS = 1e-5
TOL_GRAD = 5e-5


def _model(pr, **kw):
    from diffsims_amd import engine
    from diffsims_amd.crystallography import PhaseArrays
    from diffsims_amd.differentiable import RefinementModel

    ph = pr.ph
    pa = PhaseArrays(tuple(ph.abc), tuple(ph.angles), list(ph.symbols), np.asarray(ph.xyz, float),
                     np.asarray(ph.occ, float), np.asarray(ph.B, float), "t")
    p = pr.p
    st = engine.SimSettings(accelerating_voltage=p.kv, max_excitation_error=p.max_excitation_error,
                            shape_factor_width=p.shape_factor_width,
                            shape_model=p.shape_model if isinstance(p.shape_model, str) else "lorentzian",
                            minima_number=p.shape_kwargs.get("minima_number", 5.0),
                            precession_angle=p.precession_angle,
                            minimum_intensity=p.minimum_intensity)
    return RefinementModel(pa, p.reciprocal_radius, st, pr.shape, pr.sigma, pr.calibration,
                           clip_threshold=pr.clip, normalize=pr.normalize,
                           in_plane_angle=pr.in_plane_angle, mirrored=pr.mirrored,
                           scattering_params=p.scattering_params, **kw)


def _params(pr, eu, device):
    from diffsims_amd.differentiable import bunge_matrices, reciprocal_basis, rt_from_matrices

    e = torch.tensor(eu, dtype=torch.float64, device=device, requires_grad=True)
    abc = torch.tensor(pr.ph.abc, dtype=torch.float64, requires_grad=True)
    ang = torch.tensor(pr.ph.angles, dtype=torch.float64, requires_grad=True)
    xyz = torch.tensor(np.asarray(pr.ph.xyz), dtype=torch.float64, requires_grad=True)
    B = torch.tensor(np.asarray(pr.ph.B), dtype=torch.float64, requires_grad=True)
    Rt = rt_from_matrices(bunge_matrices(e))
    rec = reciprocal_basis(abc, ang)
    return (e, abc, ang, xyz, B), (Rt, rec, xyz, B)


def _reference(pr, eu, weight_fn):
    """FP64 value and gradients of weight_fn(P) with the oracle's frozen structure."""
    M = O.bunge_matrix(eu)
    pats, frozen, tab = G.numpy_patterns(pr, M)
    e, abc, ang, xyz, B = (torch.tensor(np.asarray(v, dtype=np.float64), requires_grad=True)
                           for v in (eu, pr.ph.abc, pr.ph.angles, pr.ph.xyz, pr.ph.B))
    P = G.torch_patterns(pr, G.bunge(e).transpose(-1, -2), G.reciprocal_basis(abc, ang), xyz, B,
                         frozen, tab.hkl)
    L = weight_fn(P)
    L.backward()
    return float(L.detach()), [t.grad.numpy() for t in (e, abc, ang, xyz, B)], frozen, pats


def _compare_grads(got, ref, names=("euler", "abc", "angles", "xyz", "B")):
    for name, g, r in zip(names, got, ref):
        g = g.detach().cpu().numpy()
        scale = max(np.abs(r).max(), 1e-30)
        err = np.abs(g - r).max() / scale
        print(f"  {name:7s} max|ref| {scale:.3e}  rel err {err:.2e}", flush=True)
        assert err <= TOL_GRAD, (name, err)


def _check_survivors(model, args, frozen):
    Rt, rec, xyz, B = args
    b = model.spots(model.tables(rec, xyz, B), Rt.detach())
    cnt = b.count.cpu().numpy()
    idx = b.idx.cpu().numpy()
    for o, fz in enumerate(frozen):
        assert np.array_equal(np.sort(idx[o, :cnt[o]]), np.sort(fz.idx)), o


CASES = {
    "lorentzian": dict(model="lorentzian"),
    "linear": dict(model="linear"),
    "sin2c": dict(model="sin2c"),
    "atanc": dict(model="atanc"),
    "precession": dict(model="lorentzian", precession=1.0),
    "unnormalised": dict(model="lorentzian", normalize=False),
    "rotated_mirrored": dict(model="lorentzian", in_plane_angle=23.0, mirrored=True),
}


@pytest.mark.parametrize("case", list(CASES))
def test_l2_loss_gradients_match_fp64(case):
    print(f"adjoint L2 case={case}", flush=True)
    pr = mono_problem(**CASES[case])
    n = 6
    eu = O.random_euler(n, 21)
    target = np.random.default_rng(2).uniform(0, 0.3, (n,) + pr.shape)
    L_ref, g_ref, frozen, _ = _reference(
        pr, eu, lambda P: ((P - torch.as_tensor(target)) ** 2).sum())
    model = _model(pr)
    leaves, args = _params(pr, eu, "cuda")
    _check_survivors(model, args, frozen)
    L = model.l2_loss(*args, torch.tensor(target, dtype=torch.float32, device="cuda"))
    L.backward()
    assert abs(float(L.detach()) - L_ref) <= TOL_LOSS * abs(L_ref), (float(L.detach()), L_ref)
    _compare_grads([t.grad for t in leaves], g_ref)


def test_pattern_gradients_match_fp64():
    print("adjoint pattern-grad case", flush=True)
    pr = mono_problem(model="lorentzian")
    n = 5
    eu = O.random_euler(n, 33)
    Wt = np.random.default_rng(4).normal(size=(n,) + pr.shape)
    L_ref, g_ref, frozen, pats = _reference(pr, eu, lambda P: (P * torch.as_tensor(Wt)).sum())
    model = _model(pr)
    leaves, args = _params(pr, eu, "cuda")
    P = model.patterns(*args)
    assert np.abs(P.detach().cpu().numpy() - pats).max() <= 1e-5 * pats.max()
    L = (P * torch.tensor(Wt, dtype=torch.float32, device="cuda")).sum()
    L.backward()
    # per-pixel pattern error <= 1e-5 (pattern maximum 1)
    assert abs(float(L.detach()) - L_ref) <= 1e-5 * np.abs(Wt).sum()
    _compare_grads([t.grad for t in leaves], g_ref)


def test_loss_without_grad_and_fused_pattern_output():
    print("adjoint no-grad case", flush=True)
    pr = mono_problem()
    n = 4
    eu = O.random_euler(n, 8)
    target = torch.rand((n,) + pr.shape, device="cuda", generator=torch.Generator("cuda").manual_seed(3))
    model = _model(pr)
    _, args = _params(pr, eu, "cuda")
    L1 = model.l2_loss(*args, target)
    with torch.no_grad():
        L0 = model.l2_loss(*args, target)
        P = model.patterns(*args)
    assert torch.allclose(L0, L1.detach(), rtol=1e-6)
    assert abs(float(L0) - float(((P - target).double() ** 2).sum())) <= 1e-5 * float(L0)


def test_empty_frame_gives_zero_gradients():
    """Every spot off the detector: P = 0, loss = sum T^2, no gradient."""
    print("adjoint empty-frame case", flush=True)
    pr = mono_problem()
    pr.calibration = 1e-4          # frame spans 0.006 1/A: no reflection lands in it
    n = 3
    eu = O.random_euler(n, 9)
    model = _model(pr)
    leaves, args = _params(pr, eu, "cuda")
    target = torch.full((n,) + pr.shape, 0.25, device="cuda")
    L = model.l2_loss(*args, target)
    L.backward()
    Lv = float(L.detach())
    assert abs(Lv - 0.0625 * n * pr.shape[0] * pr.shape[1]) < 1e-6 * Lv
    for t in leaves:
        assert float(t.grad.abs().max()) == 0.0


def test_refinement_workload_gradients_match_fp64():
    """The 24-atom monoclinic refinement case (16 of its 4,096 patterns, full
    256x256 detector) against the FP64 reference."""
    from diffsims_amd import differentiable as D
    from diffsims_amd import workloads

    print("adjoint refinement-workload case", flush=True)
    rw = workloads.refinement_monoclinic(16)
    ph = rw.phase
    pr = G.Problem(O.PhaseSpec(ph.abc, ph.angles, ph.symbols, ph.xyz, ph.occ, ph.B),
                   O.SimParams(kv=200, reciprocal_radius=rw.reciprocal_radius,
                               max_excitation_error=0.02, shape_model="lorentzian",
                               with_direct_beam=False),
                   rw.shape, rw.sigma, rw.calibration, clip=1.0)
    model = D.RefinementModel(ph, rw.reciprocal_radius, rw.settings, rw.shape, rw.sigma,
                              rw.calibration, clip_threshold=1.0)
    with torch.no_grad():
        T = model.patterns(*D.forward_args(D.leaf_parameters(rw.truth_phase, rw.truth_euler,
                                                             requires_grad=False)))
    target = T.cpu().numpy().astype(np.float64)
    L_ref, g_ref, frozen, _ = _reference(pr, rw.euler,
                                         lambda P: ((P - torch.as_tensor(target)) ** 2).sum())
    leaves = D.leaf_parameters(ph, rw.euler)
    _check_survivors(model, D.forward_args(leaves), frozen)
    L = model.l2_loss(*D.forward_args(leaves), T)
    L.backward()
    assert abs(float(L.detach()) - L_ref) <= TOL_LOSS * abs(L_ref), (float(L.detach()), L_ref)
    _compare_grads([leaves[k].grad for k in ("euler", "abc", "angles", "xyz", "B")], g_ref)


def _big_problem(**kw):
    """A 19-21 A triclinic cell: ~2,000 spots per pattern, all in a 128x128
    frame, so the render and its adjoint take the chunked large-pattern path."""
    rng = np.random.default_rng(17)
    n_atoms = 4
    ph = O.PhaseSpec((19.5, 20.5, 21.0), (88.0, 96.0, 91.0),
                     list(rng.choice(["O", "Si", "Fe"], n_atoms)), rng.uniform(0, 1, (n_atoms, 3)),
                     np.ones(n_atoms), rng.uniform(0.3, 1.0, n_atoms))
    p = O.SimParams(kv=200, reciprocal_radius=1.2, max_excitation_error=0.03,
                    shape_model=kw.pop("model", "lorentzian"), with_direct_beam=False,
                    minimum_intensity=1e-20)
    return G.Problem(ph, p, (128, 128), 1.2, 0.02, clip=1e-3, **kw)


def test_large_pattern_subpixel_render_and_gradients():
    print("adjoint large-pattern case", flush=True)
    pr = _big_problem()
    n = 3
    eu = O.random_euler(n, 41)
    target = np.random.default_rng(6).uniform(0, 0.3, (n,) + pr.shape)
    L_ref, g_ref, frozen, pats = _reference(
        pr, eu, lambda P: ((P - torch.as_tensor(target)) ** 2).sum())
    assert min(len(f.idx) for f in frozen) > 1500
    model = _model(pr)
    leaves, args = _params(pr, eu, "cuda")
    _check_survivors(model, args, frozen)
    with torch.no_grad():
        P = model.patterns(*args)                     # forward mode of the chunked kernel
    assert np.abs(P.cpu().numpy() - pats).max() <= 1e-5 * pats.max()
    L = model.l2_loss(*args, torch.tensor(target, dtype=torch.float32, device="cuda"))
    L.backward()
    assert abs(float(L.detach()) - L_ref) <= TOL_LOSS * abs(L_ref), (float(L.detach()), L_ref)
    _compare_grads([t.grad for t in leaves], g_ref)


def test_forward_mode_equals_subpixel_renderer():
    """dsx_render_adjoint's forward mode and dsx_render_subpixel (each with
    its own fixed-point scale) agree to 1e-6 of the pattern maximum on
    patterns both can hold."""
    import ctypes

    from diffsims_amd import _lib, engine

    pr = mono_problem()
    eu = O.random_euler(7, 12)
    model = _model(pr)
    _, args = _params(pr, eu, "cuda")
    t = model.tables(*args[1:])
    b = model.spots(t, args[0].detach())
    ref = engine.render_spots(b.spots, b.count, b.cap, pr.shape, pr.sigma, pr.calibration,
                              fast=False, clip_threshold=pr.clip)
    out = torch.empty_like(ref)
    L = _lib.load()
    sim = model._sim_params(t)
    status = torch.zeros(b.n, dtype=torch.int32, device="cuda")
    _lib.check(L.dsx_render_adjoint(
        None, _lib.ptr(b.spots), _lib.ptr(b.count), b.cap, b.n, None, None, 0, None,
        ctypes.byref(sim), ctypes.byref(model.render), _lib.ADJ_FORWARD, None, 0, _lib.ptr(out),
        None, None, None, None, None, 0, _lib.ptr(status), _lib.stream_handle()), "forward")
    torch.cuda.synchronize()
    assert int(status.max()) == 0
    assert float((out - ref).abs().max()) <= 1e-6 * float(ref.abs().max())


def test_broadcast_target():
    """One target shared by every orientation (stride 0) equals the repeated target."""
    pr = mono_problem()
    n = 5
    eu = O.random_euler(n, 13)
    model = _model(pr)
    T1 = torch.rand(pr.shape, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    res = []
    for T in (T1, T1.expand((n,) + pr.shape).contiguous()):
        leaves, args = _params(pr, eu, "cuda")
        L = model.l2_loss(*args, T)
        L.backward()
        res.append((float(L.detach()), [x.grad.detach().cpu().numpy() for x in leaves]))
    assert abs(res[0][0] - res[1][0]) <= 1e-6 * res[1][0]
    for a, b in zip(res[0][1], res[1][1]):
        assert np.abs(a - b).max() <= 1e-5 * max(np.abs(b).max(), 1e-30)


def _precession_problem(rr, shape, cal):
    from diffsims_amd import workloads

    d = workloads.large_precession(4)
    pa = d["phase"]
    ph = O.PhaseSpec(pa.abc, pa.angles, pa.symbols, pa.xyz, pa.occ, pa.B)
    p = O.SimParams(kv=200, reciprocal_radius=rr, max_excitation_error=0.02,
                    shape_model="lorentzian", precession_angle=1.0, with_direct_beam=False,
                    minimum_intensity=1e-20)
    return d, G.Problem(ph, p, shape, 1.0, cal, clip=1.0)


def test_large_precession_cell_gradients_reduced_radius():
    """The 500-atom triclinic precession cell at reciprocal radius 1.0
    (~3,000 spots per 256x256 pattern): fused loss and gradients against FP64."""
    print("adjoint 500-atom precession cell, r = 1.0", flush=True)
    d, pr = _precession_problem(1.0, (256, 256), 0.008)
    eu = d["euler"][:2]
    target = np.random.default_rng(8).uniform(0, 0.2, pr.shape)
    L_ref, g_ref, frozen, pats = _reference(
        pr, eu, lambda P: ((P - torch.as_tensor(target)[None]) ** 2).sum())
    print("  spots per pattern:", [len(f.idx) for f in frozen], flush=True)
    assert min(len(f.idx) for f in frozen) > 1024
    model = _model(pr)
    leaves, args = _params(pr, eu, "cuda")
    _check_survivors(model, args, frozen)
    L = model.l2_loss(*args, torch.tensor(target, dtype=torch.float32, device="cuda"))
    L.backward()
    assert abs(float(L.detach()) - L_ref) <= TOL_LOSS * abs(L_ref), (float(L.detach()), L_ref)
    _compare_grads([t.grad for t in leaves], g_ref)


def test_large_precession_cell_full_radius_forward():
    """The full 500-atom precession case (r = 3.0, ~1.6e6 reflections, ~4e4
    spots per 512x512 pattern): spot lists and sub-pixel patterns of two
    orientations against the FP64 oracle (F evaluated for the intersecting rows)."""
    print("500-atom precession cell, r = 3.0 forward", flush=True)
    from diffsims_amd import engine

    d, pr = _precession_problem(3.0, (512, 512), 0.012)
    p = pr.p
    M = O.bunge_matrix(d["euler"][:2])
    tab = engine.build_phase_table(d["phase"], 3.0, False, "lobato")
    base, rec = pr.ph.basis()
    hkl = tab.hkl_host()
    g = O.g_cartesian(hkl, rec)
    k = 1 / O.electron_wavelength(200)
    otab0 = O.PhaseTables(hkl, g, np.linalg.norm(g, axis=1), np.zeros(len(hkl)), len(hkl))
    rows = set()
    for o in range(2):
        rows |= set(np.nonzero(O.intersect(g @ M[o], k, p)[2])[0].tolist())
        # and the rows at the band edge, which the GPU may keep instead
        rows |= set(np.nonzero(P.cut_distance(otab0, M[o], k, p) < 1e-5)[0].tolist())
    rows = np.array(sorted(rows))
    F2 = np.full(len(hkl), np.nan)
    coeffs, _ = O.atom_coeffs(pr.ph.symbols, "lobato")
    F = O.structure_factor(hkl[rows], np.linalg.norm(g[rows], axis=1), pr.ph.xyz, pr.ph.occ,
                           pr.ph.B, coeffs, "lobato", "exact")
    F2[rows] = (F * F.conjugate()).real
    otab = O.PhaseTables(hkl, g, np.linalg.norm(g, axis=1), F2, len(hkl))
    print(f"  {len(hkl)} reflections, {len(rows)} intersecting rows", flush=True)
    b = engine.simulate(tab, engine.rotation_matrices_to_device(M), d["settings"], 3.0)
    pats = engine.render(b, pr.shape, 1.0, pr.calibration, fast=False, clip_threshold=1.0)
    cnt = b.count.cpu().numpy()
    pats = pats.cpu().numpy()
    stats = {}
    sp = b.spots.cpu().numpy()
    for o in range(2):
        gi = b.idx[o, :cnt[o]].cpu().numpy()
        print(f"  orientation {o}: {cnt[o]} spots", flush=True)
        assert cnt[o] > 20000
        # rows that differ must lie within 1e-6 of the precession band's edge;
        # the pattern is then compared on the GPU's survivor set
        ref, carved = P.check_orientation(otab, M[o], k, p, gi, sp[o, :cnt[o], 3], stats)
        assert carved <= 4, carved
        raw = O.render_subpixel(ref.xyz[:, :2], ref.intensity, pr.shape, 1.0, pr.calibration,
                                normalize=False, clip_threshold=1.0)
        rp = raw / raw.max()
        # a clip box whose edge moves by a pixel under FP32 coordinates changes
        # pixels worth at most clip_threshold
        edge = 1.0 / raw.max()
        err = np.abs(pats[o] - rp).max()
        assert err <= P.TOL_P + edge, err


def test_large_precession_cell_full_radius_gradients():
    """The benchmarked 500-atom precession shape itself: r = 3.0 (~1.6e6
    reflections), 512x512 sub-pixel patterns of ~4e4 spots, one target shared
    by every orientation (stride 0).  The GPU's fused loss and its gradients
    (orientation, lattice, positions, B) against the FP64 torch reference,
    which is evaluated on the survivor rows of the orientation only (F of
    ~4e4 rows instead of the whole table; the frozen structure is the same)."""
    print("adjoint 500-atom precession cell, r = 3.0, 512x512", flush=True)
    d, pr = _precession_problem(3.0, (512, 512), 0.012)
    p = pr.p
    eu = d["euler"][3:4]
    M = O.bunge_matrix(eu)
    model = _model(pr)
    leaves, args = _params(pr, eu, "cuda")
    Rt, rec_t, xyz_t, B_t = args
    b = model.spots(model.tables(rec_t, xyz_t, B_t), Rt.detach())
    c = int(b.count[0])
    gi = b.idx[0, :c].cpu().numpy()
    gI = b.spots[0, :c, 3].cpu().numpy()
    print(f"  {model.n_refl} reflections, {c} spots", flush=True)
    assert c > 20000
    # FP64 |F|^2 of the rows that intersect, or lie at the band edge
    hkl = model.hkl_np.astype(np.int64)
    base, rec = pr.ph.basis()
    g = O.g_cartesian(hkl, rec)
    k = 1 / O.electron_wavelength(200)
    otab0 = O.PhaseTables(hkl, g, np.linalg.norm(g, axis=1), np.zeros(len(hkl)), len(hkl))
    rows = np.union1d(np.nonzero(O.intersect(g @ M[0], k, p)[2])[0],
                      np.nonzero(P.cut_distance(otab0, M[0], k, p) < 1e-5)[0])
    coeffs, _ = O.atom_coeffs(pr.ph.symbols, "lobato")
    F = O.structure_factor(hkl[rows], np.linalg.norm(g[rows], axis=1), pr.ph.xyz, pr.ph.occ,
                           pr.ph.B, coeffs, "lobato", "exact")
    F2 = np.full(len(hkl), np.nan)
    F2[rows] = (F * F.conjugate()).real
    otab = O.PhaseTables(hkl, g, otab0.gnorm, F2, len(hkl))
    ref, carved = P.check_orientation(otab, M[0], k, p, gi, gI)
    assert carved <= 4, carved
    # frozen structure on the survivor rows, then the FP64 torch reference
    _, fz = G.freeze(pr, ref, rows=np.arange(c))
    target = np.random.default_rng(9).uniform(0, 0.2, pr.shape)
    e, abc, ang, xyz, B = (torch.tensor(np.asarray(v, dtype=np.float64), requires_grad=True)
                           for v in (eu, pr.ph.abc, pr.ph.angles, pr.ph.xyz, pr.ph.B))
    Pr = G.torch_patterns(pr, G.bunge(e).transpose(-1, -2), G.reciprocal_basis(abc, ang), xyz, B,
                          [fz], hkl[gi])
    L64 = ((Pr - torch.as_tensor(target)[None]) ** 2).sum()
    L64.backward()
    g_ref = [t.grad.numpy() for t in (e, abc, ang, xyz, B)]
    L = model.l2_loss(*args, torch.tensor(target, dtype=torch.float32, device="cuda"))
    L.backward()
    print(f"  loss {float(L.detach()):.6e} vs FP64 {float(L64.detach()):.6e}", flush=True)
    assert abs(float(L.detach()) - float(L64.detach())) <= TOL_LOSS * abs(float(L64.detach()))
    _compare_grads([t.grad for t in leaves], g_ref)


def test_euler_to_rt_kernel_and_backward():
    """The one-kernel Euler -> Rt map and its hand-written backward against the
    generic torch autograd of bunge_matrices (float64)."""
    from diffsims_amd import differentiable as D

    eu = torch.tensor(O.random_euler(257, 5), dtype=torch.float64, device="cuda")
    e1 = eu.clone().requires_grad_(True)
    e2 = eu.clone().requires_grad_(True)
    r1 = D.euler_to_rt(e1)
    r2 = D.rt_from_matrices(D.bunge_matrices(e2))
    assert float((r1 - r2).detach().abs().max()) <= 1e-14
    assert np.allclose(r1.detach().cpu().numpy().reshape(-1, 3, 3).transpose(0, 2, 1),
                       O.bunge_matrix(eu.cpu().numpy()), atol=1e-14)
    w = torch.randn(257, 9, dtype=torch.float64, device="cuda")
    (r1 * w).sum().backward()
    (r2 * w).sum().backward()
    assert float((e1.grad - e2.grad).abs().max()) <= 1e-12


def test_stage_atoms_matches_host_fixed_point():
    """dsx_stage_atoms (device positions -> uint32 turns, element order, float
    B) equals the host staging the forward tables use, bit for bit, including
    negative, integral and half-unit positions."""
    from diffsims_amd import _lib, engine

    rng = np.random.default_rng(5)
    n = 300
    xyz = rng.uniform(-3.0, 3.0, (n, 3))
    xyz[:10] = np.round(xyz[:10])                       # integral: 0 turns
    xyz[10:20, 0] = (np.arange(10) + 0.5) / 2.0 ** 32   # ties round half to even
    xyz[20, :] = [1.0 - 2.0 ** -40, -2.0 ** -40, 0.25]  # round up to 2^32 -> 0
    B = rng.uniform(0.1, 2.0, n)
    order = rng.permutation(n).astype(np.int64)
    dev = "cuda"
    fx = torch.empty((n, 4), dtype=torch.int32, device=dev)
    Bs = torch.empty(n, dtype=torch.float32, device=dev)
    L = _lib.load()
    t_xyz = torch.tensor(xyz, device=dev)
    t_B = torch.tensor(B, device=dev)
    t_order = torch.tensor(order, device=dev)
    _lib.check(L.dsx_stage_atoms(_lib.ptr(t_xyz), _lib.ptr(t_B), _lib.ptr(t_order), n,
                                 _lib.ptr(fx), _lib.ptr(Bs), _lib.stream_handle()), "stage")
    got = fx.cpu().numpy().view(np.uint32)
    want = engine._fixed_point(xyz[order])
    assert np.array_equal(got[:, :3], want)
    assert np.all(got[:, 3] == 0)
    assert np.array_equal(Bs.cpu().numpy(), B[order].astype(np.float32))


# -- long lists (matrix-core tiles) against the small-list kernels -----------------


def _copy_lists(b, cap):
    """The same spot lists with another capacity."""
    import torch
    from diffsims_amd import engine
    assert int(b.ncand.max()) <= b.cap
    out = engine.empty_batch(b.table, b.n, cap, b.idx.device)
    m = min(cap, b.cap)
    out.idx[:, :m], out.spots[:, :m] = b.idx[:, :m], b.spots[:, :m]
    for k in ("count", "ncand", "maxI"):
        setattr(out, k, getattr(b, k).clone())
    return out


@pytest.mark.parametrize("shape,sigma,clip,kw", [
    ((256, 256), 1.0, 1.0, {}),
    ((97, 131), 1.6, 1.0, {}),                    # partial tiles, odd rows
    ((64, 80), 6.0, 1e-3, {}),                    # boxes over many tiles: several ranges
    ((33, 400), 1.0, 1.0, {"in_plane_angle": 20.0, "mirrored": True}),
    ((128, 128), 0.6, 1.0, {"normalize": False}),
    ((16, 16), 1.0, 1.0, {}),                     # one tile
    ((1200, 1100), 1.0, 1.0, {}),                 # more tiles than eight waves' counters hold
])
def test_long_list_kernel_equals_small_list_kernel(shape, sigma, clip, kw):
    """One set of spot lists through both kernels (a capacity above 1,024
    selects the tiles): patterns, loss and every gradient.  Each side rounds a
    pixel's terms within ~1e-6 of the maximum; a gathered sum runs over at most
    some 2,000 pixels with both signs, so the gradients agree to 1e-4 of the
    largest component."""
    import torch
    from diffsims_amd import _lib, engine
    from diffsims_amd import differentiable as D
    from tests import parity as P

    print(f"tiles: {shape}, sigma {sigma}, clip {clip}, {kw}", flush=True)
    spec = P.triclinic(20, 9, edges=(7, 12))
    st = engine.SimSettings(max_excitation_error=0.02)
    cal = 3.2 / min(shape)
    m = D.RefinementModel(P.to_arrays(spec), 1.6, st, shape, sigma, cal, clip_threshold=clip, **kw)
    rng = np.random.default_rng(5)
    leaves = D.leaf_parameters(P.to_arrays(spec), rng.uniform(0, 2 * np.pi, (7, 3)), requires_grad=False)
    with torch.no_grad():
        Rt, rec, xyz, B = D.forward_args(leaves)
        t = m.tables(rec, xyz, B)
        b = m.spots(t, Rt)
    small, long_ = _copy_lists(b, 1000), _copy_lists(b, 1100)
    small.count[5], long_.count[5] = 0, 0          # an empty list
    H, W = shape
    gen = torch.Generator("cuda").manual_seed(2)
    for mode, target in ((_lib.ADJ_L2, torch.rand((7, H, W), generator=gen, device="cuda") * 0.2),
                         (_lib.ADJ_L2, torch.rand((H, W), generator=gen, device="cuda") * 0.2),
                         (_lib.ADJ_PATTERN_GRAD, torch.randn((7, H, W), generator=gen, device="cuda"))):
        got = []
        for batch in (small, long_):
            pat = torch.full((7, H, W), float("nan"), device="cuda")
            got.append((m.adjoint(t, Rt, batch, mode, target, True, pattern=pat), pat))
        (a, pa), (c, pc) = got
        top = float(pa.abs().max())
        assert not torch.isnan(pc).any() and float((pa - pc).abs().max()) <= 2e-6 * top
        if mode == _lib.ADJ_L2:
            assert torch.allclose(a[0], c[0], rtol=1e-5)
        for x, y in zip(a[1:], c[1:]):
            assert float((x - y).abs().max()) <= 1e-4 * float(x.abs().max()) + 1e-12
    fwd = engine.render_spots(long_.spots, long_.count, long_.cap, shape, sigma, cal, **m.render_kw)
    assert torch.equal(fwd, pc)


@pytest.mark.parametrize("shape,sigma", [((256, 256), 1.0), ((97, 131), 4.0)])
def test_long_list_patterns_and_losses_are_the_same_bits_in_every_run(shape, sigma):
    """Entries are numbered in list order whatever the waves' timing, in one range
    of tiles and in several; gradients may differ in their last bits."""
    import torch
    from diffsims_amd import _lib
    from diffsims_amd import differentiable as D
    from tests import parity as P

    print(f"tiles: repeated runs, {shape}, sigma {sigma}", flush=True)
    spec = P.triclinic(20, 9, edges=(7, 12))
    from diffsims_amd import engine
    m = D.RefinementModel(P.to_arrays(spec), 1.6, engine.SimSettings(max_excitation_error=0.02), shape, sigma,
                          3.2 / min(shape), clip_threshold=1e-2)
    rng = np.random.default_rng(6)
    leaves = D.leaf_parameters(P.to_arrays(spec), rng.uniform(0, 2 * np.pi, (600, 3)), requires_grad=False)
    with torch.no_grad():
        Rt, rec, xyz, B = D.forward_args(leaves)
        t = m.tables(rec, xyz, B)
        b = _copy_lists(m.spots(t, Rt), 1100)
    target = torch.rand(shape, generator=torch.Generator("cuda").manual_seed(2), device="cuda") * 0.2
    runs = []
    for _ in range(5):
        pat = torch.full((600, *shape), float("nan"), device="cuda")
        runs.append((m.adjoint(t, Rt, b, _lib.ADJ_L2, target, True, pattern=pat)[0], pat))
    for loss, pat in runs[1:]:
        assert torch.equal(pat, runs[0][1]) and torch.equal(loss, runs[0][0])


def test_long_lists_without_workspace_report_their_patterns():
    import ctypes
    import torch
    from diffsims_amd import _lib, engine
    L = _lib.load(require_gpu=True)
    p = engine.render_params((40, 40), 1.0, 1.0, fast=False)
    sim = _lib.SimParams()
    sim.k, sim.shape_width, sim.shape_model = 1.0, 1.0, _lib.SF_LINEAR
    spots = torch.full((3, 2000, 4), 5.0, device="cuda")
    cnt = torch.full((3,), 1500, dtype=torch.int32, device="cuda")
    out = torch.full((3, 40, 40), float("nan"), device="cuda")
    st = torch.zeros(3, dtype=torch.int32, device="cuda")
    _lib.check(L.dsx_render_adjoint(None, _lib.ptr(spots), _lib.ptr(cnt), 2000, 3, None, None, 0, None,
                                    ctypes.byref(sim), ctypes.byref(p), _lib.ADJ_FORWARD, None, 0,
                                    _lib.ptr(out), None, None, None, None, None, 0, _lib.ptr(st),
                                    _lib.stream_handle()), "dsx_render_adjoint")
    assert bool((st == 1).all()) and bool((out == 0).all())


@pytest.mark.parametrize("n", [60, 64, 65, 130, 20000])
def test_pixels_of_many_boxes_in_one_place_keep_fp32_precision(n):
    """n equal boxes: every pixel within the error of its terms and of the sum of
    64 of them.  A term has two exponentials (2^-23 each), five roundings of
    2^-24 and arguments of at most log2(7) that are off by three; 64 terms are 33
    additions; the sum over the sixty-fours is FP64."""
    import torch
    from diffsims_amd import engine

    print(f"tiles: {n} boxes in one place", flush=True)
    cap, H, W, sigma, X, Y = 20480, 64, 72, 6.0, 32.3, 31.7   # box edges are 0.1 and more off a pixel
    pref = 1.0 / (2.0 * np.pi * sigma ** 2)
    spots = torch.zeros((1, cap, 4), device="cuda")
    spots[0, :n] = torch.tensor([X - (W - 1) / 2, Y - (H - 1) / 2, 0.0, 7.0 / pref], device="cuda")
    count = torch.tensor([n], dtype=torch.int32, device="cuda")
    got = engine.render_spots(spots, count, cap, (H, W), sigma, 1.0, fast=False, normalize=False)[0]
    s = spots[0, 0].double().cpu().numpy()
    x, y = s[0] + (W - 1) / 2, s[1] + (H - 1) / 2
    d2 = (np.arange(W) - x) ** 2, (np.arange(H) - y) ** 2
    rad2 = 2 * sigma ** 2 * np.log(s[3] * pref)
    k = [np.where(d <= rad2, np.exp(-d / (2 * sigma ** 2)), 0.0) for d in d2]
    ref = n * s[3] * pref * np.outer(k[1], k[0])
    assert (ref > 0).sum() == 24 * 24
    # and the pixel position itself is one FP32 addition: 2^-19 at 32
    tol = 2 * 2.0 ** -23 + (5 + 33) * 2.0 ** -24 + 3 * 2.0 ** -24 * np.log(7.0)
    shift = 2.0 ** -19 / sigma ** 2 * 12 * 2
    assert (np.abs(got.cpu().numpy() - ref) <= (tol + shift) * ref).all()


def test_more_tile_entries_than_are_numbered_are_refused():
    """131,100 boxes over all 16,384 tiles of a 256 x 16,384 pattern are more than
    2^31 - 1 entries: the pattern is reported and left as zeros, its neighbour in
    the batch is not touched by it."""
    import torch
    from diffsims_amd import engine

    cap, sigma, shape = 131100, 1800.0, (256, 16384)
    print("tiles: 2^31 entries", flush=True)
    spots = torch.zeros((2, cap, 4), device="cuda")
    spots[0, :, 3] = 1e13          # radius 9,200 pixels from the centre
    spots[1, :100, 3] = 1e9        # radius 5,000
    spots[1, :100, 0] = torch.arange(100.0, device="cuda") * 8 - 400
    count = torch.tensor([cap, 100], dtype=torch.int32, device="cuda")
    status = torch.full((2,), -1, dtype=torch.int32, device="cuda")
    out = torch.full((2, *shape), float("nan"), device="cuda")
    engine.render_spots(spots, count, cap, shape, sigma, 1.0, fast=False, out=out, status=status)
    assert status.tolist() == [1, 0]
    assert not out[0].any() and float(out[1].max()) == 1.0
    alone = engine.render_spots(spots[1:, :2000].contiguous(), count[1:], 2000, shape, sigma, 1.0,
                                fast=False)
    assert torch.equal(alone[0], out[1])


# rows, atoms, elements, table: either side of the lines between the kernels with
# a thread per reflection and a lane per atom (24 to 160 atoms by the rows, 512/513
# atoms, 20/21 elements), and row counts around a wave's 16
SF_SIZES = [(1, 24, 3, "lobato"), (15, 23, 3, "lobato"), (17, 48, 20, "xtables"), (64, 64, 1, None),
            (65, 65, 2, "lobato"), (999, 47, 20, "lobato"), (1000, 100, 21, "xtables"),
            (1003, 512, 20, "lobato"), (700, 513, 5, "lobato"), (24577, 24, 2, "lobato"),
            (24576, 30, 2, None), (65537, 33, 1, "lobato"), (65536, 32, 1, "lobato"), (33000, 130, 4, "xtables"),
            (65537, 31, 2, "lobato"), (70001, 75, 2, "lobato"), (70001, 76, 2, "lobato"),
            (4096, 40, 4, "lobato"), (4097, 64, 20, "lobato"), (8192, 200, 18, None), (8193, 24, 2, "lobato"),
            (131073, 95, 3, "xtables"), (131073, 96, 3, "xtables"), (262145, 159, 2, "lobato"),
            (262145, 160, 2, "lobato"), (262145, 79, 2, "lobato"), (262145, 80, 2, "lobato")]


@pytest.mark.parametrize("n,n_atoms,n_elem,table", SF_SIZES)
def test_structure_factor_and_adjoint_of_any_table(n, n_atoms, n_elem, table):
    """F, |F|^2 and the gradients of sum w |F|^2 against FP64 on the same
    fixed-point positions, for tables of whole lines, broken lines and rows in
    any order.  Per atom the phase and the Debye-Waller factor are FP32: an
    angle off by 2^-26 turns (9.4e-8) and the errors of sincospif, expf and two
    products, together below 5e-7 of |t_a|, t_a the atom's term.  With S = sum
    |t_a|: |dF| <= 5e-7 S, |d|F|^2| <= 1e-6 S |F| + (5e-7 S)^2 + rounding, and each
    gradient within 2e-6 of its sum of magnitudes (conj(F) t_a is off by 1e-6
    S |t_a|, and the FP32 sums over the blocks as much again)."""
    import ctypes

    from diffsims_amd import _lib

    print(f"structure factors {n} rows {n_atoms} atoms {n_elem} elements {table}", flush=True)
    rng = np.random.default_rng(n + n_atoms)
    # lines of 1 to 40 rows, then some rows moved
    hkl, left = [], n
    while left:
        m = min(left, int(rng.integers(1, 41)))
        h, k, l0 = (int(v) for v in rng.integers(-12, 13, 3))
        hkl += [(h, k, l0 - i, 0) for i in range(m)]
        left -= m
    hkl = np.array(hkl, dtype=np.int32)
    moved = rng.choice(n, n // 8, replace=False)
    hkl[np.sort(moved)] = hkl[moved]
    rec = np.array([[0.05, 0.003, 0.001], [0.0, 0.04, -0.002], [0.0, 0.0, 0.03]])
    fx = rng.integers(0, 2 ** 32, (n_atoms, 4), dtype=np.uint64).astype(np.uint32)
    fx[:2, :3] = [[0, 0, 0], [2 ** 31, 2 ** 30, 3 * 2 ** 30]][:min(2, n_atoms)]
    elem = rng.integers(0, n_elem, n_atoms).astype(np.int32)
    occ = rng.uniform(0.2, 1.0, n_atoms).astype(np.float32)
    B = rng.uniform(0.0, 2.0, n_atoms).astype(np.float32)
    co = np.stack([rng.uniform(0.2, 2.0, (n_elem, 5)), rng.uniform(0.5, 8.0, (n_elem, 5))], -1)
    w = rng.uniform(-1.0, 1.0, n).astype(np.float32)
    w[rng.random(n) < 0.3] = 0.0

    L = _lib.load()
    dev = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()
    d_hkl, d_fx, d_el, d_occ, d_B, d_co, d_w = (dev(v) for v in (
        hkl, fx.view(np.int32), elem, occ, B, co.reshape(n_elem, 10), w))
    F, F2 = torch.empty((n, 2), device="cuda"), torch.empty(n, device="cuda")
    g4 = torch.empty((n, 4), device="cuda")
    dx, dB = torch.zeros((n_atoms, 3), device="cuda"), torch.zeros(n_atoms, device="cuda")
    dr = torch.zeros(9, dtype=torch.float64, device="cuda")
    rec9 = (ctypes.c_double * 9)(*rec.reshape(-1).tolist())
    sc = {None: _lib.SCATTER_NONE, "lobato": _lib.SCATTER_LOBATO, "xtables": _lib.SCATTER_XTABLES}[table]
    _lib.check(L.dsx_structure_factor(
        _lib.ptr(d_hkl), n, rec9, _lib.ptr(d_fx), _lib.ptr(d_el), _lib.ptr(d_occ), _lib.ptr(d_B),
        n_atoms, _lib.ptr(d_co), n_elem, sc, _lib.ptr(g4), _lib.ptr(F2), _lib.ptr(F),
        _lib.stream_handle()), "structure factors")
    _lib.check(L.dsx_structure_factor_adjoint(
        _lib.ptr(d_hkl), n, rec9, _lib.ptr(d_fx), _lib.ptr(d_el), _lib.ptr(d_occ), _lib.ptr(d_B),
        n_atoms, _lib.ptr(d_co), n_elem, sc, _lib.ptr(d_w), _lib.ptr(dx), _lib.ptr(dB),
        _lib.ptr(dr), _lib.stream_handle()), "adjoint")
    torch.cuda.synchronize()

    H = hkl[:, :3].astype(np.int64)
    g = H @ rec.T
    g2 = (g * g).sum(1)
    grad, mag = np.zeros((n_atoms, 4)), np.zeros((n_atoms, 4))
    gr, gm = np.zeros((3, 3)), np.zeros((3, 3))
    got, got2 = F.cpu().numpy().astype(np.float64), F2.cpu().numpy().astype(np.float64)
    assert np.abs(g4.cpu().numpy() - np.c_[g, g2]).max() <= 1e-7 * max(np.abs(g).max(), g2.max())
    for r0 in range(0, n, 4096):
        s = slice(r0, r0 + 4096)
        q = g2[s, None]
        f = O.atomic_f(g2[s], co, table)
        e = 1e-6 * np.maximum(g2[s], 1e-3)[:, None]  # central difference of f in g^2
        df = (O.atomic_f(g2[s] + e[:, 0], co, table) - O.atomic_f(g2[s] - e[:, 0], co, table)) / (2 * e)
        turn = (H[s] @ fx[:, :3].astype(np.int64).T) % 2 ** 32
        od = occ.astype(np.float64) * np.exp(-0.25 * q * B.astype(np.float64))
        ph = np.exp(2j * np.pi * (turn / 2.0 ** 32))
        t = f[:, elem] * od * ph
        tq = (df[:, elem] - 0.25 * B * f[:, elem]) * od * ph
        F64, S, SQ = t.sum(1), np.abs(t).sum(1), np.abs(tq).sum(1)
        err = np.abs(got[s, 0] + 1j * got[s, 1] - F64)
        assert (err <= 5e-7 * S).all(), (err / S).max()
        err2 = np.abs(got2[s] - np.abs(F64) ** 2)
        assert (err2 <= 1e-6 * S * np.abs(F64) + (5e-7 * S) ** 2 + 1e-7 * np.abs(F64) ** 2).all()
        ww = w[s, None].astype(np.float64)
        c = F64.conj()[:, None] * t
        m = np.abs(ww) * S[:, None] * np.abs(t)
        for j in range(3):
            grad[:, j] += (-4 * np.pi * ww * H[s, j, None] * c.imag).sum(0)
            mag[:, j] += (4 * np.pi * m * np.abs(H[s, j, None])).sum(0)
        grad[:, 3] += (-0.5 * ww * q * c.real).sum(0)
        mag[:, 3] += (0.5 * m * q).sum(0)
        dq = w[s] * 2.0 * (F64.conj() * tq.sum(1)).real
        dm = np.abs(w[s]) * 2.0 * S * SQ
        gr += np.einsum("n,ni,nj->ij", dq, 2 * g[s], H[s])
        gm += np.einsum("n,ni,nj->ij", dm, np.abs(2 * g[s]), np.abs(H[s]))
    out = np.c_[dx.cpu().numpy(), dB.cpu().numpy()]
    assert (np.abs(out - grad) <= 2e-6 * mag + 1e-30).all(), (np.abs(out - grad) / (mag + 1e-30)).max()
    out = dr.cpu().numpy().reshape(3, 3)
    assert (np.abs(out - gr) <= 2e-6 * gm + 1e-30).all(), (np.abs(out - gr) / (gm + 1e-30)).max()


@pytest.mark.parametrize("n_atoms", [48, 200])
def test_structure_factor_adjoint_sums_few_block_partials(n_atoms):
    """dL/dxyz and dL/dB of 60,000 rows: blocks of at least 256 rows add their FP32
    sums to the output.  b partial sums of random sign reach the total M as
    sqrt(i / b) M, each addition rounds with 2^-24 / sqrt(6) of that, so the error is
    2^-24 sqrt(b / 12) M; the rows' FP32 phases and factors add some 1.2e-7 M.  A
    third more is granted, over the mean of four runs (the additions' order
    varies); blocks of 64 rows come out at twice the first part."""
    import ctypes

    from diffsims_amd import _lib

    n, n_elem = 60000, 4
    print(f"structure-factor adjoint: {n} rows {n_atoms} atoms", flush=True)
    rng = np.random.default_rng(n_atoms)
    h, l = np.divmod(np.arange(n), 40)
    hkl = np.stack([h % 41 - 20, h // 41 - 18, 19 - l, 0 * l], 1).astype(np.int32)
    rec = np.array([[0.05, 0.003, 0.001], [0.0, 0.04, -0.002], [0.0, 0.0, 0.03]])
    fx = rng.integers(0, 2 ** 32, (n_atoms, 4), dtype=np.uint64).astype(np.uint32)
    elem = rng.integers(0, n_elem, n_atoms).astype(np.int32)
    occ = rng.uniform(0.5, 1.0, n_atoms).astype(np.float32)
    B = rng.uniform(0.2, 2.0, n_atoms).astype(np.float32)
    co = np.stack([rng.uniform(0.2, 2.0, (n_elem, 5)), rng.uniform(0.5, 8.0, (n_elem, 5))], -1)
    w = rng.normal(size=n).astype(np.float32)
    L = _lib.load()
    dev = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()
    d_hkl, d_fx, d_el, d_occ, d_B, d_co, d_w = (dev(v) for v in (
        hkl, fx.view(np.int32), elem, occ, B, co.reshape(n_elem, 10), w))
    rec9 = (ctypes.c_double * 9)(*rec.reshape(-1).tolist())
    got = []
    for _ in range(4):
        dx, dB = torch.zeros((n_atoms, 3), device="cuda"), torch.zeros(n_atoms, device="cuda")
        dr = torch.zeros(9, dtype=torch.float64, device="cuda")
        _lib.check(L.dsx_structure_factor_adjoint(
            _lib.ptr(d_hkl), n, rec9, _lib.ptr(d_fx), _lib.ptr(d_el), _lib.ptr(d_occ), _lib.ptr(d_B),
            n_atoms, _lib.ptr(d_co), n_elem, _lib.SCATTER_LOBATO, _lib.ptr(d_w), _lib.ptr(dx),
            _lib.ptr(dB), _lib.ptr(dr), _lib.stream_handle()), "adjoint")
        got.append(torch.cat([dx, dB[:, None]], 1).double())
    H = d_hkl[:, :3].long()
    g2 = ((H.double() @ dev(rec).T) ** 2).sum(1)
    f = dev(np.stack([O.atomic_f(g2.cpu().numpy(), c[None], "lobato")[:, 0] for c in co], 1))
    ref = torch.zeros_like(got[0])
    for s in (slice(r, r + 10000) for r in range(0, n, 10000)):
        turn = (H[s, None, :] * dev(fx[:, :3].astype(np.int64))[None]).sum(-1) & 0xffffffff
        t = f[s][:, d_el.long()] * d_occ.double() * torch.exp(-0.25 * g2[s, None] * d_B.double())
        t = t * torch.exp(2j * np.pi * (turn.double() / 2.0 ** 32))
        c = d_w[s, None].double() * t.sum(1).conj()[:, None] * t
        ref[:, :3] += torch.stack([(-4 * np.pi * H[s, j, None] * c.imag).sum(0) for j in range(3)], 1)
        ref[:, 3] += (-0.5 * g2[s, None] * c.real).sum(0)
    tol = 1.33 * np.hypot(2.0 ** -24 * np.sqrt(n / 256 / 12), 1.2e-7)
    for part in (slice(0, 3), slice(3, 4)):
        err = [float((v[:, part] - ref[:, part]).norm() / ref[:, part].norm()) for v in got]
        assert np.mean(err) <= tol, (err, tol)


@pytest.mark.parametrize("atoms_of_cell,reps,radius", [(8, 2, 1.5), (4, 2, 1.5), (8, 2, 2.5), (8, 3, 0.7)])
def test_extinct_reflections_of_large_cells_stay_extinct(atoms_of_cell, reps, radius):
    """Supercells of the diamond and face-centred cell: every reflection that is
    not one of the small cell's, or is extinct in it, has |F|^2 below 1e-20 of the
    largest, the relative cut's default, where the positions (eighths) are exact
    in 32-bit fixed point; for the 3 x 3 x 3 cell, whose thirds are off by up to
    2^-33 turns per index (|h| + |k| + |l| <= 3 x 12), within (2 pi 36 / 2^33)^2 =
    7e-16 x 64 of it (all the error in one direction, FP32 phases 1.3e-7)."""
    from diffsims_amd import engine
    from diffsims_amd.crystallography import PhaseArrays

    si = np.array([(0, 0, 0), (0, 2, 2), (2, 0, 2), (2, 2, 0), (1, 1, 1), (1, 3, 3), (3, 1, 3),
                   (3, 3, 1)])[:atoms_of_cell] / 4.0
    xyz = np.concatenate([(si + np.array(t)) / reps for t in np.ndindex(reps, reps, reps)])
    pa = PhaseArrays((5.43 * reps,) * 3, (90.0,) * 3, ["Si"] * len(xyz), xyz, np.ones(len(xyz)),
                     np.full(len(xyz), 0.3), "t")
    tab = engine.build_phase_table(pa, radius, False, "lobato")
    hkl = tab.hkl_host()[:, :3].astype(np.int64)
    F2 = tab.F2.cpu().numpy().astype(np.float64)[:len(hkl)]
    sub = (hkl % reps == 0).all(1)
    m = hkl // reps
    allowed = sub & ((m % 2 == m[:, :1] % 2).all(1))
    if atoms_of_cell == 8:
        allowed &= (m % 2 == 1).all(1) | (m.sum(1) % 4 == 0)
    print(f"{len(hkl)} reflections, {allowed.sum()} allowed", flush=True)
    assert allowed.any() and (F2[allowed] > 0).all()
    assert F2[~allowed].max() <= (1e-20 if reps == 2 else 7e-14) * F2.max()
