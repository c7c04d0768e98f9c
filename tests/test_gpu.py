"""Parity of the HIP path (through the C ABI) with the oracle and with the
compiled reference's fixtures.  Needs an MI355X.

Bars: FP64 forces RMS relative error <= 1e-10 against the oracle (and every
printed REVCON digit of the reference), energies/virials <= 1e-11 relative,
neighbour pair set bit-exact; mixed precision forces RMS relative error
<= 1e-5, energies <= 1e-6."""
import os
import tempfile

import numpy as np
import pytest

import fixtures
import oracle
from dlpx import fileio, lib, runner, systems

pytestmark = pytest.mark.gpu

STATIC = [n for n in fixtures.NAMES if "nve" not in n]
TRAJ = [n for n in fixtures.NAMES if "nve" in n]


def rms_rel(f, ref):
    return float(np.sqrt(((f - ref) ** 2).sum() / (ref ** 2).sum()))


def gpu_two_body(s, precision=lib.FP64, pos=None, **kw):
    ctx = lib.Context(s, precision=precision, **kw)
    p = s.pos if pos is None else pos
    ctx.link_cell_pairs(p)
    r = ctx.two_body_forces(p)
    return ctx, r


def energy_scales(o, mixed=False):
    """The largest term of engcpe, vircpe, engsrp and virsrp in an oracle
    result: engcpe is the sum of the self, reciprocal, real-space and
    exclusion-correction energies, which cancel where the charges are weak (a
    mixture: +5.5e6 reciprocal, -6.6e6 self, -1.1e6 total) or the molecules
    are polar (2e7 terms, 7e4 total); the rounding of the terms is what bounds
    the total.  The same terms bound vircpe: the real-space Coulomb virial is
    the real-space stress trace less the vdW virial, and with exclusions the
    reciprocal sum carries each molecule's own smooth interaction (the size of
    the self and correction energies) until the FP64 correction removes it.
    engsrp and virsrp are likewise sums of pair terms of both signs (repulsive
    ZBL pairs beside attractive ones, a molecule's repulsive and attractive
    neighbours): their rounding scales with the summed magnitudes, of which
    1e-2 (FP64: summation order) or all (mixed: every pair term carries its
    own FP32 rounding) bound the error with the check's relative tolerance."""
    b = o["buffer"]
    eng = max(abs(o["eng_recip"]), abs(o["eng_self"]), abs(b[11]), abs(b[15]))
    f = 1.0 if mixed else 1e-2
    return dict(engcpe=eng, vircpe=max(eng, abs(b[8]), abs(b[10]), abs(b[12]), abs(b[16])),
                engsrp=f * o["engvdw_abs"], virsrp=f * o["virvdw_abs"])


def check_energies(r, ref, tol, scales=None):
    """Energies and virials within tol relative to the reference value, or to
    scales[k] where that is larger (see energy_scales)."""
    for k in ("engsrp", "engcpe", "virsrp", "vircpe"):
        scale = max(abs(ref[k]), 1.0, (scales or {}).get(k, 0.0))
        assert abs(r[k] - ref[k]) <= tol * scale, (k, r[k], ref[k])


@pytest.mark.parametrize("name", STATIC)
def test_fp64_matches_oracle_and_reference(name):
    s, ref = fixtures.load(name)
    print("case", name, flush=True)
    o = oracle.two_body(s)
    ctx, r = gpu_two_body(s)
    assert rms_rel(r["frc"], o["frc"]) <= 1e-10
    assert np.abs(r["frc"] - o["frc"]).max() <= 1e-10 * np.abs(o["frc"]).max()
    check_energies(r, o, 1e-11, energy_scales(o))
    assert np.abs(r["stress"] - o["stress"]).max() <= 1e-11 * np.abs(o["stress"]).max()
    assert np.allclose(r["buffer"], o["buffer"], rtol=1e-11, atol=1e-9)
    # and the reference itself: all printed force digits, full-precision energies
    bound = fixtures.printed_digits_bound(ref["frc"]) + 1e-12 * np.abs(ref["frc"]).max()
    assert (np.abs(fixtures.frozen_zeroed(s, r["frc"]) - ref["frc"]) / bound).max() <= 1.05
    check_energies(r, ref, 1e-11, energy_scales(o))
    # the reference's own forces at full precision (its two_body_forces output)
    assert rms_rel(r["frc"], ref["frc64"]) <= 1e-12
    assert np.abs(r["frc"] - ref["frc64"]).max() <= 1e-11 * np.abs(ref["frc64"]).max()
    ctx.close()


@pytest.mark.parametrize("name", ["nacl_1000_k45_27_25_s6", "nacl_1000_k30_36_40_s6", "mix_4000_k36"])
def test_generic_and_line_ffts_agree(name, monkeypatch):
    """The FFT lengths with compiled line kernels (the default for them) and
    the generic Stockham kernels (DLPX_FFT_LINES=0, every length) agree to
    FP64 rounding in forces, energies and the reciprocal stress, and each
    matches the oracle, in both precisions; the meshes cover odd, even and
    mixed-radix edges (45, 27, 25; 30, 36, 40; 36)."""
    s, _ = fixtures.load(name)
    print("case", name, flush=True)
    o = oracle.two_body(s)
    for precision, tol in ((lib.FP64, 1e-10), (lib.MIXED, 1e-5)):
        res = {}
        for lines in ("1", "0"):
            monkeypatch.setenv("DLPX_FFT_LINES", lines)
            ctx, res[lines] = gpu_two_body(s, precision)
            ctx.close()
            assert rms_rel(res[lines]["frc"], o["frc"]) <= tol
            check_energies(res[lines], o, 1e-11 if precision == lib.FP64 else 1e-6,
                           energy_scales(o, mixed=precision == lib.MIXED))
        a, b = res["1"], res["0"]
        agree = 1e-12 if precision == lib.FP64 else 1e-6
        assert rms_rel(a["frc"], b["frc"]) <= agree
        assert np.abs(a["stress"] - b["stress"]).max() <= agree * np.abs(b["stress"]).max()
        assert abs(a["engcpe"] - b["engcpe"]) <= agree * abs(b["engcpe"])


@pytest.mark.parametrize("name", ["nacl_1000_k32", "mix_4000_k36", "nacl_4096_k48", "mol3_2592_k32"])
def test_plane_and_line_ffts_agree(name, monkeypatch):
    """The x and y passes fused per z-plane (the default for meshes with
    K1 = K2 of a line-kernel length) and the separate x and y line kernels
    (DLPX_FFT_PLANES=0) agree to FP64 rounding in forces, energies and the
    reciprocal stress, and each matches the oracle, in both precisions
    (meshes 32 = 8x4, 36 = 6x6, 48 = 12x4)."""
    s, _ = fixtures.load(name)
    print("case", name, flush=True)
    o = oracle.two_body(s)
    for precision, tol in ((lib.FP64, 1e-10), (lib.MIXED, 1e-5)):
        res = {}
        for planes in ("1", "0"):
            monkeypatch.setenv("DLPX_FFT_PLANES", planes)
            ctx, res[planes] = gpu_two_body(s, precision)
            ctx.close()
            assert rms_rel(res[planes]["frc"], o["frc"]) <= tol
            check_energies(res[planes], o, 1e-11 if precision == lib.FP64 else 1e-6,
                           energy_scales(o, mixed=precision == lib.MIXED))
        a, b = res["1"], res["0"]
        agree = 1e-12 if precision == lib.FP64 else 1e-6
        assert rms_rel(a["frc"], b["frc"]) <= agree
        assert np.abs(a["stress"] - b["stress"]).max() <= agree * np.abs(b["stress"]).max()
        assert abs(a["engcpe"] - b["engcpe"]) <= agree * abs(b["engcpe"])


def test_diverged_coordinates_stay_in_range():
    """Coordinates scaled by 1e30, as a diverging run leaves them: the fold
    at the list build cannot bring them back (its rounding exceeds the cell
    by far), so every link cell's atoms reach the spreading with grid
    coordinates beyond the int range.  The window bounds are held to
    +-2^20 (unbounded, they saturated, overflowed in the window's
    one-period test and indexed the grid out of range), so the call returns
    normally in both precisions (the forces are meaningless)."""
    s, _ = fixtures.load("nacl_1000_k32")
    pos = np.array(s.pos, dtype=np.float64, copy=True) * 1.0e30
    for precision in (lib.FP64, lib.MIXED):
        print("case diverged precision", precision, flush=True)
        ctx, r = gpu_two_body(s, precision, pos=pos)
        ctx.close()
        assert r["frc"].shape == pos.shape


@pytest.mark.parametrize("k", [25, 27, 45])
def test_plane_kernels_on_odd_meshes(k, monkeypatch):
    """The plane kernels with an odd edge (25 = 5x5, 27 = 9x3, 45 = 9x5):
    the last row pair of a plane holds one real row, and the half spectrum
    has no Nyquist column.  NaCl 1000 on a k^3 mesh (S = 6) against the
    oracle and against the separate line kernels, both precisions."""
    import dataclasses
    s0, _ = fixtures.load("nacl_1000_k32")
    s = dataclasses.replace(s0, kvec=(k, k, k), nsplines=6)
    print("case odd mesh", k, flush=True)
    o = oracle.two_body(s)
    for precision, tol in ((lib.FP64, 1e-10), (lib.MIXED, 1e-5)):
        res = {}
        for planes in ("1", "0"):
            monkeypatch.setenv("DLPX_FFT_PLANES", planes)
            ctx, res[planes] = gpu_two_body(s, precision)
            ctx.close()
            assert rms_rel(res[planes]["frc"], o["frc"]) <= tol
            check_energies(res[planes], o, 1e-11 if precision == lib.FP64 else 1e-6,
                           energy_scales(o, mixed=precision == lib.MIXED))
        agree = 1e-12 if precision == lib.FP64 else 1e-6
        assert rms_rel(res["1"]["frc"], res["0"]["frc"]) <= agree
        assert np.abs(res["1"]["stress"] - res["0"]["stress"]).max() <= agree * np.abs(res["0"]["stress"]).max()


@pytest.mark.parametrize("name", ["mix_4000_k36", "mix4_4000_k36", "mol3_2592_k32"])
def test_mixed_relative_and_fp64_separations_agree(name, monkeypatch):
    """The mixed combined-table pair kernel with separations from
    subcell-relative FP32 positions and list codes (the default where the
    list is built over subcells) and with FP64 minimum-image separations
    (DLPX_REL_PAIRS=0): both within the mixed bar of the oracle, and within
    it of each other."""
    s, _ = fixtures.load(name)
    print("case", name, flush=True)
    o = oracle.two_body(s)
    res = {}
    for rel in ("1", "0"):
        monkeypatch.setenv("DLPX_REL_PAIRS", rel)
        ctx, res[rel] = gpu_two_body(s, lib.MIXED)
        ctx.close()
        assert rms_rel(res[rel]["frc"], o["frc"]) <= 1e-5
        check_energies(res[rel], o, 1e-6, energy_scales(o, mixed=True))
    assert rms_rel(res["1"]["frc"], res["0"]["frc"]) <= 1e-5


@pytest.mark.parametrize("name", [n for n in STATIC if "tab_pot" in fixtures.load(n)[1]])
def test_reference_vdw_tables_through_set_vdw_tables(name):
    """The host-table route: DL_POLY's own vdws%tab_potential / tab_force
    (dumped from the reference run) and its vdws%elrc / vlrc given through
    dlpx_set_vdw_tables and dlpx_set_lrc, as a Fortran host passes them.
    FP64 forces against the reference's full-precision forces (1e-12 RMS),
    energies against its two_body_forces output; mixed within 1e-5."""
    s, ref = fixtures.load(name)
    print("case", name, flush=True)
    mg, pot, frc, ltp = fixtures.reference_tables(s, ref)
    tables = dict(max_grid=mg, vdw_pot=pot, vdw_frc=frc, ltp=ltp)
    o = oracle.two_body(s)
    for precision, tf in ((lib.FP64, 1e-12), (lib.MIXED, 1e-5)):
        scales = energy_scales(o, mixed=precision == lib.MIXED)
        ctx = lib.Context(s, precision=precision, tables=tables, lrc=(ref["elrc"], ref["vlrc"]))
        if s.electrostatics:
            ctx._chk(ctx.lib.dlpx_generate_erfc_tables(ctx.h))
        ctx.link_cell_pairs(s.pos)
        r = ctx.two_body_forces(s.pos)
        ctx.close()
        assert rms_rel(r["frc"], ref["frc64"]) <= tf
        dump = {k: ref["dump_" + k] for k in ("engcpe", "vircpe", "engsrp", "virsrp")}
        check_energies(r, dump, 1e-11 if precision == lib.FP64 else 1e-6, scales)


@pytest.mark.parametrize("name", STATIC)
def test_pair_set_bit_exact(name):
    s, _ = fixtures.load(name)
    print("case", name, flush=True)
    ctx = lib.Context(s)
    npairs, ibig = ctx.link_cell_pairs(s.pos)
    g = ctx.get_pairs()
    o = oracle.pairs(s.cell, s.pos, s.cutoff + s.padding, "cells")
    # ibig counts every pair within reach, excluded ones too (neighbours.F90:1189)
    counts = np.bincount(o[:, :2].ravel(), minlength=s.natms)
    assert ibig == counts.max()
    excl = s.exclusions()
    if excl is not None:
        # excluded pairs leave the list (neighbours.F90:1229-1250)
        keep = np.array([p[1] not in set(excl[p[0]]) for p in o], bool)
        assert (~keep).sum() > 0
        o = o[keep]
    if s.frozen is not None:
        # so do pairs of two frozen atoms (neighbours.F90:1198-1225)
        keep = ~(s.frozen[o[:, 0]] & s.frozen[o[:, 1]])
        assert (~keep).sum() > 0
        o = o[keep]
    assert npairs == len(o) == len(g)
    assert {tuple(p) for p in g} == {tuple(p) for p in o}
    ctx.close()


@pytest.mark.parametrize("name", ["nacl_4096_k48", "mix_4000_k36", "argon_4000_jit"])
def test_count_pairs_matches_host_count(name):
    """dlpx_count_pairs (device count of listed pairs closer than r) equals the
    count of dlpx_get_pairs' pairs closer than r measured on the host, at the
    cutoff and inside it."""
    s, _ = fixtures.load(name)
    print("case", name, flush=True)
    ctx = lib.Context(s, precision=lib.FP64)
    ctx.link_cell_pairs(s.pos)
    p = ctx.get_pairs()
    L = np.diag(s.cell.reshape(3, 3))
    x = s.pos - L * np.floor(s.pos / L + 0.5)
    d2 = ((x[p[:, 0]] - (x[p[:, 1]] + p[:, 2:5] * L)) ** 2).sum(1)
    for r in (max(s.cutoff, s.vdw_cutoff), 0.8 * s.cutoff):
        assert ctx.count_pairs(r) == int((d2 < r * r).sum())
    ctx.close()


@pytest.mark.parametrize("name", ["argon_4000_jit", "nacl_4096_k48"])
def test_link_cell_and_subcell_builds_give_the_same_set(name, monkeypatch):
    # boxes with >= 3 link cells per axis use the subcell build by default;
    # DLPX_LIST_SUBCELLS=0 (read at context creation) selects the link-cell build
    s, _ = fixtures.load(name)
    print("case", name, flush=True)
    sets = []
    for flag in ("0", "1"):
        monkeypatch.setenv("DLPX_LIST_SUBCELLS", flag)
        ctx = lib.Context(s)
        npairs, ibig = ctx.link_cell_pairs(s.pos)
        g = ctx.get_pairs()
        assert npairs == len(g)
        sets.append(({tuple(p) for p in g}, ibig))
        ctx.close()
    assert sets[0] == sets[1]


@pytest.mark.parametrize("name", STATIC)
def test_mixed_precision_error_budget(name):
    s, _ = fixtures.load(name)
    print("case", name, flush=True)
    o = oracle.two_body(s)
    ctx, r = gpu_two_body(s, precision=lib.MIXED)
    assert rms_rel(r["frc"], o["frc"]) <= 1e-5
    check_energies(r, o, 1e-6, energy_scales(o, mixed=True))
    ctx.close()


@pytest.mark.parametrize("name", STATIC)
def test_per_particle_matches_oracle_and_reference_heat_flux(name):
    """stats%collect_pp through dlpx_set_per_particle / dlpx_add_per_particle:
    every atom's energy and stress against the oracle (FP64, 1e-10 of the
    largest), the reference's HEATFLUX record and its per-particle-mode stress;
    the next call without collection is back on the k-space stress; mixed
    precision within 1e-5 RMS."""
    s, ref = fixtures.load(name)
    print("case", name, flush=True)
    z = np.load(os.path.join(fixtures.GOLDEN, name + ".npz"))
    o = oracle.two_body(s, per_particle=True)
    ctx = lib.Context(s)
    ctx.link_cell_pairs(s.pos)
    r = ctx.two_body_forces(s.pos, per_particle=True)
    assert np.abs(r["pp_energy"] - o["pp_energy"]).max() <= 1e-10 * np.abs(o["pp_energy"]).max()
    assert np.abs(r["pp_stress"] - o["pp_stress"]).max() <= 1e-10 * np.abs(o["pp_stress"]).max()
    hf, want = fixtures.heat_flux(s, r["pp_energy"], r["pp_stress"]), z["ref_heatflux"]
    assert np.abs(hf - want).max() <= 1e-10 * np.abs(want).max()
    assert np.abs(r["stress"] - z["ref_pp_stress"]).max() <= 1e-11 * np.abs(z["ref_pp_stress"]).max()
    assert rms_rel(r["frc"], o["frc"]) <= 1e-10
    r2 = ctx.two_body_forces(s.pos)
    assert "pp_energy" not in r2
    assert np.abs(r2["stress"] - ref["stress"]).max() <= 1e-11 * np.abs(ref["stress"]).max()
    ctx.close()
    ctx = lib.Context(s, precision=lib.MIXED)
    ctx.link_cell_pairs(s.pos)
    rm = ctx.two_body_forces(s.pos, per_particle=True)
    assert rms_rel(rm["pp_energy"], o["pp_energy"]) <= 1e-5
    assert rms_rel(rm["pp_stress"], o["pp_stress"]) <= 1e-5
    ctx.close()


def _tiny_nacl(n_pairs=4, L=26.0, seed=5):
    """A few ions scattered (at least 2.4 A apart) in a box just over twice
    the cutoff: fewer atoms than a wavefront, 2 link cells per axis (the
    link-cell list path), most cells empty."""
    rng = np.random.default_rng(seed)
    pos = []
    while len(pos) < 2 * n_pairs:
        p = rng.uniform(-L / 2, L / 2, 3)
        if all(np.linalg.norm((p - q) - L * np.round((p - q) / L)) > 2.4 for q in pos):
            pos.append(p)
    base = systems.nacl(ncells=1, kvec=(24, 24, 24), cutoff=12.0, padding=0.5)
    types = np.array([0, 1] * n_pairs, np.int32)
    order = np.argsort(types, kind="stable")
    vel = rng.normal(scale=5.0, size=(2 * n_pairs, 3))
    return systems.System(name="tiny", cell=np.diag([L, L, L]).reshape(9), pos=np.array(pos)[order],
                          vel=vel[order], types=types[order], type_names=base.type_names, masses=base.masses,
                          charges=base.charges, vdw=base.vdw, cutoff=12.0, padding=0.5, vdw_cutoff=12.0,
                          electrostatics=True, alpha=0.28, kvec=(24, 24, 24), nsplines=8, timestep=0.002)


@pytest.mark.parametrize("n_pairs", [1, 4, 40])
def test_tiny_systems_match_oracle(n_pairs):
    """2 to 80 ions: partial wavefronts and workgroups, empty link cells, the
    link-cell (not subcell) list build; FP64 to 1e-10, mixed to 1e-5, and
    the pair set exactly."""
    s = _tiny_nacl(n_pairs)
    print("case tiny", s.natms, flush=True)
    o = oracle.two_body(s)
    ctx, r = gpu_two_body(s)
    assert rms_rel(r["frc"], o["frc"]) <= 1e-10
    check_energies(r, o, 1e-11, energy_scales(o))
    g = ctx.get_pairs()
    op = oracle.pairs(s.cell, s.pos, s.cutoff + s.padding, "brute")
    assert {tuple(p) for p in g} == {tuple(p) for p in op}
    ctx.close()
    ctx, rm = gpu_two_body(s, precision=lib.MIXED)
    assert rms_rel(rm["frc"], o["frc"]) <= 1e-5
    ctx.close()


def _split_types(s, scale=1.01):
    """Every species split into two atom types (alternate atoms), the copies'
    vdW energy parameters scaled by ``scale``: 2 ntypes types whose distinct
    tables no longer fit in LDS beside the erfc table."""
    nt = s.ntypes
    types = np.where(np.arange(s.natms) % 2 == 1, s.types + nt, s.types).astype(np.int32)
    order = np.argsort(types, kind="stable")
    par = {(max(a, b), min(a, b)): (k, p) for (a, b, k, p) in s.vdw}
    energy_param = {1: (0, 1), 2: (0,), 3: (0,), 4: (0, 2), 5: (0, 3, 4), 6: (0, 1), 8: (0,)}
    vdw = []
    for i in range(2 * nt):
        for j in range(i + 1):
            k, p = par[(max(i % nt, j % nt), min(i % nt, j % nt))]
            f = scale ** ((i >= nt) + (j >= nt))
            vdw.append((i, j, k, tuple(v * f if q in energy_param[k] else v for q, v in enumerate(p))))
    return systems.System(name=s.name + "_split", cell=s.cell, pos=s.pos[order], vel=s.vel[order],
                          types=types[order], type_names=list(s.type_names) + [n + "2" for n in s.type_names],
                          masses=np.concatenate([s.masses, s.masses]), charges=np.concatenate([s.charges, s.charges]),
                          vdw=vdw, cutoff=s.cutoff, padding=s.padding, vdw_cutoff=s.vdw_cutoff,
                          electrostatics=s.electrostatics, alpha=s.alpha, kvec=s.kvec, nsplines=s.nsplines,
                          timestep=s.timestep)


def test_many_types_read_vdw_tables_from_global_memory():
    """Six atom types with 21 distinct vdW tables (336 KiB in FP64, 168 KiB
    in FP32): beyond the LDS, so the pair kernel reads them from global
    memory; FP64 to 1e-10 of the oracle, mixed to 1e-5."""
    s0, _ = fixtures.load("mix_4000_k36")
    s = _split_types(s0)
    print("case split mixture", s.ntypes, "types", flush=True)
    o = oracle.two_body(s)
    ctx, r = gpu_two_body(s)
    assert rms_rel(r["frc"], o["frc"]) <= 1e-10
    check_energies(r, o, 1e-11, energy_scales(o))
    ctx.close()
    ctx, rm = gpu_two_body(s, precision=lib.MIXED)
    assert rms_rel(rm["frc"], o["frc"]) <= 1e-5
    ctx.close()


def test_half_empty_box_matches_oracle():
    """Argon atoms kept only in the lower half of the box (z < 0): half the
    link cells and subcells are empty."""
    s, _ = fixtures.load("argon_4000_jit")
    keep = s.pos[:, 2] < 0.0
    s.pos, s.vel, s.types = s.pos[keep], s.vel[keep], s.types[keep]
    print("case half-empty argon", s.natms, flush=True)
    o = oracle.two_body(s)
    ctx, r = gpu_two_body(s)
    assert rms_rel(r["frc"], o["frc"]) <= 1e-10
    check_energies(r, o, 1e-11)
    ctx.close()


def test_unfolded_positions_give_the_same_forces():
    """Positions outside the cell (a third of the ions moved by a lattice
    vector, as a host that does not fold them would pass them): the same
    forces, energies and pair set as the folded configuration."""
    s, _ = fixtures.load("nacl_1000_k32")
    print("case unfolded nacl 1000", flush=True)
    L = np.diag(s.cell.reshape(3, 3))
    rng = np.random.default_rng(2)
    shift = rng.integers(-1, 2, size=s.pos.shape) * (rng.random(s.natms) < 1 / 3)[:, None]
    ctx, r = gpu_two_body(s)
    ctx2, r2 = gpu_two_body(s, pos=s.pos + shift * L)
    assert np.abs(r2["frc"] - r["frc"]).max() <= 1e-11 * np.abs(r["frc"]).max()
    for k in ("engsrp", "engcpe", "virsrp", "vircpe"):
        assert abs(r2[k] - r[k]) <= 1e-12 * max(abs(r[k]), abs(r["buffer"][10]), 1.0), k
    assert {tuple(p[:2]) for p in ctx.get_pairs()} == {tuple(p[:2]) for p in ctx2.get_pairs()}
    ctx.close()
    ctx2.close()


def test_forces_added_to_existing_and_aos_stride():
    """Forces are added to what the caller's arrays hold, and a 64-byte
    array-of-structures record (DL_POLY's corePart: x, y, z, charge, fx,
    fy, fz, one spare double per atom) through dlpx_atoms' byte stride gives
    the same pairs, forces and energies as packed arrays."""
    s, _ = fixtures.load("nacl_1000_k32")
    ctx = lib.Context(s)
    ctx.link_cell_pairs(s.pos)
    base = np.full((s.natms, 3), 7.25)
    r1 = ctx.two_body_forces(s.pos)
    r2 = ctx.two_body_forces(s.pos, frc=base.copy())
    assert np.array_equal(r2["frc"] - 7.25, r1["frc"] + 7.25 - 7.25) or \
        np.abs(r2["frc"] - 7.25 - r1["frc"]).max() < 1e-12 * np.abs(r1["frc"]).max()
    # the same call on a 64-byte record per atom, forces starting from 1.5
    rec = np.zeros((s.natms, 8))
    rec[:, 0:3] = s.pos
    rec[:, 3] = ctx.q
    rec[:, 4:7] = 1.5
    b = rec.ctypes.data
    a = lib.Atoms(natms=s.natms, stride=64, x=b, y=b + 8, z=b + 16, chge=b + 24, fx=b + 32, fy=b + 40, fz=b + 48,
                  ltype=ctx.ltype.ctypes.data)
    npairs, ibig = lib.C.c_int64(), lib.C.c_int32()
    ctx._chk(ctx.lib.dlpx_link_cell_pairs(ctx.h, lib._ptr(ctx.cell), lib.C.byref(a), lib.C.byref(npairs),
                                          lib.C.byref(ibig)))
    o = lib.TwoBodyOut()
    ctx._chk(ctx.lib.dlpx_two_body_forces(ctx.h, lib._ptr(ctx.cell), lib.C.byref(a), lib.C.byref(o)))
    ctx.close()
    assert np.abs(rec[:, 4:7] - 1.5 - r1["frc"]).max() <= 1e-12 * np.abs(r1["frc"]).max()
    assert np.array_equal(rec[:, 0:3], s.pos) and np.all(rec[:, 7] == 0.0)  # inputs and the spare word untouched
    assert abs(o.engsrp - r1["engsrp"]) <= 1e-12 * abs(r1["engsrp"])
    assert abs(o.engcpe - r1["engcpe"]) <= 1e-12 * abs(r1["engcpe"])


@pytest.mark.parametrize("name", TRAJ)
def test_nve_trajectory_matches_reference(name):
    s, ref = fixtures.load(name)
    print("case", name, flush=True)
    ctx = lib.Context(s)
    ctx.md_load(s.pos, runner.start_velocities(s))
    e, nreb = ctx.md_run(ref["steps"], s.timestep)
    x, v, f = ctx.md_store()
    L = np.diag(s.cell.reshape(3, 3))
    dx = x - ref["pos"]
    dx -= L * np.round(dx / L)
    assert (np.abs(dx) / (fixtures.printed_digits_bound(ref["pos"]) + 1e-12)).max() <= 1.05
    assert (np.abs(v - ref["vel"]) / (fixtures.printed_digits_bound(ref["vel"]) + 1e-12)).max() <= 1.05
    bound = fixtures.printed_digits_bound(ref["frc"]) + 1e-12 * np.abs(ref["frc"]).max()
    assert (np.abs(f - ref["frc"]) / bound).max() <= 1.05
    assert abs(e[-1, 2] - ref["engsrp"]) <= 1e-10 * abs(ref["engsrp"])
    assert abs(e[-1, 0] - ref["engcpe"]) <= 1e-10 * max(abs(ref["engcpe"]), 1.0)
    ctx.close()


@pytest.mark.parametrize("precision", [lib.FP64, lib.MIXED])
@pytest.mark.parametrize("name", TRAJ)
def test_dlpoly_inputs_run_to_the_reference_statis(name, precision):
    """CONFIG/FIELD/CONTROL read back by the host, run on the GPU, and the
    STATIS written for every step compared with the reference's STATIS for the
    same inputs by the reference harness's rule (relative 1e-5,
    utils/beetest:39-48): every column in FP64; the scalar columns (energies,
    virials, temperature, pressure) in mixed precision, whose pressure-tensor
    off-diagonals are too small for a relative test.  For polar molecules the
    Coulomb energy and virial are small sums of large terms (7e4 of 2.4e7
    terms): in mixed precision the columns containing them get the mixed error
    budget of test_mixed_precision_error_budget (1e-6 of the largest term)
    where the relative rule is tighter."""
    s, ref = fixtures.load(name)
    print("case", name, precision, flush=True)
    want = fileio.read_statis(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "statis",
                                           name + ".STATIS"))
    with tempfile.TemporaryDirectory() as d:
        fileio.write_inputs(d, s, steps=int(ref["steps"]))
        res = runner.run_directory(d, precision=precision)
        got = fileio.read_statis(res["statis"])
        rc = fileio.read_config(res["revcon"])
    assert sorted(got) == sorted(want)
    ncol = len(want[0][1])
    cols = range(ncol) if precision == lib.FP64 else [c - 1 for c in fileio.STATIS_COLUMNS.values()]
    budget = {}
    if precision == lib.MIXED:
        # the mixed budget of the Coulomb energy and virial, carried into
        # every column that contains them (statistics.F90:1096-1098,1118-1160)
        sc = energy_scales(oracle.two_body(s), mixed=True)
        de, dv = 1e-6 * sc["engcpe"], 1e-6 * sc["vircpe"]
        col = {k: v - 1 for k, v in fileio.STATIS_COLUMNS.items()}
        budget = {col["eng_cou"]: de, col["eng_cfg"]: de, col["eng_tot"]: de, col["vir_cou"]: dv,
                  col["vir_cfg"]: dv, col["eng_pv"]: de + dv / 3.0,
                  col["press"]: dv / (3.0 * s.volume) * fileio.PRSUNT}

    def ok(k, g, w):
        return fileio.statis_equal(g, w, 1e-5) or (k in budget and abs(g - w) <= budget[k])
    bad = [(step, k + 1, got[step][1][k], w[k]) for step, (_, w) in want.items() for k in cols
           if not ok(k, got[step][1][k], w[k])]
    assert not bad, bad[:10]
    # the written REVCON holds the run's last configuration
    L = np.diag(s.cell.reshape(3, 3))
    dx = rc["pos"] - ref["pos"]
    dx -= L * np.round(dx / L)
    assert np.abs(dx).max() <= (1e-8 if precision == lib.FP64 else 1e-4)


def test_list_overflow_returns_error_106():
    s, _ = fixtures.load("nacl_1000_k32")
    ctx = lib.Context(s, max_list=64)
    with pytest.raises(lib.DlpxError) as ei:
        ctx.link_cell_pairs(s.pos)
    assert ei.value.code == 106 and ei.value.ibig > 64
    ctx.close()


def test_cutoff_beyond_half_cell_returns_error_95():
    s = systems.nacl(ncells=3, kvec=(20, 20, 20), cutoff=9.0, padding=0.5)
    ctx = lib.Context(s)
    with pytest.raises(lib.DlpxError) as ei:
        ctx.link_cell_pairs(s.pos)
    assert ei.value.code == 95
    ctx.close()


def test_vnl_check_trigger():
    s, _ = fixtures.load("nacl_1000_k32")
    ctx = lib.Context(s)
    ctx.link_cell_pairs(s.pos)
    p = s.pos.copy()
    p[17, 0] += 0.2  # < padding/2
    assert ctx.vnl_check(p) is False
    p[17, 0] += 0.06  # 0.26 >= padding/2
    assert ctx.vnl_check(p) is True
    ctx.close()


@pytest.fixture(scope="module")
def nacl64k():
    s = systems.nacl(ncells=20, kvec=(128, 128, 128))
    o = oracle.two_body(s)
    return s, o


def test_full_size_nacl_fp64_and_mixed(nacl64k):
    s, o = nacl64k
    print("case nacl 64000 K=128", flush=True)
    ctx, r = gpu_two_body(s)
    assert rms_rel(r["frc"], o["frc"]) <= 1e-10
    check_energies(r, o, 1e-11)
    ctx.close()
    ctx, rm = gpu_two_body(s, precision=lib.MIXED)
    assert rms_rel(rm["frc"], o["frc"]) <= 1e-5
    check_energies(rm, o, 1e-6, energy_scales(o, mixed=True))
    # net force vanishes (pair forces antisymmetric, mean reciprocal force removed)
    assert np.abs(r["frc"].sum(0)).max() <= 1e-8 * np.abs(r["frc"]).max() * np.sqrt(s.natms)
    ctx.close()


def _resident_forces_vs_oracle(s, steps, precision):
    """Forces of the last resident step against the oracle at the positions
    that step ended with."""
    ctx = lib.Context(s, precision=precision)
    ctx.md_load(s.pos, s.vel)
    ctx.md_run(steps, s.timestep)
    x, v, f = ctx.md_store()
    ctx.close()
    o = oracle.two_body(s, pos=x)
    return rms_rel(f, o["frc"])


@pytest.mark.parametrize("name", ["nacl_4096_k48", "nacl_1440_orth_q", "mol4_3456_k32"])
def test_resident_step_forces_match_oracle(name):
    s, _ = fixtures.load(name)
    print("case", name, flush=True)
    assert _resident_forces_vs_oracle(s, 3, lib.FP64) <= 1e-10
    assert _resident_forces_vs_oracle(s, 3, lib.MIXED) <= 1e-5


def test_resident_step_forces_full_size(nacl64k):
    s, _ = nacl64k
    print("case nacl 64000 K=128 resident", flush=True)
    assert _resident_forces_vs_oracle(s, 2, lib.FP64) <= 1e-10


def test_full_size_1728k_against_strided_oracle_fixture():
    """1,728,000-ion NaCl, mesh 360^3: FP64 forces of every 1000th atom and
    the energies against the oracle (tests/golden/large), mixed against FP64."""
    import os
    z = np.load(os.path.join(fixtures.GOLDEN, "large", "nacl_1728k_strided.npz"))
    s = systems.nacl(ncells=60, kvec=(360, 360, 360), padding=0.5)
    assert np.allclose([s.pos.sum(), (s.pos ** 2).sum()], z["pos_checksum"], rtol=1e-13, atol=0)
    print("case nacl 1728000 K=360", flush=True)
    idx = z["idx"]
    ctx, r = gpu_two_body(s)
    err = np.sqrt(((r["frc"][idx] - z["frc"]) ** 2).mean()) / float(z["frc_rms"])
    assert err <= 1e-10
    e = [r["engcpe"], r["vircpe"], r["engsrp"], r["virsrp"]]
    assert np.all(np.abs(np.array(e) - z["energies"]) <= 1e-11 * np.abs(z["energies"]))
    # ~5e8 pair terms summed in a different order from the oracle's: 1e-10
    assert np.abs(r["stress"] - z["stress"]).max() <= 1e-10 * np.abs(z["stress"]).max()
    f64 = r["frc"]
    assert np.abs(f64.sum(0)).max() <= 1e-8 * np.abs(f64).max() * np.sqrt(s.natms)
    ctx.close()
    ctx, rm = gpu_two_body(s, precision=lib.MIXED)
    assert rms_rel(rm["frc"], f64) <= 1e-5
    check_energies(rm, r, 1e-6)
    ctx.close()


def _chunked_md(s, precision, graphs, chunks=3, steps=12):
    """Resident NVE in chunks; state after each chunk.  DLPX_GRAPHS is read
    when the context is created."""
    import os
    old = os.environ.get("DLPX_GRAPHS")
    os.environ["DLPX_GRAPHS"] = "1" if graphs else "0"
    try:
        ctx = lib.Context(s, precision=precision)
    finally:
        if old is None:
            del os.environ["DLPX_GRAPHS"]
        else:
            os.environ["DLPX_GRAPHS"] = old
    ctx.md_load(s.pos, s.vel)
    out = []
    for _ in range(chunks):
        _, nreb = ctx.md_run(steps, s.timestep, energies=False)
        out.append(ctx.md_store() + (nreb,))
    ctx.close()
    return out


@pytest.mark.parametrize("precision,tol", [(lib.FP64, 1e-9), (lib.MIXED, 1e-5)])
def test_graph_replayed_steps_match_eager_steps(precision, tol):
    """Steps 2..n-1 of each dlpx_md_run replay one captured graph; every chunk
    (several replays, with list rebuilds and host synchronisation between
    them) must agree with the eager path.  The only difference is the order of
    the charge-spreading atomics."""
    s, _ = fixtures.load("nacl_4096_k48")
    print("case graphs vs eager, precision", precision, flush=True)
    eager = _chunked_md(s, precision, graphs=False)
    graph = _chunked_md(s, precision, graphs=True)
    L = np.diag(s.cell.reshape(3, 3))
    assert sum(c[3] for c in eager) > 0  # the run crosses list rebuilds
    for (xe, ve, fe, ne), (xg, vg, fg, ng) in zip(eager, graph):
        assert ne == ng
        dx = xg - xe
        dx -= L * np.round(dx / L)
        assert np.abs(dx).max() <= tol * L.max()
        assert rms_rel(vg, ve) <= tol and rms_rel(fg, fe) <= 10 * tol


@pytest.mark.parametrize("overlap", ["0", "1", "2"])
def test_step_branch_layouts_agree(overlap, monkeypatch):
    """Every layout of a resident step's branches (DLPX_OVERLAP: the
    reciprocal chain on either stream, the pair kernel free or held until the
    spreading is done) and one-step graphs (DLPX_GRAPH_STEPS=1) give the
    eager steps' trajectory, across list rebuilds."""
    s, _ = fixtures.load("nacl_4096_k48")
    print("case layout", overlap, flush=True)
    eager = _chunked_md(s, lib.MIXED, graphs=False)
    monkeypatch.setenv("DLPX_OVERLAP", overlap)
    monkeypatch.setenv("DLPX_GRAPH_STEPS", "1" if overlap == "1" else "8")
    graph = _chunked_md(s, lib.MIXED, graphs=True)
    L = np.diag(s.cell.reshape(3, 3))
    for (xe, ve, fe, ne), (xg, vg, fg, ng) in zip(eager, graph):
        assert ne == ng
        dx = xg - xe
        dx -= L * np.round(dx / L)
        assert np.abs(dx).max() <= 1e-5 * L.max()
        assert rms_rel(vg, ve) <= 1e-5 and rms_rel(fg, fe) <= 1e-4


def test_ensemble_matches_separate_runs():
    """dlpx_md_run_ensemble over systems of different kinds and sizes gives
    each system's own dlpx_md_run (up to the order of the spreading atomics)."""
    syss = [systems.argon(ncells=6, seed=5), systems.nacl(ncells=5, kvec=(32, 32, 32), seed=6),
            systems.nacl(ncells=6, kvec=(40, 40, 40), seed=7)]
    print("case ensemble of", [s.natms for s in syss], flush=True)
    steps = 15
    ref = []
    for s in syss:
        ctx = lib.Context(s)
        ctx.md_load(s.pos, s.vel)
        _, nreb = ctx.md_run(steps, s.timestep, energies=False)
        ref.append(ctx.md_store() + (nreb,))
        ctx.close()
    ctxs = []
    for s in syss:
        ctx = lib.Context(s)
        ctx.md_load(s.pos, s.vel)
        ctxs.append(ctx)
    nreb = lib.md_run_ensemble(ctxs, steps)
    for k, (s, ctx) in enumerate(zip(syss, ctxs)):
        x, v, f = ctx.md_store()
        xr, vr, fr, nr = ref[k]
        L = np.diag(s.cell.reshape(3, 3))
        dx = x - xr
        dx -= L * np.round(dx / L)
        assert nreb[k] == nr
        assert np.abs(dx).max() <= 1e-9 * L.max()
        assert rms_rel(v, vr) <= 1e-9 and rms_rel(f, fr) <= 1e-8
        ctx.close()


@pytest.mark.parametrize("precision,tol", [(lib.FP64, 1e-8), (lib.MIXED, 1e-5)])
def test_ensemble_tuned_run_matches_separate_runs(precision, tol, tmp_path, monkeypatch):
    """A batch run long enough to tune its launch shapes (48 steps: six
    candidate shapes of six steps each, then graph replays) gives each
    system's own dlpx_md_run, writes the chosen shape to DLPX_TUNE_CACHE, and
    a second run of the same size class (which takes the cached shape) does
    too."""
    syss = [systems.argon(ncells=6, seed=15), systems.nacl(ncells=5, kvec=(32, 32, 32), seed=16),
            systems.nacl(ncells=6, kvec=(40, 40, 40), seed=17)]
    print("case tuned ensemble of", [s.natms for s in syss], "precision", precision, flush=True)
    steps = 48
    cache = tmp_path / "tune.txt"
    monkeypatch.setenv("DLPX_AUTOTUNE", "1")
    monkeypatch.setenv("DLPX_TUNE_CACHE", str(cache))
    ref = []
    for s in syss:
        ctx = lib.Context(s, precision=precision)
        ctx.md_load(s.pos, s.vel)
        _, nreb = ctx.md_run(steps, s.timestep, energies=False)
        ref.append(ctx.md_store() + (nreb,))
        ctx.close()
    for run in range(2):
        ctxs = []
        for s in syss:
            ctx = lib.Context(s, precision=precision)
            ctx.md_load(s.pos, s.vel)
            ctxs.append(ctx)
        nreb = lib.md_run_ensemble(ctxs, steps)
        for k, (s, ctx) in enumerate(zip(syss, ctxs)):
            x, v, f = ctx.md_store()
            xr, vr, fr, nr = ref[k]
            L = np.diag(s.cell.reshape(3, 3))
            dx = x - xr
            dx -= L * np.round(dx / L)
            assert nreb[k] == nr
            assert np.abs(dx).max() <= tol * L.max()
            assert rms_rel(v, vr) <= tol and rms_rel(f, fr) <= 10 * tol
            ctx.close()
        lines = cache.read_text().split("\n")
        tuned = [ln.split() for ln in lines if ln.strip()]
        assert tuned and all(len(w) == 3 for w in tuned)
        assert any(int(w[1]) in (4, 8, 16) and int(w[2]) in (8, 16) for w in tuned)


def _ensemble_sample(syss, n=32):
    """Indices of n systems of the ensemble: the smallest and largest of each
    kind, one per NaCl mesh edge, the rest spread evenly over each kind."""
    pick = []
    for kind in (False, True):
        idx = [k for k, s in enumerate(syss) if bool(s.electrostatics) == kind]
        idx.sort(key=lambda k: syss[k].natms)
        want = [idx[0], idx[-1]]
        if kind:
            for K in sorted(set(syss[k].kvec[0] for k in idx)):
                want.append(next(k for k in idx if syss[k].kvec[0] == K))
        for k in np.linspace(0, len(idx) - 1, n // 2).astype(int):
            if len(set(want)) >= n // 2:
                break
            want.append(idx[k])
        pick += list(dict.fromkeys(want))[: n // 2]
    return pick


def test_ensemble256_sampled_systems_match_oracle():
    """The 256-system batched ensemble (systems.ensemble_systems(), seed
    20261202: half argon, half NaCl with meshes 40-64 including the odd 45),
    stepped as one batch: after a few resident steps, the forces and the last
    step's energies of 32 sampled systems against the oracle at the positions
    reached.  FP64 forces <= 1e-10 RMS relative, energies <= 1e-11 of their
    largest term; mixed forces <= 1e-5, energies <= 1e-6."""
    import concurrent.futures as cf
    syss = systems.ensemble_systems()
    pick = _ensemble_sample(syss)
    assert len(pick) == 32
    steps = 4
    for precision, tf, te in ((lib.FP64, 1e-10, 1e-11), (lib.MIXED, 1e-5, 1e-6)):
        print("case ensemble256 precision", precision, flush=True)
        ctxs = []
        for s in syss:
            ctx = lib.Context(s, precision=precision)
            ctx.md_load(s.pos, s.vel)
            ctxs.append(ctx)
        nreb, e = lib.md_run_ensemble(ctxs, steps, energies=True)
        states = {k: ctxs[k].md_store() for k in pick}
        for c in ctxs:
            c.close()
        with cf.ThreadPoolExecutor(8) as ex:
            orc = dict(zip(pick, ex.map(lambda k: oracle.two_body(syss[k], pos=states[k][0]), pick)))
        for k in pick:
            x, v, f = states[k]
            o = orc[k]
            err = rms_rel(f, o["frc"])
            assert err <= tf, (k, syss[k].natms, err)
            last = dict(zip(("engcpe", "vircpe", "engsrp", "virsrp"), e[k, -1, :4]))
            check_energies(last, o, te, energy_scales(o, mixed=precision == lib.MIXED))


def test_nve_energy_conservation_fp64_and_mixed():
    s = systems.nacl(ncells=8, kvec=(48, 48, 48), seed=3)
    for prec, tol in ((lib.FP64, 2e-5), (lib.MIXED, 5e-5)):
        ctx = lib.Context(s, precision=prec)
        ctx.md_load(s.pos, s.vel)
        e, nreb = ctx.md_run(200, s.timestep)
        etot = e[:, 0] + e[:, 2] + e[:, 4]
        # total energy fluctuates at the 1e-5 level and does not drift
        assert np.abs(etot - etot[0]).max() <= tol * abs(etot[0])
        assert nreb > 0
        ctx.close()


def _fortran_demo_system():
    """The configuration dl-poly_amd/fortran/dlpx_host_demo.F90 builds, with the
    same arithmetic in the same order."""
    nc = 5
    a = 5.64 * 1.08
    L = nc * a
    basis = [(0.0, 0.0, 0.0), (0.0, 0.5, 0.5), (0.5, 0.0, 0.5), (0.5, 0.5, 0.0)]
    pos = []
    for sp in (1, 2):
        for ix in range(nc):
            for iy in range(nc):
                for iz in range(nc):
                    for b in basis:
                        x = a * (ix + b[0]) - 0.5 * L
                        y = a * (iy + b[1]) - 0.5 * L
                        z = a * (iz + b[2]) - 0.5 * L
                        if sp == 2:
                            x = x + 0.5 * a
                        if x >= 0.5 * L:
                            x = x - L
                        pos.append([x, y, z])
    pos = np.array(pos)
    for n in range(1, len(pos) + 1):
        for d in range(1, 4):
            pos[n - 1, d - 1] += 0.1 * (((37 * n + 11 * d) % 101) / 100.0 - 0.5)
    s = systems.nacl(ncells=5, kvec=(32, 32, 32))
    s.pos = pos
    return s


@pytest.mark.parametrize("precision", [0, 1])
def test_fortran_host_through_iso_c_binding(tmp_path, precision):
    import os
    import subprocess
    exe = os.path.join(fixtures.ROOT, "dl-poly_amd", "fortran", "dlpx_host_demo")
    out = tmp_path / "demo.bin"
    r = subprocess.run([exe, str(precision), str(out)], capture_output=True, text=True, timeout=120)
    print(r.stdout, r.stderr)
    assert r.returncode == 0
    raw = np.fromfile(out, dtype="<f8")
    s = _fortran_demo_system()
    n = s.natms
    eng, stress, buf = raw[:4], raw[4:13], raw[13:33]
    frc = raw[33:33 + 3 * n].reshape(-1, 3)
    md_x, md_v, md_f = (raw[33 + 3 * n * (k + 1):33 + 3 * n * (k + 2)].reshape(-1, 3) for k in range(3))
    ctx, py = gpu_two_body(s, precision=precision)
    # same inputs through two hosts; the only difference is the order of the
    # atomic adds of charge spreading (FP64: ~1e-16, FP32 mixed grid: ~1e-7)
    tol = 1e-12 if precision == 0 else 2e-6
    assert np.abs(frc - py["frc"]).max() <= tol * np.abs(py["frc"]).max()
    assert np.allclose(eng, [py["engcpe"], py["vircpe"], py["engsrp"], py["virsrp"]], rtol=tol)
    assert np.abs(stress - py["stress"]).max() <= tol * np.abs(py["stress"]).max()
    assert np.abs(buf - py["buffer"]).max() <= tol * np.abs(py["buffer"]).max()
    if precision == 0:
        o = oracle.two_body(s)
        assert rms_rel(frc, o["frc"]) <= 1e-10
    ctx.close()
    # the resident steps, with velocities and masses passed in their own arrays
    vel = np.zeros((n, 3))
    for i in range(1, n + 1):
        for d in range(3):
            vel[i - 1, d] = 0.02 * (((53 * i + 7 * (d + 1)) % 97) / 96.0 - 0.5)
    ctx = lib.Context(s, precision=precision)
    ctx.md_load(s.pos, vel)
    ctx.md_run(10, 0.002, energies=False)
    x, v, f = ctx.md_store()
    ctx.close()
    L = np.diag(s.cell.reshape(3, 3))
    dx = md_x - x
    dx -= L * np.round(dx / L)
    tol_md = 1e-10 if precision == 0 else 1e-5
    assert np.abs(dx).max() <= tol_md * L.max()
    assert rms_rel(md_v, v) <= tol_md and rms_rel(md_f, f) <= 10 * tol_md


# mesh, spline order: meshes of whole and partial tiles (16 x 8 x 16 points),
# the smallest that hold a tile and its reach, two link cells per axis (bins
# are link cells) and more (subcells), every spline order
@pytest.mark.parametrize("ncells,kvec,order", [((5, 5, 5), (32, 32, 32), 8), ((5, 6, 7), (27, 30, 24), 4),
                                               ((7, 8, 9), (45, 50, 54), 6), ((7, 7, 7), (36, 40, 48), 10),
                                               ((8, 7, 6), (48, 36, 40), 12), ((6, 6, 6), (40, 36, 45), 14),
                                               ((7, 7, 8), (50, 48, 40), 16)])
def test_tile_and_cell_spreading_agree(ncells, kvec, order, monkeypatch):
    """The spreading by mesh tiles, which a list's second evaluation takes, and
    by link cells (DLPX_SPREAD_TILES=0): on the list's own positions, on
    moved ones, on ones moved further than the tiles' lists allow for (every
    atom by up to 3 A without a rebuild) and in a cell scaled by half a
    percent since the build; and in resident steps across rebuilds.  Both add
    the same products in FP64: 1e-12 apart at most in FP64.  Mixed results, of
    either spreading, are held to the mode's own bar (forces 1e-5 RMS, energies
    1e-6) against FP64's."""
    s = systems.nacl(ncells=ncells, kvec=kvec, nsplines=order, seed=11)
    rng = np.random.default_rng(12)
    near = s.pos + rng.uniform(-0.14, 0.14, s.pos.shape)
    far = s.pos + rng.uniform(-3.0, 3.0, s.pos.shape)
    ref = None
    for precision, tol, etol in ((lib.FP64, 1e-12, 1e-12), (lib.MIXED, 1e-5, 1e-6)):
        for tiles in ("0", "1"):
            monkeypatch.setenv("DLPX_SPREAD_TILES", tiles)
            ctx = lib.Context(s, precision=precision)
            ctx.link_cell_pairs(s.pos)
            got = [ctx.two_body_forces(p) for p in (s.pos, s.pos, near, far, near)]
            ctx.cell = ctx.cell * 1.005
            got += [ctx.two_body_forces(p) for p in (near * 1.005, far)]
            ctx.cell = ctx.cell / 1.005
            ctx.link_cell_pairs(near)
            got += [ctx.two_body_forces(near), ctx.two_body_forces(s.pos)]
            ctx.md_load(s.pos, s.vel)
            ctx.md_run(12, s.timestep)
            got.append(dict(frc=ctx.md_store()[2], engcpe=ctx.md_last_output()["engcpe"]))
            ctx.close()
            ref = ref or got  # FP64 by link cells
            for k, (a, b) in enumerate(zip(got, ref)):
                # 12 steps let the differences of the first grow tenfold at most
                f = 10.0 if k == len(ref) - 1 else 1.0
                print("case", ncells, order, precision, tiles, k, rms_rel(a["frc"], b["frc"]), flush=True)
                assert rms_rel(a["frc"], b["frc"]) <= f * tol, (precision, k)
                assert abs(a["engcpe"] - b["engcpe"]) <= f * etol * abs(b["engcpe"]), (precision, k)


def test_tile_lists_longer_than_their_room(monkeypatch):
    """A droplet: all the ions of one corner of the box, so that a tile's list
    outgrows its room (sized by the mean density) and the tile adds it in
    several rounds.  Against the spreading by link cells, FP64 to rounding."""
    s = systems.nacl(ncells=10, kvec=(64, 64, 64), seed=13)
    s.pos = s.pos * 0.35 - 0.3 * s.cell[0]
    s.cutoff = s.vdw_cutoff = 6.0
    got = {}
    for tiles in ("1", "0"):
        monkeypatch.setenv("DLPX_SPREAD_TILES", tiles)
        ctx = lib.Context(s, precision=lib.FP64)
        ctx.link_cell_pairs(s.pos)
        got[tiles] = [ctx.two_body_forces(s.pos) for _ in range(3)]
        ctx.close()
    for a, b in zip(got["1"], got["0"]):
        # the close ions' real-space forces dominate; the reciprocal energy shows the spreading
        assert rms_rel(a["frc"], b["frc"]) <= 1e-12
        assert abs(a["buffer"][9] - b["buffer"][9]) <= 1e-12 * abs(b["buffer"][9])


# atom counts on both sides of the lines between the launch shapes (4,096 and
# 8,192 atoms), a lone pair of atoms and an odd count
@pytest.mark.parametrize("kind,size", [("argon", 2), ("argon", 777), ("argon", 4096), ("argon", 4097),
                                       ("argon", 8192), ("argon", 8193), ("nacl", (5, 5, 5)), ("nacl", (8, 8, 8)),
                                       ("nacl", (8, 8, 9)), ("nacl", (8, 8, 16)), ("nacl", (8, 8, 17))])
def test_pair_launch_shapes_agree(kind, size, monkeypatch):
    """The pair kernels' default launch shape and four lanes to an atom
    (DLPX_PAIR_LANES=4): the same pairs with the same arithmetic, summed in
    another order.  FP64 to 1e-12; mixed results of either shape to the mode's
    bar (forces 1e-5 RMS, energies 1e-6) against FP64's."""
    if kind == "argon":
        s = systems.argon(ncells=13, jitter=0.2)
        s.pos, s.vel, s.types = s.pos[:size].copy(), s.vel[:size].copy(), s.types[:size].copy()
    else:
        s = systems.nacl(ncells=size, kvec=(32, 32, 32), seed=14)
    ref = None
    for precision, tol, etol in ((lib.FP64, 1e-12, 1e-12), (lib.MIXED, 1e-5, 1e-6)):
        for lanes in ("4", None):
            if lanes:
                monkeypatch.setenv("DLPX_PAIR_LANES", lanes)
            else:
                monkeypatch.delenv("DLPX_PAIR_LANES", raising=False)
            ctx = lib.Context(s, precision=precision)
            ctx.link_cell_pairs(s.pos)
            r = ctx.two_body_forces(s.pos)
            ctx.close()
            ref = ref or r
            print("case", kind, size, precision, lanes, rms_rel(r["frc"], ref["frc"]), flush=True)
            assert rms_rel(r["frc"], ref["frc"]) <= tol
            assert abs(r["engsrp"] - ref["engsrp"]) <= etol * abs(ref["engsrp"])


@pytest.mark.parametrize("size", [(8, 8, 8), (8, 8, 16), (8, 8, 17)])
@pytest.mark.parametrize("direct", [False, True])
def test_per_particle_and_direct_launch_shapes_agree(size, direct):
    """Per-particle output and analytic vdW forms on both sides of the line
    between 32 and 8 lanes to an atom (8,192 atoms): per-particle evaluations
    give the plain ones' forces (another kernel with the same arithmetic, 1e-12),
    analytic forms the tables' (the tables' interpolation error, below 1e-5),
    and each atom's energies and stresses add up the same with the atoms taken
    in reverse order (1e-12 of the largest)."""
    s = systems.nacl(ncells=size, kvec=(32, 32, 32), seed=15)
    rev = systems.nacl(ncells=size, kvec=(32, 32, 32), seed=15)
    for k in ("pos", "vel", "types"):
        setattr(rev, k, getattr(s, k)[::-1].copy())
    got = {}
    for name, sys_, pp in (("plain", s, False), ("pp", s, True), ("rev", rev, True)):
        sys_.vdw_direct = direct
        ctx = lib.Context(sys_, precision=lib.FP64)
        ctx.link_cell_pairs(sys_.pos)
        got[name] = ctx.two_body_forces(sys_.pos, per_particle=pp)
        ctx.close()
    s.vdw_direct = False
    ctx = lib.Context(s, precision=lib.FP64)
    ctx.link_cell_pairs(s.pos)
    tables = ctx.two_body_forces(s.pos)
    ctx.close()
    a, b = got["pp"], got["rev"]
    print("case", size, direct, rms_rel(a["frc"], got["plain"]["frc"]), flush=True)
    assert rms_rel(a["frc"], got["plain"]["frc"]) <= 1e-12
    assert rms_rel(a["frc"], tables["frc"]) <= 1e-5
    assert rms_rel(b["frc"][::-1], a["frc"]) <= 1e-12
    st = np.abs(a["pp_stress"]).max()
    assert np.abs(b["pp_stress"][::-1] - a["pp_stress"]).max() <= 1e-12 * st


@pytest.mark.parametrize("n", [135, 144, 150, 160, 162, 180, 192, 200, 216, 225, 240, 256, 270, 288, 300, 320, 324, 360])
def test_long_line_transforms_agree(n, monkeypatch):
    """Meshes with an axis beyond 128 points: the line kernels and the generic
    ones (DLPX_FFT_LINES=0) along x, y and z, the other axes shorter and of odd
    line counts.  The same transform in another order of factors: FP64 forces,
    energy and stress to 1e-12, mixed ones to the mode's bar (forces 1e-5 RMS,
    energies 1e-6) against FP64's.  One call on host arrays and two resident steps
    (the batched kernels)."""
    for kvec in ((n, 27, 25), (25, n, 27), (30, 25, n)):
        s = systems.nacl(ncells=5, kvec=kvec, seed=17)
        ref = None
        for precision, tol, etol in ((lib.FP64, 1e-12, 1e-12), (lib.MIXED, 1e-5, 1e-6)):
            for lines in ("0", "1"):
                monkeypatch.setenv("DLPX_FFT_LINES", lines)
                ctx = lib.Context(s, precision=precision)
                ctx.link_cell_pairs(s.pos)
                r = ctx.two_body_forces(s.pos)
                ctx.md_load(s.pos, s.vel)
                ctx.md_run(3, s.timestep)
                md = ctx.md_store()[2]
                ctx.close()
                ref = ref or (r, md)
                print("case", kvec, precision, lines, rms_rel(r["frc"], ref[0]["frc"]), flush=True)
                assert rms_rel(r["frc"], ref[0]["frc"]) <= tol
                assert rms_rel(md, ref[1]) <= 10.0 * tol
                assert abs(r["engcpe"] - ref[0]["engcpe"]) <= etol * abs(ref[0]["engcpe"])
                assert np.abs(r["stress"] - ref[0]["stress"]).max() <= max(tol, etol) * np.abs(ref[0]["stress"]).max()


@pytest.mark.parametrize("lanes", ["4", "16", None])
def test_pair_workgroups_of_512_threads(lanes, monkeypatch):
    """DLPX_COMB_THREADS=512 has one shape, 8 lanes to an atom, whatever the
    lanes asked for: every atom is served (mixed against FP64, 1e-5 RMS)."""
    s = systems.nacl(ncells=6, kvec=(32, 32, 32), seed=18)
    monkeypatch.setenv("DLPX_COMB_THREADS", "512")
    if lanes:
        monkeypatch.setenv("DLPX_PAIR_LANES", lanes)
    frc = []
    for precision in (lib.FP64, lib.MIXED):
        ctx = lib.Context(s, precision=precision)
        ctx.link_cell_pairs(s.pos)
        frc.append(ctx.two_body_forces(s.pos)["frc"])
        ctx.close()
    assert rms_rel(frc[1], frc[0]) <= 1e-5


@pytest.mark.parametrize("size", [(5, 5, 5), (8, 8, 17)])
def test_coulomb_only_system_matches_oracle(size):
    """Ions without any vdW interaction: no vdW table rows, so the pair kernel
    has none to load, in both of its launch shapes (32 and 8 lanes to an atom),
    with and without per-particle output and force-shifting (which keeps mixed
    precision off the combined tables).  FP64 to 1e-10 of the oracle, mixed to
    1e-5."""
    s = systems.nacl(ncells=size, kvec=(32, 32, 32), seed=21)
    s.vdw = []
    # per-particle output takes the reciprocal virial from the atoms' stresses, in the oracle too
    oracles = {pp: oracle.two_body(s, per_particle=pp) for pp in (False, True)}
    for precision, tol, etol in ((lib.FP64, 1e-10, 1e-11), (lib.MIXED, 1e-5, 1e-6)):
        for pp, shift in ((False, False), (True, False), (False, True)):
            print("case coulomb only", s.natms, precision, pp, shift, flush=True)
            s.vdw_force_shift = shift
            o = oracles[pp]
            ctx = lib.Context(s, precision=precision)
            ctx.link_cell_pairs(s.pos)
            r = ctx.two_body_forces(s.pos, per_particle=pp)
            ctx.close()
            assert rms_rel(r["frc"], o["frc"]) <= tol
            assert r["engsrp"] == 0.0
            sc = energy_scales(o, precision == lib.MIXED)
            for k in ("engcpe", "vircpe"):
                assert abs(r[k] - o[k]) <= etol * max(abs(o[k]), sc[k]), k
            if pp:
                assert rms_rel(r["pp_energy"], o["pp_energy"]) <= tol
                assert rms_rel(r["pp_stress"], o["pp_stress"]) <= tol


@pytest.mark.parametrize("precision,tol", [(lib.FP64, 1e-12), (lib.MIXED, 1e-6)])
@pytest.mark.parametrize("ncells,kvec", [((5, 5, 5), (32, 32, 32)), ((7, 8, 9), (45, 50, 54))])
def test_one_atom_moved_within_its_bin(ncells, kvec, precision, tol, monkeypatch):
    """A trial move without a rebuild: one atom 1, 2 and 3 A along an axis, every
    other at its place in the list, so that the atom stays in the bin of the
    list build (it starts in the lowest quarter of a subcell, and one of two
    link cells is longer still) but reaches mesh tiles that did not list it.
    The reciprocal energy and forces of a list's second and later evaluations,
    which spread by tiles, are those by link cells: to 1e-12 in FP64, to the
    FP32 grid's rounding mixed."""
    s = systems.nacl(ncells=ncells, kvec=kvec, seed=23)
    s.vdw = []  # an ion moved onto another adds no vdW force that hides the mesh's
    L = np.diag(s.cell.reshape(3, 3))
    nc = np.floor(L / (s.cutoff + s.padding + 1e-6))
    frac = ((s.pos / L + 0.5) * 2 * nc) % 1.0
    movers = np.flatnonzero((frac < 0.25).all(1))[:12]
    assert len(movers) >= 6
    got = {}
    for tiles in ("0", "1"):
        monkeypatch.setenv("DLPX_SPREAD_TILES", tiles)
        ctx = lib.Context(s, precision=precision)
        ctx.link_cell_pairs(s.pos)
        ctx.two_body_forces(s.pos)
        got[tiles] = []
        for i in movers:
            for d in range(3):
                for step in (1.0, 2.0, 3.0):
                    p = s.pos.copy()
                    p[i, d] += step
                    r = ctx.two_body_forces(p)
                    got[tiles].append((r["buffer"][9], r["frc"]))
        got[tiles].append((ctx.two_body_forces(s.pos)["buffer"][9], None))  # and back
        ctx.close()
    for k, (a, b) in enumerate(zip(got["1"], got["0"])):
        print("case moved", ncells, precision, k, a[0] / b[0] - 1.0, flush=True)
        assert abs(a[0] - b[0]) <= tol * abs(b[0])
        if a[1] is not None:
            assert rms_rel(a[1], b[1]) <= tol


@pytest.mark.parametrize("precision,tol", [(lib.FP64, 1e-9), (lib.MIXED, 1e-5)])
@pytest.mark.parametrize("graphs,scale", [("0", 1.03), ("1", 1.03), ("1", 1.007)])
def test_run_in_another_cell_than_the_list(graphs, scale, precision, tol, monkeypatch):
    """dlpx_md_load, a force call in a cell 0.7 or 3 % longer (the latter five
    link cells to an axis instead of four) and a run there: the run and its
    per-step energies are those of the configuration loaded in that cell, and
    force calls after it, on positions with one atom moved, spread by tiles as
    by link cells."""
    monkeypatch.setenv("DLPX_GRAPHS", graphs)
    s = systems.nacl(ncells=10, kvec=(64, 64, 64), seed=24)
    pos = s.pos * scale
    steps, got = 12, {}
    for name, tiles in (("there", "0"), ("there", "1"), ("loaded", "0")):
        monkeypatch.setenv("DLPX_SPREAD_TILES", tiles)
        ctx = lib.Context(s, precision=precision)
        if name == "there":
            ctx.md_load(s.pos, s.vel)
            ctx.cell = ctx.cell * scale
            ctx.two_body_forces(pos)
        else:
            ctx.cell = ctx.cell * scale
            ctx.md_load(pos, s.vel)
        e, reb = ctx.md_run(steps, s.timestep)
        assert reb > 0
        x, _, f = ctx.md_store()
        after = []
        for i in range(0, s.natms, 401):
            for d in range(3):
                p = x.copy()
                p[i, d] += 2.0
                after.append(ctx.two_body_forces(p)["buffer"][9])
        ctx.close()
        got[name, tiles] = (f, e, np.array(after))
    ref = got["loaded", "0"]
    for k in (("there", "0"), ("there", "1")):
        f, e, after = got[k]
        print("case cell", graphs, scale, precision, k, rms_rel(f, ref[0]), flush=True)
        assert rms_rel(f, ref[0]) <= tol
        assert np.abs(e - ref[1]).max() <= tol * np.abs(ref[1]).max()
        assert np.abs(after - ref[2]).max() <= tol * np.abs(ref[2]).max()


@pytest.mark.parametrize("ncells,order,kvec", [(10, 4, (64, 64, 64)), (10, 8, (50, 45, 54)), (10, 16, (64, 45, 54)),
                                               (15, 4, (50, 45, 54)), (15, 8, (96, 90, 100)), (15, 16, (64, 45, 54))])
def test_moved_atoms_beyond_a_tiles_room(ncells, order, kvec, monkeypatch):
    """Positions further from the list's than the tiles' lists allow for, with
    8,000 ions (every tile tests every atom) and 27,000 (lists from where the
    atoms are), at meshes of whole and partial tiles.  A droplet, whose tiles hold more atoms than
    their room, and the same ions over the whole box, most of them charged and
    one in seven not.  FP64 against the spreading by link cells, to rounding."""
    s = systems.nacl(ncells=ncells, kvec=kvec, nsplines=order, seed=25)
    s.cutoff = s.vdw_cutoff = 6.0
    s.vdw = []
    rng = np.random.default_rng(26)
    wide = s.pos + rng.uniform(-2.0, 2.0, s.pos.shape)
    drop = s.pos * 0.4 - 0.25 * s.cell[0]
    far = drop + rng.uniform(-2.0, 2.0, s.pos.shape)
    got = {}
    for tiles in ("1", "0"):
        monkeypatch.setenv("DLPX_SPREAD_TILES", tiles)
        ctx = lib.Context(s, precision=lib.FP64)
        ctx.q = np.where(np.arange(s.natms) % 7 == 0, 0.0, ctx.q)
        got[tiles] = []
        for at, to in ((s.pos, wide), (drop, far)):
            ctx.link_cell_pairs(at)
            got[tiles] += [ctx.two_body_forces(p) for p in (at, to, at, to)]
        ctx.close()
    for k, (a, b) in enumerate(zip(got["1"], got["0"])):
        print("case strays", ncells, order, kvec, k, a["buffer"][9] / b["buffer"][9] - 1.0, flush=True)
        assert rms_rel(a["frc"], b["frc"]) <= 1e-12
        assert abs(a["buffer"][9] - b["buffer"][9]) <= 1e-12 * abs(b["buffer"][9])


@pytest.mark.parametrize("edge,subcells", [(26.0, "1"), (40.0, "1"), (40.0, "0")])
def test_pair_set_in_a_long_cell(edge, subcells, monkeypatch):
    """A cell of edge x edge x 6,000 A (two and four link cells on the short
    axes, 631 on the long one), where FP32 coordinates are 2e-4 A apart: atoms
    in pairs whose distances lie within 1.2e-4 of the cutoff with padding,
    relative, in any direction and across every face.  The pair set is the one
    of FP64 distances."""
    monkeypatch.setenv("DLPX_LIST_SUBCELLS", subcells)
    rng = np.random.default_rng(27)
    L = np.array([edge, edge, 6000.0])
    n, rc = 3000, 9.5
    base = rng.uniform(-0.5, 0.5, (n, 3)) * L
    base[: n // 3, 2] = np.sign(base[: n // 3, 2]) * (3000.0 - rng.uniform(0.0, 6.0, n // 3))  # at the long axis's faces
    u = rng.normal(size=(n, 3)) * (0.3, 0.3, 1.0)
    u /= np.linalg.norm(u, axis=1)[:, None]
    other = base + u * (rc * (1.0 + rng.uniform(-1.2e-4, 1.2e-4, n)))[:, None]
    s = systems.argon(ncells=10)
    s.pos = np.stack([base, other], 1).reshape(-1, 3)
    s.pos = s.pos - L * np.floor(s.pos / L + 0.5)
    s.vel, s.types = np.zeros_like(s.pos), np.zeros(2 * n, np.int32)
    s.cell = np.diag(L).reshape(9)
    s.cutoff = s.vdw_cutoff = rc - s.padding
    ctx = lib.Context(s, precision=lib.FP64)
    ctx.link_cell_pairs(s.pos)
    got = {tuple(p[:2]) for p in ctx.get_pairs()}
    ctx.close()
    want = {tuple(p[:2]) for p in oracle.pairs(s.cell, s.pos, rc, "brute")}
    print("case long cell", edge, subcells, len(got), len(want), len(got ^ want), flush=True)
    assert not got ^ want


def test_memory_of_the_splines_only_for_tiles(monkeypatch):
    """A context that spreads by link cells holds no splines of its atoms (3 S
    + 4 reals and 8 bytes an atom): device memory in use after a list build,
    by tiles and by cells."""
    import ctypes
    hip = ctypes.CDLL("libamdhip64.so")

    def free():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    s = systems.nacl(ncells=30, kvec=(128, 128, 128), seed=28)
    used = {}
    for tiles in ("0", "1", "0", "1"):  # the first two load the kernels
        monkeypatch.setenv("DLPX_SPREAD_TILES", tiles)
        before = free()
        ctx = lib.Context(s, precision=lib.FP64)
        ctx.link_cell_pairs(s.pos)
        for _ in range(3):
            ctx.two_body_forces(s.pos)
        used[tiles] = before - free()
        ctx.close()
    splines = s.natms * (8 * (3 * 8 + 4) + 8)
    print("case memory", s.natms, used, splines, flush=True)
    assert used["1"] - used["0"] >= splines


def test_calls_after_a_failed_one_match_fresh_ones():
    """List builds and loads that fail after they have queued their upload (a
    cell too small for the cutoff), each at once followed by a good one with
    other positions: the pinned rows are not written while the load still reads
    them, and forces are a fresh context's."""
    s = systems.nacl(ncells=20, kvec=(64, 64, 64), seed=29)
    rng = np.random.default_rng(30)
    ctx, fresh = lib.Context(s), lib.Context(s)
    cell = ctx.cell.copy()
    for k in range(4):
        p = s.pos + rng.uniform(-0.1, 0.1, s.pos.shape)
        for load in (False, True):
            ctx.cell = cell * 0.1
            with pytest.raises(lib.DlpxError) as e:
                ctx.md_load(s.pos, s.vel) if load else ctx.link_cell_pairs(s.pos)
            assert e.value.code == 95
            ctx.cell = cell.copy()
            ctx.link_cell_pairs(p)
            fresh.link_cell_pairs(p)
            a, b = ctx.two_body_forces(p), fresh.two_body_forces(p)
            assert rms_rel(a["frc"], b["frc"]) <= 1e-13
            assert a["engcpe"] == pytest.approx(b["engcpe"], rel=1e-13)
    ctx.close()
    fresh.close()


@pytest.mark.parametrize("graphs", ["0", "1"])
def test_run_from_a_force_call_on_moved_positions(graphs, monkeypatch):
    """A force call with one atom just beyond half the padding, then a run whose
    first drift brings it back, so that nothing is rebuilt: the tiles' lists, not
    those of the force call, with 27,000 ions (whose force call puts atoms on
    lists where they are).  Against link cells, FP64 to rounding."""
    monkeypatch.setenv("DLPX_GRAPHS", graphs)
    s = systems.nacl(ncells=15, kvec=(96, 96, 96), seed=31, temperature=1.0)
    p, v = s.pos.copy(), s.vel.copy()
    p[11, 0] += 0.5 * s.padding + 0.01
    v[11] = (-20.0, 0.0, 0.0)
    got = {}
    for tiles in ("0", "1"):
        monkeypatch.setenv("DLPX_SPREAD_TILES", tiles)
        ctx = lib.Context(s, precision=lib.FP64)
        ctx.md_load(s.pos, v)
        ctx.two_body_forces(p)
        e, reb = ctx.md_run(3, s.timestep)
        got[tiles] = (e, reb, ctx.md_store()[2])
        ctx.close()
    (e1, r1, f1), (e0, r0, f0) = got["1"], got["0"]
    assert r1 == r0 == 0
    assert np.abs(e1 - e0).max() <= 1e-11 * np.abs(e0).max()
    assert rms_rel(f1, f0) <= 1e-10


@pytest.mark.parametrize("size", [(8, 8, 8), (8, 8, 17)])
def test_per_particle_energies_in_host_order(size):
    """Each atom's energy and stress on both sides of the line between 32 and 8
    lanes to an atom, with the atoms given forwards and in reverse (which moves
    the vdW energy of pairs across the cell's faces to their other atom), against
    the oracle: FP64 to 1e-10 of the largest, mixed to 1e-5 RMS."""
    for order in (1, -1):
        s = systems.nacl(ncells=size, kvec=(32, 32, 32), seed=32)
        for k in ("pos", "vel", "types"):
            setattr(s, k, getattr(s, k)[::order].copy())
        o = oracle.two_body(s, per_particle=True)
        for precision in (lib.FP64, lib.MIXED):
            ctx = lib.Context(s, precision=precision)
            ctx.link_cell_pairs(s.pos)
            r = ctx.two_body_forces(s.pos, per_particle=True)
            ctx.close()
            for k in ("pp_energy", "pp_stress"):
                print("case per particle", s.natms, order, precision, k, rms_rel(r[k], o[k]), flush=True)
                if precision == lib.FP64:
                    assert np.abs(r[k] - o[k]).max() <= 1e-10 * np.abs(o[k]).max()
                else:
                    assert rms_rel(r[k], o[k]) <= 1e-5
