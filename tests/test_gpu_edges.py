"""Kernels at the sizes where their tiles and reductions end: one molecule more
or less than a block, the smallest and the largest of a range, against the
oracle.  Bars are those of the larger tests of the same paths."""
import numpy as np
import pytest

from swinmd_amd import _lib as L
from swinmd_amd import systems as S
from tests.helpers import rel, rel_rms

pytestmark = pytest.mark.gpu

RHO = 33.43


def _water_cfg(n):
    s = S.water(n, density_mol=RHO, seed=n, subset=True, jitter=0.01)
    half = 0.5 * s.box[0]
    cfg = dict(cutoff=min(0.6, 0.8 * half), cut_buff=0.02, alpha=3.5, kcut=S.kcut_for(27, s.box[0]), dt=0.002,
               temperature=300.0, coupl=0.1, use_cells=half > 0.93)
    return s, cfg


@pytest.mark.parametrize("n", [1, 21, 63, 64, 65, 129, 216])
def test_rigid_water_step_sizes_match_the_oracle(n):
    """Blocks of the SHAKE and kinetics kernel hold 64 molecules: 8 steps with
    list rebuilds, FP64; positions 1e-10, velocities and energies 1e-8."""
    from oracle import oracle as O
    from swinmd_amd.forces import Context, WaterMD
    s, cfg = _water_cfg(n)
    o = O.Oracle(s)
    vel = o.init_velocity(300.0, 3, per_atom=False, ndf=max(3 * n - 3, 3)) if n > 1 else np.full((3, 3), 0.1)
    ref = O.md_from_cfg(o, cfg, 8, velocity=vel)
    print(f"case water n={n} list updates {ref['list_updates']}", flush=True)
    ctx = Context(s)
    ctx.set_velocities(vel)
    md = WaterMD(ctx, **{k: cfg[k] for k in ("cutoff", "cut_buff", "alpha", "kcut", "dt", "temperature", "coupl",
                                             "use_cells")})
    md.init()
    rep = md.run(3)
    rep = md.run(5)
    assert rep["list_updates"] == ref["list_updates"]
    assert rel_rms(ctx.positions(), ref["pos"]) <= 1e-10
    assert rel_rms(ctx.velocities(), ref["vel"]) <= 1e-8
    for k in ("e_real", "e_long", "e_intra", "atom_ke2"):
        if ref[k]:
            assert rel(rep[k], ref[k]) <= 1e-8, k


class _BoxedWater(S.System):
    """A water system in a box of given edges (System's own is a cube)."""
    edges = None

    @property
    def box(self):
        return np.array(self.edges, dtype=np.float64)


# molecules, edges, k cut as a count of the longest edge's waves: one k-row and
# function, rows past a 16-row tile, atoms past a 64-atom table, more than 16
# and more than 32 functions of nz, tables at their narrow stride
@pytest.mark.parametrize("n,edges,waves", [(1, (1.2, 1.2, 1.2), 1.2), (21, (1.4, 1.4, 1.4), 5.2),
                                           (22, (1.4, 1.4, 1.4), 5.2), (64, (1.3, 1.5, 1.7), 11.2),
                                           (85, (1.5, 1.5, 7.5), 20.3), (43, (1.0, 1.0, 12.0), 49.5)])
@pytest.mark.parametrize("mixed", [False, True])
def test_reciprocal_space_shapes_match_the_oracle(n, edges, waves, mixed):
    """Forces, energy, virial and volume derivatives of EwaldForce.compute_long:
    1e-10 in FP64, 1e-5 mixed (forces) as in the larger parity tests."""
    from oracle import oracle as O
    from swinmd_amd.forces import Context, EwaldForce
    s = S.water(n, box=min(edges), seed=n, subset=True, jitter=0.01)
    s.__class__ = _BoxedWater
    s.edges = edges
    s.pos = s.pos * (np.array(edges) / min(edges)) if n > 40 else s.pos
    kcut = 2 * np.pi * waves / max(edges)
    print(f"case recip n={n} edges={edges} waves={waves} mixed={mixed}", flush=True)
    ctx = Context(s)
    ctx.compute_mol_centers()
    ew = EwaldForce(ctx, alpha=3.5, real_cut=0.5, kcut=kcut, prec=L.PREC_MIXED if mixed else L.PREC_FP64)
    f = np.zeros((s.n_atoms, 3))
    out = ew.compute_long(f)
    fo, eo = O.Oracle(s).ewald_recip(kcut, 3.5)
    tol = 1e-5 if mixed else 1e-10
    assert rel_rms(f, fo) <= tol
    for k in ("energy", "deriv", "deriv2"):
        assert abs(out[k] - eo[k]) <= tol * max(abs(eo[k]), abs(eo["energy"])), k
    assert rel_rms(out["virial"], eo["virial"]) <= tol


# cutoffs of one k-row and up, the last that the row passes' LDS takes (16
# waves along the edge), the direct passes past it, and two replicas whose
# rows differ in their number of functions
@pytest.mark.parametrize("n2", [(1,), (20, 81), (256,), (306,)])
def test_sheared_reciprocal_space_matches_the_oracle(n2):
    """Two steps at a tilt: forces and energies 1e-8, the same k count."""
    from oracle import oracle as O
    from swinmd_amd.nemd import ShearBatch
    systems = [S.water(n, density_mol=RHO, seed=n, subset=True) for n in (256, 275)[:len(n2)]]
    kcut = [S.kcut_for(k, s.box[0]) for k, s in zip(n2, systems)]
    gam, tilt = [3.0, -2.0][:len(n2)], [0.31, -0.2][:len(n2)]
    vels = [O.Oracle(s).init_velocity(300.0, 5, per_atom=False, ndf=3 * s.n_mols - 3) for s in systems]
    print(f"case shear n2={n2}", flush=True)
    b = ShearBatch(systems, gam, cutoff=0.8, cut_buff=0.08, alpha=3.5, kcut=kcut, dt=0.002, temperature=300.0,
                   coupl=0.1)
    b.set_state([s.pos for s in systems], vels, tilt)
    b.start()
    b.run(2)
    st, rep = b.state(), b.reports()
    for r, s in enumerate(systems):
        want = O.sllod_run(O.Oracle(s), dict(cutoff=0.8, cut_buff=0.08, alpha=3.5, kcut=kcut[r], dt=0.002,
                                             temperature=300.0, coupl=0.1), gam[r], 2, velocity=vels[r], tilt=tilt[r])
        assert rep[r]["n_kvec"] == want["K"]
        assert rel(rep[r]["e_long"], want["e_long"]) <= 1e-8
        assert rel_rms(b.split(st["force"])[r], want["force"]) <= 1e-8
        assert rel_rms(b.split(st["pos"])[r], want["pos"]) <= 1e-10
        assert np.max(np.abs(rep[r]["virial"] - want["virial"])) <= 1e-7 * np.max(np.abs(want["virial"]))


@pytest.mark.parametrize("n", [256, 512])
@pytest.mark.parametrize("prec", [L.PREC_FP64, L.PREC_MIXED])
def test_row_lanes_by_size_give_the_small_boxes_forces(n, prec):
    """Eight copies of a box are the same infinite lattice, so every copy's
    short-range forces, fields and induced dipoles are the small box's: 768
    and 1,536 sites run 64 lanes per atom row, their copies 32 (6,144 sites,
    the line itself) and 16 (12,288, the other line).  FP64 1e-10 (rounding of
    another order), mixed 1e-5 (the form's own bar)."""
    from swinmd_amd.forces import Context, EwaldForce, Induction, LJForce, Multipole
    print(f"case {n} waters and eight copies, prec {prec}", flush=True)
    base = S.water(n, density_mol=RHO, seed=5, subset=True, r_oh=0.09572, hoh_deg=108.5, types=S.AMOEBA_TYPES)
    big = S.water(8 * n, density_mol=RHO, seed=5, subset=True, r_oh=0.09572, hoh_deg=108.5, types=S.AMOEBA_TYPES)
    Lb = base.box[0]
    shifts = [(i - 0.5, j - 0.5, k - 0.5) for i in range(2) for j in range(2) for k in range(2)]
    big.pos = np.concatenate([base.pos + Lb * np.array(s) for s in shifts])
    solve_tol = 1e-12 if prec == L.PREC_FP64 else 1e-6
    out = []
    for s in (base, big):
        ctx = Context(s)
        ctx.compute_mol_centers()
        ctx.set_pairlist(0.7, 0.05, s is big)
        kcut = S.kcut_for(3, s.box[0])
        pc, mpf, indf = (np.zeros((s.n_atoms, 3)) for _ in range(3))
        LJForce(ctx, cutoff=0.7, prec=prec).compute(pc)
        EwaldForce(ctx, alpha=3.5, real_cut=0.7, kcut=kcut, prec=prec).compute(pc)
        mp = Multipole(ctx, alpha=3.5, real_cut=0.7, kcut=kcut, prec=prec)
        a = mp.compute(mpf)
        ind = Induction(ctx, cutoff_ind=0.7, a_damp=0.39, damp_tij=True, do_min=True, tol=solve_tol * L.DEBYE_E_NM,
                        precond=2, guess=2, prec=prec)
        ind.setup_terms(alpha=3.5, real_cut=0.7, kcut=kcut, prec=prec)
        ind.induce()
        b = ind.compute(indf)
        _, _, e0, mu = ind.results()
        out.append((pc, mpf, indf, e0, mu, np.array([a["real_energy"], b["real_energy"]])))
    tol = 1e-10 if prec == L.PREC_FP64 else 1e-5
    for name, x, y in zip(("pairs", "multipole", "induction", "e0", "mu"), out[0], out[1]):
        assert rel_rms(np.asarray(y).reshape(8, -1), np.tile(np.asarray(x).reshape(1, -1), (8, 1))) <= tol, name
    assert np.abs(out[1][5] / (8 * out[0][5]) - 1).max() <= tol


# one row, a row more than a 16-row tile and than a pair of tiles, a slice of
# one pair left over, and both sides of the line between 4 and 8 waves a block
@pytest.mark.parametrize("rows", [1, 17, 33, 2081, 16384, 16385])
def test_network_gradient_rows_match_the_oracle(rows):
    """Loss, gradients of every layer and outputs, oracle with BF16 products;
    the bars are those of the other batches."""
    from oracle import learned_guess as G
    from swinmd_amd.forces import Context, LearnedGuess
    print(f"case network gradient rows {rows}", flush=True)
    ctx = Context(S.water(27, density_mol=RHO, seed=2, types=S.AMOEBA_TYPES))
    net = LearnedGuess(ctx, seed=3)
    rng = np.random.default_rng(rows)
    p32 = G.init_params(7).astype(np.float32)
    p32[G.NPARAMS - 3:] = [0.3, -0.1, 0.2]
    net.set_params(p32)
    x = rng.normal(size=(rows, G.NF)).astype(np.float32)
    t = rng.normal(scale=0.5, size=(rows, G.NO)).astype(np.float32)
    loss, g = net.loss_grad(x, t)
    wl, wg = G.loss_grad(p32.astype(np.float64), x.astype(np.float64), t.astype(np.float64), emulate=True)
    assert abs(loss - wl) <= 1e-4 * wl
    assert rel_rms(g, wg) <= 2e-3
    offs = np.cumsum([0] + [int(np.prod(s)) for _, s in G.PUB_SHAPES])
    for b, (name, _) in enumerate(G.PUB_SHAPES):
        gb, wb = g[offs[b]:offs[b + 1]], wg[offs[b]:offs[b + 1]]
        assert rel_rms(gb, wb) <= 1e-2, name
    assert rel_rms(net.forward(x), G.forward(p32.astype(np.float64), x.astype(np.float64))[0]) <= 1e-3
    ctx.close()


@pytest.mark.parametrize("case", ["few", "uniform", "crowded", "outside"])
def test_cell_list_rows_match_the_oracle(case):
    """Rows of the cell-built list, in order, for few atoms a cell, for tiles
    with every remainder, for one cell beyond its share of the hit bits with
    rows too long for LDS, and for atoms more than 3/4 of a box away; with up
    to nine exclusions on an atom."""
    from oracle import oracle as O
    from swinmd_amd.forces import Context
    n = {"few": 40, "uniform": 3100, "crowded": 1700, "outside": 900}[case]
    print(f"case cell list {case} n={n}", flush=True)
    rng = np.random.default_rng(n)
    s = S.lj_fcc(1)
    s.density = n / 27.0                       # a box of 3
    if case == "outside":
        pos = rng.uniform(-4.0, 4.0, (n, 3))
    else:
        pos = rng.uniform(-1.5, 1.5, (n, 3))
    if case == "crowded":
        pos[:1400] = rng.uniform(0.6, 1.4, (1400, 3))
    s.pos, s.type, s.mol = pos, np.zeros(n, dtype=np.int32), np.arange(n, dtype=np.int32)
    s.bonds = [(0, k, 0) for k in range(1, 10)] + [(k, k + 1, 0) for k in range(20, n - 1, 3)]
    off, nb, used = O.Oracle(s).pairlist(0.85, 0.1, True)
    assert used
    ctx = Context(s)
    ctx.set_pairlist(0.85, 0.1, True)
    goff, gnb = ctx.pairlist()
    np.testing.assert_array_equal(goff, off)
    np.testing.assert_array_equal(gnb, nb)
    ctx.close()


@pytest.mark.parametrize("cells", [1, 2, 3, 4])
def test_lj_step_sizes_match_the_oracle(cells):
    """4, 32, 108 and 256 atoms: part of a block of the update and kinetics
    kernel, and whole blocks with and without a remainder; 10 steps in
    reduced units with list rebuilds, the trajectory tests' bars."""
    from oracle import oracle as O
    from swinmd_amd.forces import Context, WaterMD
    s = S.lj_fcc(cells, jitter=0.02)
    half = 0.5 * s.box[0]
    c = dict(cutoff=min(2.5, 0.8 * half), cut_buff=0.02, dt=0.004, temperature=0.8 / 0.0083145112, coupl=0.5,
             constraint=False, ewald=False, switch_on=True, use_cells=half > 1.5 * 2.52, atom_thermo=True)
    print(f"case lj step {s.n_atoms} atoms", flush=True)
    o = O.Oracle(s)
    vel = o.init_velocity(c["temperature"], 2, per_atom=True, ndf=3 * s.n_atoms - 3)
    ref = O.md_from_cfg(o, c, 10, velocity=vel)
    ctx = Context(s)
    ctx.set_velocities(vel)
    md = WaterMD(ctx, cutoff=c["cutoff"], cut_buff=c["cut_buff"], dt=c["dt"], temperature=c["temperature"],
                 coupl=c["coupl"], atom_thermo=True, constraint=False, ewald=False, switch_on=True,
                 use_cells=c["use_cells"])
    md.init()
    md.run(4)
    rep = md.run(6)
    assert rep["list_updates"] == ref["list_updates"]
    assert rel_rms(ctx.positions(), ref["pos"]) <= 1e-10
    assert rel_rms(ctx.velocities(), ref["vel"]) <= 1e-8
    for k in ("e_lj", "atom_ke2"):
        assert rel(rep[k], ref[k]) <= 1e-8, k
    ctx.close()


@pytest.mark.parametrize("kind", ["lj", "water"])
@pytest.mark.parametrize("cells", [True, False])
@pytest.mark.parametrize("prec", [L.PREC_FP64, L.PREC_MIXED])
def test_rows_outgrowing_the_list_in_a_step_are_an_error(kind, cells, prec):
    """Atoms in a box of 4 fall towards its middle, every distance shrinking by
    the same factor, so that rows pass the capacity fixed when the step was
    set up (1.5 times the first rows, and more) in a rebuild inside the run.
    The pair kernels of that step and the next walk the cut rows; the run
    ends with the capacity's error."""
    from swinmd_amd._lib import SMD_ECAPACITY, SmdError
    from swinmd_amd.forces import Context, WaterMD
    print(f"case outgrown rows {kind} cells={cells} prec={prec}", flush=True)
    dt, steps, shrink = 0.002, 10, 0.5 if kind == "lj" else 0.6
    if kind == "lj":
        s = S.lj_fcc(5, rho=500 / 64.0, sigma=0.15, eps=1e-6)
        com = s.pos
    else:
        s = S.water(343, box=4.0, seed=4, subset=True, jitter=0.0)
        com = np.repeat(s.pos.reshape(-1, 3, 3).mean(1), 3, axis=0)
    ctx = Context(s)
    vel = -com * (1 - shrink) / (steps * dt)
    # the thermostat holds the fall's own kinetic energy
    temperature = float((s.mass[:, None] * vel ** 2).sum() / ((3 if kind == "lj" else 2) * s.n_atoms * 0.0083145112))
    ctx.set_velocities(vel)
    md = WaterMD(ctx, cutoff=0.9, cut_buff=0.1, dt=dt, temperature=temperature, coupl=10.0, use_cells=cells, prec=prec,
                 constraint=kind == "water", ewald=kind == "water", kcut=S.kcut_for(3, 4.0))
    md.init()
    assert md.run(2)["list_updates"] >= 1
    with pytest.raises(SmdError) as e:
        md.run(steps)
    assert e.value.code == SMD_ECAPACITY
    ctx.close()


def _turned_over(s, m, dt):
    """Velocities that take molecule m's first hydrogen past its oxygen in one
    step: the new bond is twice as long and points 0.01 of it back, which
    SHAKE refuses (LFIntegrator.cpp:1519-1523) at its first constraint."""
    v = np.zeros((s.n_atoms, 3))
    bond = s.pos[3 * m] - s.pos[3 * m + 1]
    side = np.cross(bond, [0.3, 0.5, 0.8])
    new = -0.01 * bond + 2 * np.linalg.norm(bond) * side / np.linalg.norm(side)
    v[3 * m] = (new - bond) / dt
    return v


@pytest.mark.parametrize("wrap", [False, True])
def test_a_step_shake_refuses_leaves_its_molecule_unmoved(wrap):
    """The run ends with the constraint error, and the refused molecule is
    where its velocities took it, within the forces' dt^2 F / m < 0.01 nm, not
    where the refused quotient would put it, 15 nm away.  wrap: a molecule
    across the box face, where the sweeps take minimum images."""
    from swinmd_amd._lib import SMD_ESHAKE, SmdError
    from swinmd_amd.forces import Context, WaterMD
    s, cfg = _water_cfg(64)
    print(f"case refused step wrap={wrap}", flush=True)
    box, dt = s.box[0], 1e-4
    if wrap:   # hydrogens and oxygens of one molecule on either side of a face
        s.pos = s.pos - s.pos[0] * [1, 0, 0] + [0.5 * box - 1e-3, 0, 0]
        s.pos = s.pos - box * np.rint(s.pos / box)
    ctx = Context(s)
    vel = _turned_over(s, 0, dt)
    if wrap:
        whole = s.pos[:3] - box * np.rint((s.pos[:3] - s.pos[1]) / box)
        assert np.abs(whole - s.pos[:3]).max() > 1
    ctx.set_velocities(vel)
    md = WaterMD(ctx, **{**{k: cfg[k] for k in ("cutoff", "cut_buff", "alpha", "kcut", "use_cells")}, "dt": dt,
                         "temperature": 300.0, "coupl": 1e3})
    md.init()
    with pytest.raises(SmdError) as e:
        md.run(1)
    assert e.value.code == SMD_ESHAKE
    d = ctx.positions()[:3] - (s.pos[:3] + dt * vel[:3])
    d -= box * np.rint(d / box)
    assert np.abs(d).max() < 0.01
    ctx.close()


def test_a_replica_step_shake_refuses_leaves_its_molecule_unmoved():
    """As the step above, for the sheared replicas' step."""
    from swinmd_amd._lib import SMD_ESHAKE, SmdError
    from swinmd_amd.nemd import ShearBatch
    s = S.water(256, density_mol=RHO, seed=8, subset=True)
    print("case refused replica step", flush=True)
    box, dt = s.box[0], 1e-4
    vel = _turned_over(s, 7, dt)
    b = ShearBatch([s], [0.5], cutoff=0.8, cut_buff=0.08, alpha=3.5, n2max=20, dt=dt, temperature=300.0, coupl=1e3)
    b.set_state([s.pos], [vel], [0.0])
    b.start()
    with pytest.raises(SmdError) as e:
        b.run(1)
    assert e.value.code == SMD_ESHAKE
    d = b.state()["pos"][21:24] - (s.pos[21:24] + dt * vel[21:24])
    d -= box * np.rint(d / box)
    assert np.abs(d).max() < 0.01
    b.close()


@pytest.mark.parametrize("n2", [20, 306])
def test_autotuner_times_the_tiles_that_the_passes_read(n2):
    """The row force pass has no k tiles, so they are neither timed nor
    changed; past its tables' size the direct pass has."""
    from swinmd_amd.nemd import ShearBatch
    s = S.water(256, density_mol=RHO, seed=9, subset=True)
    print(f"case autotuned tiles n2={n2}", flush=True)
    b = ShearBatch([s], [1.0], cutoff=0.8, cut_buff=0.08, alpha=3.5, n2max=n2, dt=0.002)
    b.set_tiles(kforce_tile=192)
    b.set_state([s.pos], [np.zeros_like(s.pos)], [0.0])
    b.start()
    best, table = b.autotune(reps=2)
    timed = [row["kforce_tile"] for row in table if "kforce_tile" in row]
    assert sum("pair_lanes" in row for row in table) == 4 and sum("sfac_chunk" in row for row in table) == 3
    if n2 == 20:
        assert not timed and best["kforce_tile"] == 192
    else:
        assert len(timed) == 3 and best["kforce_tile"] in timed
    b.close()


@pytest.mark.parametrize("prec,tiles", [(L.PREC_FP64, dict(kforce_tile=64, sfac_chunk=64)),
                                        (L.PREC_FP64, dict(kforce_tile=1536, sfac_chunk=512)), (L.PREC_MIXED, {}),
                                        (L.PREC_MIXED, dict(kforce_tile=128, sfac_chunk=256))])
def test_direct_sheared_reciprocal_passes_match_the_oracle(prec, tiles):
    """The passes for k sets past the row tables, in both precisions and with
    tiles that end inside the k set and the atoms: forces and energies after
    two steps at a tilt, FP64 1e-8, mixed 1e-5 (the form's own bar)."""
    from oracle import oracle as O
    from swinmd_amd.nemd import ShearBatch
    s = S.water(275, density_mol=RHO, seed=275, subset=True)
    kcut = S.kcut_for(306, s.box[0])
    vel = O.Oracle(s).init_velocity(300.0, 5, per_atom=False, ndf=3 * s.n_mols - 3)
    print(f"case direct sheared passes prec={prec} {tiles}", flush=True)
    b = ShearBatch([s], [3.0], cutoff=0.8, cut_buff=0.08, alpha=3.5, kcut=[kcut], dt=0.002, temperature=300.0,
                   coupl=0.1, prec=prec)
    if tiles:
        b.set_tiles(**tiles)
    b.set_state([s.pos], [vel], [0.31])
    b.start()
    b.run(2)
    st, rep = b.state(), b.reports()[0]
    want = O.sllod_run(O.Oracle(s), dict(cutoff=0.8, cut_buff=0.08, alpha=3.5, kcut=kcut, dt=0.002,
                                         temperature=300.0, coupl=0.1), 3.0, 2, velocity=vel, tilt=0.31)
    tol = 1e-8 if prec == L.PREC_FP64 else 1e-5
    assert rep["n_kvec"] == want["K"]
    assert rel(rep["e_long"], want["e_long"]) <= tol
    assert rel_rms(st["force"], want["force"]) <= tol
    b.close()


def test_ewald_setup_takes_the_memory_its_passes_use():
    """5,462 waters, |n|^2 <= 81: the structure factors' partials are 128 chunks
    of five weights (26 MB: two sets of row tiles a chunk, a block per CU), the
    phases 0.8 MB; 12 MB for the tables and the allocator's pages."""
    import ctypes as C
    from swinmd_amd.forces import Context, EwaldForce
    s = S.water(5462, density_mol=RHO, seed=1, subset=True)
    print("case ewald memory", flush=True)
    ctx = Context(s)
    ctx.compute_mol_centers()
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()

    def left():
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    before = left()
    ew = EwaldForce(ctx, alpha=3.5, real_cut=0.9, kcut=S.kcut_for(81, s.box[0]))
    took = before - left()
    rows = sum(1 for x in range(10) for y in range(0 if x == 0 else -9, 10) if x * x + y * y <= 81)
    assert took <= 128 * 5 * 4 * 10 * rows * 8 + 48 * s.n_atoms + 12e6, took
    # the passes with and without Lustig sums stay inside it
    assert np.isfinite(ew.compute_long(np.zeros((s.n_atoms, 3)))["energy"])
    ctx.close()


@pytest.mark.parametrize("crowd", [0.8, 0.3])
def test_cell_list_follows_a_crowded_cell(crowd):
    """Builds before and after the hit bits grow to a crowded cell, and a
    uniform one after that: rows in order, as the oracle's.  The smaller crowd
    has rows past the first capacity as well."""
    from oracle import oracle as O
    from swinmd_amd.forces import Context
    n = 2500
    print(f"case crowded cell {crowd}", flush=True)
    rng = np.random.default_rng(11)
    s = S.lj_fcc(1)
    s.density = n / 125.0                      # a box of 5
    even = rng.uniform(-2.5, 2.5, (n, 3))
    packed = even.copy()
    packed[:700] = 1.5 + rng.uniform(-0.5, 0.5, (700, 3)) * crowd
    s.type, s.mol = np.zeros(n, dtype=np.int32), np.arange(n, dtype=np.int32)
    s.pos = packed
    ctx = Context(s)
    for pos in (packed, packed, even, packed):
        s.pos = pos
        off, nb, used = O.Oracle(s).pairlist(0.9, 0.1, True)
        assert used
        ctx.set_positions(pos)
        ctx.set_pairlist(0.9, 0.1, True)
        goff, gnb = ctx.pairlist()
        np.testing.assert_array_equal(goff, off)
        np.testing.assert_array_equal(gnb, nb)
    ctx.close()


def test_captured_steps_outlive_a_list_that_grew():
    """A captured step after host builds that replaced the list's buffers (a
    crowd of atoms in one cell) runs on the new ones: the same trajectory as
    without them."""
    from swinmd_amd.forces import Context, WaterMD
    s = S.lj_fcc(8)                            # 2,048 atoms, box 13.4
    print("case captured step and grown list", flush=True)
    vel = np.random.default_rng(3).normal(0.0, 0.8, (s.n_atoms, 3))
    crowd = s.pos.copy()
    crowd[:900] = np.random.default_rng(4).uniform(0.2, 1.8, (900, 3))
    out = []
    for grow in (False, True):
        ctx = Context(s)
        ctx.set_velocities(vel - vel.mean(0))
        md = WaterMD(ctx, cutoff=2.5, cut_buff=0.3, dt=0.004, temperature=0.8 / 0.0083145112, coupl=0.5,
                     constraint=False, ewald=False, switch_on=True)
        md.init()
        md.run(3)
        pos = ctx.positions()
        if grow:
            ctx.set_positions(crowd)
            ctx.set_pairlist(2.5, 0.3, True)
        ctx.set_positions(pos)
        ctx.set_pairlist(2.5, 0.3, True)
        md.run(3)
        out.append(ctx.positions())
        ctx.close()
    assert rel_rms(out[1], out[0]) <= 1e-12


@pytest.mark.parametrize("n", [1, 26, 27, 40])
def test_cell_list_of_fewer_atoms_than_cells(n):
    """A grid of 27 cells with less than an atom a cell and with one or more:
    the rows of the oracle; two atoms are neighbours."""
    from oracle import oracle as O
    from swinmd_amd.forces import Context
    print(f"case dilute cell list n={n}", flush=True)
    rng = np.random.default_rng(n)
    s = S.lj_fcc(1)
    s.density = n / 27.0                       # a box of 3
    s.pos = rng.uniform(-1.5, 1.5, (n, 3))
    if n > 1:
        s.pos[1] = s.pos[0] + [0.1, 0.0, 0.0]
    s.type, s.mol = np.zeros(n, dtype=np.int32), np.arange(n, dtype=np.int32)
    off, nb, used = O.Oracle(s).pairlist(0.9, 0.05, True)
    assert used
    ctx = Context(s)
    ctx.set_pairlist(0.9, 0.05, True)
    goff, gnb = ctx.pairlist()
    np.testing.assert_array_equal(goff, off)
    np.testing.assert_array_equal(gnb, nb)
    ctx.close()


# molecules, edges, k cut as a count of the longest edge's waves: many units of
# rows and functions in several sets, functions past 16 with atoms enough for
# the FP64 walk, five tiles, one tile over several tables a chunk, and eight and
# nine functions, on both sides of the shared columns
@pytest.mark.parametrize("n,edges,waves", [(1100, (3.2, 3.2, 3.2), 11.85), (1000, (1.5, 1.5, 18.0), 49.5),
                                           (2200, (4.04, 4.04, 4.04), 7.04), (5600, (5.5, 5.5, 5.5), 2.1),
                                           (700, (2.8, 2.8, 2.8), 7.9), (700, (2.8, 2.8, 2.8), 8.1)])
@pytest.mark.parametrize("mixed", [False, True])
def test_lustig_sums_of_many_atoms_match_the_oracle(n, edges, waves, mixed):
    """Forces, energy, virial and volume derivatives of EwaldForce.compute_long,
    the bars of the smaller shapes; and the step's k-space, which forms no
    d-weighted sums, gives the same energy and forces."""
    from oracle import oracle as O
    from swinmd_amd.forces import Context, EwaldForce, LJForce, WaterMD
    s = S.water(n, box=edges[0], seed=n, subset=True, jitter=0.01)
    s.__class__ = _BoxedWater
    s.pos = s.pos + (np.repeat(s.pos[1::3], 3, axis=0) * (np.array(edges) / edges[0] - 1))   # whole molecules
    s.edges = edges
    kcut = 2 * np.pi * waves / max(edges)
    prec = L.PREC_MIXED if mixed else L.PREC_FP64
    print(f"case lustig n={n} edges={edges} waves={waves} mixed={mixed}", flush=True)
    ctx = Context(s)
    ctx.compute_mol_centers()
    ew = EwaldForce(ctx, alpha=3.5, real_cut=0.5, kcut=kcut, prec=prec)
    f = np.zeros((s.n_atoms, 3))
    out = ew.compute_long(f)
    fo, eo = O.Oracle(s).ewald_recip(kcut, 3.5)
    tol = 1e-5 if mixed else 1e-10
    assert rel_rms(f, fo) <= tol
    for k in ("energy", "deriv", "deriv2"):
        assert abs(out[k] - eo[k]) <= tol * max(abs(eo[k]), abs(eo["energy"])), k
    assert rel_rms(out["virial"], eo["virial"]) <= tol
    ctx.set_pairlist(0.5, 0.05, False)
    LJForce(ctx, cutoff=0.5, prec=prec).compute(f)
    ew.compute(f)
    ctx.set_velocities(np.zeros_like(f))
    md = WaterMD(ctx, cutoff=0.5, cut_buff=0.05, alpha=3.5, kcut=kcut, dt=1e-4, temperature=300.0, use_cells=False,
                 prec=prec)
    md.init()
    assert rel(md.run(1)["e_long"], out["energy"]) <= tol
    assert rel_rms(ctx.forces(), f) <= tol
    ctx.close()
