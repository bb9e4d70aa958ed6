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
