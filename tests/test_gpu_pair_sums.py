"""Three-body term of molecules by pair sums (every pair's sum over all third
atoms, from per-pair records) against the oracle, at the edges of its tiles (8
or 16 positions a side, 4 or 8 third atoms a chunk), with a switching width,
another exponent, ghost atoms and distances at the cutoff; and the list route
that larger molecules keep."""
import sys

import numpy as np
import pytest
import torch

import oracle as O
from helpers import BJ, ZERO, cell

pytestmark = pytest.mark.gpu


def _step(msg):
    print(f"[gpu-pair-sums] {msg}", flush=True)
    sys.stdout.flush()


def _molecule(seed, n, shape=None):
    """n atoms at about 0.1 per cubic Angstrom in random order, at least 1 Angstrom apart."""
    rng = np.random.default_rng(seed)
    shape = shape or [int(np.ceil(n ** (1.0 / 3.0)))] * 3
    grid = np.stack(np.meshgrid(*[np.arange(m) for m in shape], indexing="ij"), axis=-1).reshape(-1, 3)
    pos = 4.07 * (rng.permutation(grid)[:n] + rng.uniform(-0.23, 0.23, (n, 3)))
    return rng.choice([1, 6, 7, 8], size=n, p=[0.5, 0.3, 0.1, 0.1]), pos


def _check(out, systems, mixed):
    off = 0
    for k, s in enumerate(systems):
        n = len(s["numbers"])
        width3 = s.get("cutoff", {}).get("width3", 0.0)
        disp3 = s.get("cutoff", {}).get("disp3", O.DEFAULT_CUTOFF[2])
        cut = (*O.DEFAULT_CUTOFF[:2], disp3, O.DEFAULT_CUTOFF[3], width3)
        ref = O.dispersion(s["numbers"], s["positions"], s.get("lattice"), [True] * 3 if "lattice" in s else None,
                           O.ZERO if s.get("kind") == "zero" else O.RATIONAL, s["param"], cut)
        e, er = out["energy"][k].item(), ref["energy"]
        assert abs(e - er) <= (1e-8 * n if mixed else 1e-10 * abs(er)), (k, n, e, er)
        if "gradient" in out:
            g, sg = out["gradient"][off:off + n].cpu().numpy(), out["sigma"][k].cpu().numpy()
            assert np.abs(g - ref["gradient"]).max() <= (1e-7 if mixed else 1e-9), (k, n)
            assert np.abs(sg - ref["virial"]).max() <= (1e-7 * n if mixed else 1e-9), (k, n)
        off += n


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("many", [False, True])
def test_tile_edges(many, precision, grad):
    """Molecules of 2 to 131 atoms around a cell in one batch: tiles of 8
    positions, and, with many of them, tiles of 16."""
    from dftd3 import torch_api
    _step(f"tile edges, many={many}, {precision}, grad={grad}")
    systems = []
    for k, n in enumerate((2, 3, 7, 8, 9, 15, 16, 17, 31, 33, 64, 65, 127, 131)):
        num, pos = _molecule(100 + n, n)
        par = dict(BJ if k % 2 else ZERO, alp=16.0 if k % 3 == 0 else 14.0)
        systems.append(dict(numbers=num, positions=pos, param=par, kind="rational" if k % 2 else "zero",
                            cutoff=dict(width3=6.0, disp3=14.0) if k % 4 == 1 else dict(disp3=25.0)))
    num, pos, lat = cell(7, 6, 11.0)
    systems.insert(5, dict(numbers=num, positions=pos, lattice=lat, periodic=[True] * 3, param=BJ))
    # 40 tile pairs of 16 positions in a molecule of 130 atoms
    extra = [dict(numbers=_molecule(7, 130)[0], positions=_molecule(7, 130)[1], param=BJ)] * (15 if many else 0)
    spec, pos = torch_api.batch_spec(systems + extra)
    p = torch.as_tensor(pos, dtype=torch.float64, device="cuda").contiguous()
    _check(torch_api.run_batch(spec, p, precision=precision, grad=grad), systems + extra[:1], precision == "mixed")
    plan = torch_api.BatchPlan(spec, p, precision=precision, grad=grad)
    _check(plan.execute(), systems + extra[:1], precision == "mixed")


@pytest.mark.parametrize("scale", [1.0, 1.0 + 3e-10, 1.0 - 3e-10])
@pytest.mark.parametrize("shape", [(5, 4, 4), (11, 8, 8)])
@pytest.mark.parametrize("grad", [True, False])
def test_distances_at_the_cutoff(grad, shape, scale):
    """Grids of spacing 3 bohr and a cutoff of 6 bohr: distances at the cutoff
    to the last bit, or within the band that the reference's arithmetic
    decides (tiles of 8 and of 16 positions)."""
    from dftd3 import torch_api
    _step(f"cutoff band, {shape}, scale 1{scale - 1.0:+.0e}, grad={grad}")
    rng = np.random.default_rng(9)
    g = np.stack(np.meshgrid(*[np.arange(m) for m in shape], indexing="ij"), axis=-1).reshape(-1, 3)
    s = dict(numbers=rng.choice([1, 6], size=len(g)), param=BJ, cutoff=dict(disp3=6.0),
             positions=3.0 * scale * rng.permutation(g) + np.array([0.1, 0.7, -0.3]))
    _check(torch_api.get_dispersion_batch([s], precision="fp64", grad=grad), [s], False)


@pytest.mark.parametrize("n", [5, 150])
def test_ghosts_and_pairs(n):
    """Ghost atoms have no three-body term; the pair energies are symmetric."""
    from dftd3.interface import DispersionModel, RationalDampingParam
    _step(f"ghosts and pair energies, {n} atoms")
    num, pos = _molecule(n, n)
    ghost = np.zeros(n, dtype=np.int32)
    ghost[[1, n - 2]] = 1
    model = DispersionModel(num, pos)
    model.set_ghost_atoms(np.flatnonzero(ghost))
    out = model.get_dispersion(RationalDampingParam(**BJ), grad=True)
    ref = O.dispersion(num, pos, None, None, O.RATIONAL, BJ, O.DEFAULT_CUTOFF, ghost=ghost)
    assert abs(float(out["energy"]) - ref["energy"]) <= 1e-10 * abs(ref["energy"])
    assert np.abs(out["gradient"] - ref["gradient"]).max() <= 1e-9
    pairs = model.get_pairwise_dispersion(RationalDampingParam(**BJ))
    r2, r3 = O.pairwise(num, pos, None, None, O.RATIONAL, BJ, O.DEFAULT_CUTOFF, ghost=ghost)
    got = pairs["non-additive pairwise energy"]
    np.testing.assert_allclose(got, r3, rtol=0, atol=1e-10)
    np.testing.assert_array_equal(got, got.T)


@pytest.mark.parametrize("n,precision", [(1750, "mixed"), (1751, "mixed"), (3501, "fp64")])
def test_largest_of_the_route_and_beyond(n, precision):
    """A rod of n atoms, at the size limit of the route and just above it (lists)."""
    from dftd3 import torch_api
    _step(f"rod of {n} atoms, {precision}")
    num, pos = _molecule(n, n, (8, 8, (n + 63) // 64))
    s = dict(numbers=num, positions=pos, param=BJ)
    _check(torch_api.get_dispersion_batch([s], precision=precision, grad=True), [s], precision == "mixed")
