"""Three-body lists of large molecules (more than 512 atoms): each triple is
visited from its last atom in the storage order instead of the one with the
largest index, and tile pairs whose slots are mostly within the cutoff are
evaluated without the accepted-pair ring.  Compared with the oracle at the
bars of the parity tests."""
import sys

import numpy as np
import pytest
import torch

import oracle as O
from helpers import BJ, ZERO, cell

pytestmark = pytest.mark.gpu


def _step(msg):
    print(f"[gpu-storage-order] {msg}", flush=True)
    sys.stdout.flush()


def _molecule(seed, n):
    """n atoms at about 0.1 per cubic Angstrom in random order, at least 1 Angstrom apart."""
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    grid = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), axis=-1).reshape(-1, 3)
    pos = 4.07 * (rng.permutation(grid)[:n] + rng.uniform(-0.23, 0.23, (n, 3)))
    return rng.choice([1, 6, 7, 8], size=n, p=[0.5, 0.3, 0.1, 0.1]), pos


def _compare(out, off, k, ref, n, mixed):
    e, er = out["energy"][k].item(), ref["energy"]
    assert abs(e - er) <= (1e-8 * n if mixed else 1e-10 * abs(er)), (e, er)
    if "gradient" in out:
        assert np.abs(out["gradient"][off:off + n].cpu().numpy() - ref["gradient"]).max() <= (1e-7 if mixed else 1e-9)
        assert np.abs(out["sigma"][k].cpu().numpy() - ref["virial"]).max() <= (1e-7 * n if mixed else 1e-9)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("scale", [1.0, 1.0 + 3e-10, 1.0 - 3e-10])
def test_distances_at_the_cutoff(precision, scale):
    """A 9 x 8 x 8 grid of spacing 3 bohr in random order with a three-body
    cutoff of 6 bohr: distances at the cutoff to the last bit, or inside the
    band (1e-9 of the squared cutoff) that is decided by the reference's
    arithmetic, for listed pairs and for the third side of the triples."""
    from dftd3 import torch_api
    _step(f"cutoff band, scale 1{scale - 1.0:+.0e}, {precision}")
    rng = np.random.default_rng(9)
    g = np.array([[x, y, z] for x in range(9) for y in range(8) for z in range(8)], dtype=float)
    pos = 3.0 * scale * rng.permutation(g) + np.array([0.1, 0.7, -0.3])
    num = rng.choice([1, 6], size=len(pos))
    out = torch_api.get_dispersion_batch(
        [dict(numbers=num, positions=pos, param=BJ, cutoff=dict(disp3=6.0))], precision=precision)
    cut = (O.DEFAULT_CUTOFF[0], O.DEFAULT_CUTOFF[1], 6.0, 0.0, 0.0)
    ref = O.dispersion(num, pos, None, None, O.RATIONAL, BJ, cut)
    _compare(out, 0, 0, ref, len(num), precision == "mixed")


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("n,kind,width3", [(513, "rational", 0.0), (577, "zero", 8.0), (640, "rational", 0.0)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_large_molecule_among_others(precision, n, kind, width3, grad):
    """One large molecule (one atom past eight tiles, a ragged last tile,
    whole tiles) in a batch with a small molecule and a cell, whose lists
    keep the reference's triangle, through the batch entry point and through
    every launch shape of a plan."""
    from dftd3 import library, torch_api
    _step(f"{n} atoms {kind} width3={width3} {precision} grad={grad}")
    systems = []
    for num, pos, lat, par in ((*_molecule(n, n), None, ZERO if kind == "zero" else BJ),
                               (*_molecule(3, 30), None, BJ), (*cell(17, 12, 13.0), BJ)):
        s = dict(numbers=num, positions=pos, param=par, kind="zero" if par is ZERO else "rational",
                 cutoff=dict(width3=width3))
        if lat is not None:
            s.update(lattice=lat, periodic=[True] * 3)
        systems.append(s)
    spec, pos = torch_api.batch_spec(systems)
    p = torch.as_tensor(pos, dtype=torch.float64, device="cuda").contiguous()
    out = torch_api.run_batch(spec, p, precision=precision, grad=grad)
    cut = (*O.DEFAULT_CUTOFF[:4], width3)
    refs = [O.dispersion(s["numbers"], s["positions"], s.get("lattice"), [True] * 3 if "lattice" in s else None,
                         O.ZERO if s["kind"] == "zero" else O.RATIONAL, s["param"], cut, grad=grad) for s in systems]
    off = 0
    for k, s in enumerate(systems):
        _compare(out, off, k, refs[k], len(s["numbers"]), precision == "mixed")
        off += len(s["numbers"])
    plan = torch_api.BatchPlan(spec, p, precision=precision, grad=grad)
    for shape in library.plan_candidate_shapes():
        plan.set_shape(*shape)
        _compare(plan.execute(), 0, 0, refs[0], n, precision == "mixed")
    assert not plan.overflowed()
