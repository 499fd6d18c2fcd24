"""Analytic Hessian of molecules, whose three-body term is summed pair by pair,
against the oracle: edges of the tiles of 8 and 16 positions, another exponent,
distances at the three-body cutoff, and a batch whose other systems keep the
lists.  Tolerance as in the Hessian tests: 1e-10 of the largest element."""
import sys

import numpy as np
import pytest
import torch

import oracle as O
from helpers import BJ, ZERO, cell

pytestmark = pytest.mark.gpu


def _step(msg):
    print(f"[gpu-hessian-pair-sums] {msg}", flush=True)
    sys.stdout.flush()


def _compare(systems):
    from dftd3 import torch_api
    spec, pos = torch_api.batch_spec(systems)
    out = torch_api.run_hessian(spec, torch.as_tensor(pos, dtype=torch.float64, device="cuda").contiguous())
    blocks = torch_api.hessian_blocks(out)
    for k, s in enumerate(systems):
        disp3 = s.get("cutoff", {}).get("disp3", O.DEFAULT_CUTOFF[2])
        cut = (*O.DEFAULT_CUTOFF[:2], disp3, *O.DEFAULT_CUTOFF[3:])
        ref = O.hessian(s["numbers"], s["positions"], s.get("lattice"), [True] * 3 if "lattice" in s else None,
                        O.ZERO if s.get("kind") == "zero" else O.RATIONAL, s["param"], cut)
        h = blocks[k].cpu().numpy()
        np.testing.assert_allclose(h, ref["hessian"], rtol=0, atol=1e-10 * np.abs(ref["hessian"]).max())
        assert abs(out["energy"][k].item() - ref["energy"]) <= 1e-10 * abs(ref["energy"])


@pytest.mark.parametrize("many", [False, True])
def test_tile_edges(many):
    from dftd3 import synthetic
    _step(f"tile edges, many={many}")
    systems = []
    for k, n in enumerate((2, 3, 7, 8, 9, 16, 17, 33)):
        num, pos = synthetic.molecule_c0(seed=60 + n, n=n)
        systems.append(dict(numbers=num, positions=pos, kind="zero" if k % 2 else "rational",
                            param=dict(ZERO if k % 2 else BJ, alp=15.0 if k % 3 == 0 else 14.0),
                            cutoff=dict(disp3=9.0 if k % 2 else 40.0)))
    num, pos, lat = cell(9, 4, 9.5)
    systems.insert(3, dict(numbers=num, positions=pos, lattice=lat, periodic=[True] * 3, param=BJ))
    if many:  # enough tile pairs for tiles of 16 positions
        num, pos = synthetic.molecule_c0(seed=61, n=20)
        systems += [dict(numbers=num, positions=pos + 0.01 * k, param=BJ) for k in range(220)]
    _compare(systems)


@pytest.mark.parametrize("scale", [1.0, 1.0 + 3e-10, 1.0 - 3e-10])
def test_distances_at_the_cutoff(scale):
    _step(f"cutoff band, scale 1{scale - 1.0:+.0e}")
    rng = np.random.default_rng(9)
    g = np.stack(np.meshgrid(np.arange(4), np.arange(3), np.arange(3), indexing="ij"), axis=-1).reshape(-1, 3)
    _compare([dict(numbers=rng.choice([1, 6], size=len(g)), param=BJ, cutoff=dict(disp3=6.0),
                   positions=3.0 * scale * rng.permutation(g) + np.array([0.1, 0.7, -0.3]))])
