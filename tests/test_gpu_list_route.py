"""Three-body lists of molecules above the sizes of the pair sums: lists by
storage order, with the dense form of the kernel for tile pairs that are mostly
within the cutoff.  Compared with the oracle at the bars of the parity tests."""
import sys

import numpy as np
import pytest
import torch

import oracle as O
from helpers import BJ

pytestmark = pytest.mark.gpu


def _step(msg):
    print(f"[gpu-list-route] {msg}", flush=True)
    sys.stdout.flush()


def _molecule(seed, n, shape):
    """n atoms at about 0.1 per cubic Angstrom in random order, at least 1 Angstrom apart."""
    rng = np.random.default_rng(seed)
    grid = np.stack(np.meshgrid(*[np.arange(m) for m in shape], indexing="ij"), axis=-1).reshape(-1, 3)[:n]
    pos = 4.07 * (rng.permutation(grid) + rng.uniform(-0.23, 0.23, (n, 3)))
    return rng.choice([1, 6, 7, 8], size=n, p=[0.5, 0.3, 0.1, 0.1]), pos


def _reference(s, grad=True):
    c = {**dict(disp2=60.0, disp3=40.0, cn=40.0, width2=0.0, width3=0.0), **s.get("cutoff", {})}
    return O.dispersion(s["numbers"], s["positions"], s.get("lattice"), [True] * 3 if "lattice" in s else None,
                        O.ZERO if s.get("kind") == "zero" else O.RATIONAL, s["param"],
                        (c["cn"], c["disp2"], c["disp3"], c["width2"], c["width3"]), grad=grad)


def _compare(out, off, k, ref, n, mixed, grad):
    e, er = out["energy"][k].item(), ref["energy"]
    assert abs(e - er) <= (1e-8 * n if mixed else 1e-10 * abs(er)), (k, e, er)
    if grad:
        assert np.abs(out["gradient"][off:off + n].cpu().numpy() - ref["gradient"]).max() <= (1e-7 if mixed else 1e-9)
        assert np.abs(out["sigma"][k].cpu().numpy() - ref["virial"]).max() <= (1e-7 * n if mixed else 1e-9)


@pytest.mark.parametrize("n,shape,disp3,m", [(1751, (13, 13, 11), 40.0, 1), (300, (7, 7, 7), 12.0, 14)])
def test_capture_without_an_evaluation_before(n, shape, disp3, m):
    """A plan holds every buffer of an evaluation, so that its first one can
    be recorded: lists of a large molecule, and of a batch of small ones with
    a short cutoff."""
    from dftd3 import library, torch_api
    _step(f"capture first, {m} x {n} atoms")
    num, pos = _molecule(n, n, shape)
    s = dict(numbers=num, positions=pos, param=BJ, cutoff=dict(disp3=disp3))
    spec, p = torch_api.batch_spec([s] * m)
    p = torch.as_tensor(p, dtype=torch.float64, device="cuda").contiguous()
    plan = torch_api.BatchPlan(spec, p, precision="mixed")
    plan.capture()
    ref = _reference(s)
    for _ in range(3):
        for v in plan.out.values():
            v.zero_()
        _compare(plan.replay(), 0, 0, ref, n, True, True)
