"""Batches whose pair sums do not fit the free device memory take three-body
lists, which need less.  The memory is filled from the host; every launched
kernel runs as usual."""
import sys

import numpy as np
import pytest
import torch

from helpers import BJ

pytestmark = pytest.mark.gpu


def _step(msg):
    print(f"[gpu-memory-fallback] {msg}", flush=True)
    sys.stdout.flush()


def _wires(m, n):
    """m wires of 2 x 2 atoms: short lists, dense records and sums."""
    systems = []
    for seed in range(m):
        rng = np.random.default_rng(seed)
        grid = np.stack(np.meshgrid([0, 1], [0, 1], np.arange(n // 4), indexing="ij"), axis=-1).reshape(-1, 3)
        pos = 4.07 * (rng.permutation(grid) + rng.uniform(-0.23, 0.23, (n, 3)))
        systems.append(dict(numbers=rng.choice([1, 6, 7, 8], size=n), positions=pos, param=BJ))
    return systems


def test_lists_when_the_pair_sums_do_not_fit():
    """Four wires of 3,000 atoms, FP64, buffers a quarter larger than needed:
    1.4 GB of pair records, 2.2 GB of records and sums of the pair sums, a few
    MB of lists; with 2.2 GB of memory free."""
    from dftd3 import library, torch_api
    systems = _wires(4, 3000)
    spec, pos = torch_api.batch_spec(systems)
    p = torch.as_tensor(pos, dtype=torch.float64, device="cuda").contiguous()
    ws = library.new_workspace()
    library.set_kernel_timing(ws, True)
    ref = torch_api.run_batch(spec, p, precision="fp64", ws=ws)
    torch.cuda.synchronize()
    assert library.get_kernel_time(ws, "atm_list")[1] == 0
    del ws
    out = {k: torch.zeros_like(v) for k, v in ref.items()}
    ws = library.new_workspace()
    library.set_kernel_timing(ws, True)
    torch.cuda.empty_cache()
    free, _ = torch.cuda.mem_get_info()
    held = torch.empty(free - int(2.2e9), dtype=torch.uint8, device="cuda")
    try:
        try:
            torch.empty(int(3.0e9), dtype=torch.uint8, device="cuda")
            pytest.skip("more memory is free than the device reported")
        except torch.OutOfMemoryError:
            pass
        _step("batch call with 2.2 GB free")
        torch_api.run_batch(spec, p, precision="fp64", out=out, ws=ws)
        torch.cuda.synchronize()
    finally:
        del held
        torch.cuda.empty_cache()
    assert library.get_kernel_time(ws, "atm_list")[1] > 0
    for key in ("energy", "gradient", "sigma"):
        assert (out[key] - ref[key]).abs().max() <= 1e-11 * ref[key].abs().max(), key
