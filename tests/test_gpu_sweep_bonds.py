"""One two-site DMRG sweep at the batched workload's full size (dmrg(),
dmrg.cpp:702-755) against the oracle's run of the same sweep
(tests/golden/sweep_cyl6x12_m2048.json), bond by bond: the energy of every bond, where
the truncation binds as well, agrees to 1e-10 per site.  That needs the canonical form of the
random start (rc(), qtt.cpp:821-850) to span the right spaces near the chain's ends, where
its matrices are graded over more than 15 decades: canonical tensors that miss them move
the bond energies by 1e-7 per site and leave the initial energy, the kept dimensions and the
bonds before the end unchanged."""

import numpy as np
import pytest

from test_gpu_sweep import GOLD, N, run
from ttgpu import lib as T

pytestmark = pytest.mark.gpu


def test_every_bond_matches_the_oracle():
    r = run(T.FP64)
    d = np.abs(r["bond_E"] - np.array(GOLD["bond_E"])) / N
    print(f"max per-bond |dE|/N {d.max():.2e} at bond {int(d.argmax())}, final {abs(r['E'] - GOLD['E']) / N:.2e}", flush=True)
    assert d.max() <= 1e-10
    assert abs(r["E"] - GOLD["E"]) / N <= 1e-10
    assert np.abs(r["trunc_err"] - np.array(GOLD["trunc_err"])).max() <= 1e-13
