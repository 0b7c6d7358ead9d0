"""The colour pass's single-precision pair test (kf_device.hpp, F32Filter)
against the reference arithmetic on 2^19 pairs at its thresholds
(tests/gpu_checks/kf_f32_check.hip, built by __graft_entry__.build()): every
pair that it decides has the exact decision, over the cell sides, bond
ranges and patch angles that contexts may have; and trajectories at sizes
where a team's register slots are exactly filled or overflow are those of
the other team widths."""
import os
import re
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXE = os.path.join(ROOT, "patchyparticles_amd", "bin", "kf_f32_check")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side,reach,cosmax", [(1.0, 1.12, 0.92), (1.49, 1.12, 0.92), (8.0, 1.12, 0.92), (1.1, 1.5, 0.7),
                                               (1.0, 1.05, 0.995), (2.0, 3.0, 0.2), (60.0, 1.12, 0.92),
                                               (1.2, 1.12, 0.0), (1.2, 1.12, -0.5)])
def test_single_precision_decisions_at_the_thresholds(side, reach, cosmax):
    if not os.path.exists(EXE):
        pytest.fail(f"{EXE} is not built: run __graft_entry__.build()")
    res = subprocess.run([EXE, str(side), str(reach), str(cosmax)], capture_output=True, text=True, timeout=120)
    m = re.search(r"pairs (\d+) decided (\d+) unsure (\d+) mismatches (\d+)", res.stdout)
    assert m, res.stdout + res.stderr
    pairs, decided, unsure, bad = map(int, m.groups())
    assert bad == 0 and decided + unsure == pairs, res.stdout
    # five sixths of the pairs sit within 1e-9 to 1e-3 of a threshold
    # (uniform in the logarithm); a filter that is in use decides the others
    # at least, below its smallest cosine none but the pairs out of reach
    assert unsure > 0 and (decided > pairs // 6 or cosmax < 1e-3), res.stdout


@pytest.mark.parametrize("trials", [0, 16])
@pytest.mark.parametrize("rho,occupancy", [(0.05, 0.0), (0.5, 0.0), (0.6, 0.0), (0.6, 3.0), (0.3, 6.0)])
def test_trajectories_across_team_widths(rho, occupancy, trials):
    # candidates of a cell from about 2 to 160: one register slot, two, and
    # the neighbours beyond them
    import patchyparticles_amd as pp
    r, O, box = pp.generate(1500, rho, 12)
    got = []
    for tpc in (16, 32, 64):
        with pp.System(r, O, box, T=0.12, seed=9, threads_per_cell=tpc, block_size=64, cell_occupancy=occupancy,
                       trials_per_cell=trials) as s:
            s.do_ensemble(30)
            bonds, ov, total, any_ov = s.energy()
            assert not any_ov and total == s.counters()["bonds"]
            got.append(s.state())
    for x in got[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(got[0], x))
