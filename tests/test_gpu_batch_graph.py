"""A batch that is run, autotuned and run again: the autotuner tries shapes
that need larger tile maps, and the graph of the first run must not outlive
the map it was captured with.  The results are those of the batch that is not
tuned (whatever the shape, as in test_gpu_batch: 1e-13)."""
import numpy as np
import pytest

import orc
from finess_amd import Batch, problems

pytestmark = pytest.mark.gpu


def test_autotune_between_runs():
    # 40 x 40: 9 tiles of 15 x 16, 12 of 7 x 32, 14 of 3 x 64
    sizes = [(40, 40)] * 90
    mem = [problems.sw_bump(nx=nx, ny=ny, A=0.1 + 0.002 * k)[:2] for k, (nx, ny) in enumerate(sizes)]
    res = []
    for tune in (False, True):
        with Batch(mem[0][0], sizes) as b:
            for k, (p, q) in enumerate(mem):
                b.set_state(k, q, 0.0, p.initial_dt)
            for _ in range(3):
                b.run(10)
                if tune:
                    b.autotune(3)
            res.append([b.get_state(k)[0] for k in range(len(mem))])
    for (p, _), a, c in zip(mem, *res):
        assert np.all(orc.rel_linf(orc.interior(p, a), orc.interior(p, c)) <= 1e-13)
