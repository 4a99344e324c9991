"""The resident solve on the GPU where its parts, waves and launches meet:
the finalize of one-workgroup solves, long solves, launches of several kinds
in a row, batches that do not fit it."""
import numpy as np
import pytest

from test_gpu_resident import _spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,shuffle,bf16", [(9, 9, False, False), (32, 32, False, False), (27, 19, True, False),
                                                (16, 32, False, True)])
def test_finalize_takes_every_row_of_the_solution(gpu, nx, ny, shuffle, bf16):
    """One workgroup: x is stored in the plan's row order and read in row
    order.  pos and vel are exactly the last solution's (one FP32 operation
    each), in every substep."""
    from chysx import scenes

    cloth = scenes.DeviceCloth(_spec(nx, ny, 100 * nx + ny, shuffle))
    cloth.sim.set_bf16_blocks(bf16)
    inv_dt = np.float32(1.0) / np.float32(cloth.spec.dt)
    for step in range(20):
        before = cloth.state()[0].astype(np.float32)
        cloth.step()
        pos, vel = (a.astype(np.float32) for a in cloth.state())
        dx = cloth.sim.debug_dump_last_solve()[5]
        assert np.array_equal(pos, before + dx) and np.array_equal(vel, dx * inv_dt), step
