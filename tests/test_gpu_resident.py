"""The resident solve against the streaming one on the GPU, at the sizes
where its plans change form: one part and several, a last part of one row,
sums over more than 64 parts, any vertex numbering, a caller's rows, and
batches whose parts outnumber the workgroups.

Both solvers do the same operations per row and sum FP64 products in another
order, so alpha and beta differ by FP32 rounding at most: positions agree to
1e-6 of their size after a few substeps (the solve's own tolerance, on
displacements well below the cloth's size), iteration counts to one."""
import numpy as np
import pytest

import helpers

pytestmark = pytest.mark.gpu


def _spec(nx, ny, seed, shuffle=False):
    from chysx import scenes

    rng = np.random.default_rng(seed)
    pos, tris = scenes.cloth_grid(nx, ny)
    pos = pos + rng.normal(0.0, 1.0e-4, pos.shape).astype(pos.dtype)
    start = pos.copy()
    start[:, 1] += 0.02 * np.sin(7.0 * pos[:, 0] + 4.0 * pos[:, 2])
    pins = np.array([0, nx - 1], np.int32)
    if shuffle:
        perm = rng.permutation(nx * ny)
        inv = np.empty(nx * ny, np.int32)
        inv[perm] = np.arange(nx * ny, dtype=np.int32)
        pos, start, tris, pins = pos[perm], start[perm], inv[tris], np.sort(inv[pins])
    return scenes.ClothSpec(pos=pos, tris=tris, pins=pins, k_stretch=100.0, k_shear=100.0, k_bend=1.0e-4,
                            k_pin=1.0e6, density=0.2, dt=1.0 / 600.0, max_iter=60, tol=1.0e-6, pos_start=start)


def _pair(spec):
    from chysx import scenes

    a, b = scenes.DeviceCloth(spec), scenes.DeviceCloth(spec)
    b.sim.set_lds_staging(False)  # the streaming solve
    return a, b


@pytest.mark.parametrize("nx,ny,shuffle", [
    (2, 2, False), (8, 8, False), (5, 13, False), (32, 32, False), (25, 41, False), (64, 64, False),
    (131, 127, False), (16, 32, True), (27, 19, True), (40, 39, True), (130, 129, True)])
def test_resident_step_matches_the_streaming_step(gpu, nx, ny, shuffle):
    a, b = _pair(_spec(nx, ny, 100 * nx + ny, shuffle))
    for step in range(3):
        a.step()
        b.step()
        ia, ib = a.sim.last_pcg_iterations(), b.sim.last_pcg_iterations()
        print(f"{nx}x{ny} step {step}: {ia} / {ib} iterations", flush=True)
        assert abs(ia - ib) <= 1
        assert helpers.rel_maxnorm(a.state()[0], b.state()[0]) <= 1e-6


@pytest.mark.parametrize("nx,ny,shuffle", [(8, 8, False), (16, 32, False), (27, 19, False), (64, 64, False), (27, 19, True)])
def test_resident_bf16_step_matches_the_streaming_step(gpu, nx, ny, shuffle):
    """BF16 blocks: half sheets of one part (512 rows) and several, and the
    general plan.  The BF16 matrix is the same; the residual that is reached
    (tolerance 1e-6, or the cap) is compared, not the iterations."""
    from chysx import scenes

    a, b = (scenes.DeviceCloth(_spec(nx, ny, 100 * nx + ny, shuffle)) for _ in range(2))
    for c in (a, b):
        c.sim.set_bf16_blocks(True)
    b.sim.set_lds_staging(False)
    for step in range(2):
        a.step()
        b.step()
        print(f"{nx}x{ny} step {step}: {a.sim.last_pcg_iterations()} / {b.sim.last_pcg_iterations()} iterations", flush=True)
        assert helpers.rel_maxnorm(a.state()[0], b.state()[0]) <= 1e-5


def _rows_system(n, extra=0):
    """A diagonally dominant block matrix over an n-by-n grid, and a right-hand side."""
    import torch

    import chysx

    rng = np.random.default_rng(n)
    N = n * n
    y, x = np.divmod(np.arange(N), n)
    off = [(1, 0), (0, 1), (1, 1), (-1, 1)] + [(k, 0) for k in range(2, 2 + extra)]
    ri, ci = [], []
    for dx, dy in off:
        ok = (x + dx >= 0) & (x + dx < n) & (y + dy < n)
        i = np.arange(N)[ok]
        ri += [i, i + dy * n + dx]
        ci += [i + dy * n + dx, i]
    rows, cols = np.concatenate(ri).astype(np.int32), np.concatenate(ci).astype(np.int32)
    order = np.lexsort((cols, rows))
    rows, cols = rows[order], cols[order]
    lo, hi = np.minimum(rows, cols), np.maximum(rows, cols)
    w = (1.0 + np.mod(lo * 7919.0 + hi * 104729.0, 13.0)).astype(np.float32)
    vals = -w[:, None, None] * (np.eye(3, dtype=np.float32) + 0.1)
    diag = np.zeros((N, 3, 3), np.float32)
    np.add.at(diag, rows, -vals)
    diag += 3.0 * np.eye(3, dtype=np.float32)
    A = chysx.BlockCSR3()
    A.build_topology(N, rows, cols)
    A.upload(diag, vals)
    b = torch.from_numpy(rng.normal(size=(N, 3)).astype(np.float32)).cuda()
    return A, b


@pytest.mark.parametrize("n,extra", [(8, 0), (23, 0), (64, 0), (40, 9)])
def test_rows_plan_matches_streamed_rows(gpu, n, extra):
    """A caller's matrix: the resident solve (eight lanes per row) against
    four lanes per row, which streams; `extra` blocks per row widen it past
    the plan's limit for some rows, where both stream."""
    import torch

    import chysx

    A, b = _rows_system(n, extra)
    out = []
    for lanes in (8, 4):
        x = torch.zeros_like(b)
        S = chysx.PCGSolver()
        S.solve(A, b.data_ptr(), x.data_ptr(), max_iterations=40, tolerance=1e-6, lanes_per_row=lanes)
        out.append((x.cpu().numpy(), S.last_iterations()))
    assert abs(out[0][1] - out[1][1]) <= 1
    assert helpers.rel_maxnorm(out[0][0], out[1][0]) <= 1e-5


def test_launch_numbers_start_over(gpu):
    """Tags name 255 launches; then the exchange area is cleared.  The same
    solve on three parts gives the same bits across that point."""
    import torch

    import chysx

    A, b = _rows_system(23)
    S = chysx.PCGSolver()
    first = None
    for k in range(520):
        x = torch.zeros_like(b)
        S.solve(A, b.data_ptr(), x.data_ptr(), max_iterations=3 + k % 2)
        x = x.cpu().numpy()
        if k < 2:
            first = [x] if k == 0 else first + [x]
        assert np.array_equal(x, first[k % 2]), k


@pytest.mark.parametrize("blocks", [0, 16, 24])
def test_batch_with_more_parts_than_workgroups(gpu, blocks):
    """Large items that span groups of workgroups, and small ones dealt to
    idle workgroups; the same bits as each cloth alone."""
    import chysx
    from chysx import scenes

    specs = [_spec(n, n + 1, n) for n in (12, 33, 47, 90, 64, 17, 32, 100, 21, 35, 55, 48)]
    alone = [scenes.DeviceCloth(s) for s in specs]
    mixed = [scenes.DeviceCloth(s) for s in specs]
    batch = chysx.ClothBatch()
    for c in mixed:
        batch.add_instance(c.sim)
    if blocks:
        batch.set_grid_blocks(blocks)
    for step in range(3):
        for c in alone:
            c.step()
        batch.step(specs[0].dt)
        assert batch.last_pcg_iterations() == [c.sim.last_pcg_iterations() for c in alone]
    for a, m in zip(alone, mixed):
        assert np.array_equal(a.state()[0], m.state()[0]) and np.array_equal(a.state()[1], m.state()[1])


def test_batch_follows_a_cloth_that_is_rebuilt(gpu):
    """Other pins on a bound cloth rebuild its matrix and its plan: the batch
    steps as one that was bound afterwards."""
    import chysx
    from chysx import scenes

    specs = [_spec(40, 41, 1), _spec(30, 33, 2)]
    results = []
    for late in (True, False):
        cloths = [scenes.DeviceCloth(s) for s in specs]
        batch = chysx.ClothBatch()
        for c in cloths:
            batch.add_instance(c.sim)
        if late:
            batch.finalize(specs[0].dt)
        pins = np.array([5, 77], np.int32)
        cloths[0].sim.set_pins(pins, specs[0].pos[pins], 1.0e6)
        if not late:
            batch.finalize(specs[0].dt)
        for _ in range(2):
            batch.step(specs[0].dt)
        results.append([c.state()[0] for c in cloths])
    for p, q in zip(*results):
        assert np.array_equal(p, q)
