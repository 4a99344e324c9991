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


def _true_residual(cloth):
    """||b - A dx|| / ||b|| of the last solve, in FP64."""
    diag, ro, ci, val, rhs, dx = (np.asarray(a, np.float64) for a in cloth.sim.debug_dump_last_solve())
    ro, ci = ro.astype(np.int64), ci.astype(np.int64)
    rows = np.repeat(np.arange(len(diag)), np.diff(ro))
    Ax = np.einsum("nij,nj->ni", diag, dx)
    np.add.at(Ax, rows, np.einsum("nij,nj->ni", val, dx[ci]))
    return np.linalg.norm(rhs - Ax) / np.linalg.norm(rhs)


def _solve_from_rest(cloth, start, warm, cap, tol, dt=1.0 / 60.0):
    """One substep from `start` at rest, the solve from `warm`; its iterations."""
    cloth.pos.copy_(start)
    cloth.vel.zero_()
    cloth.sim.debug_set_warm_start(warm)
    cloth.sim.set_pcg_iterations(cap)
    cloth.sim.set_pcg_tolerance(tol)
    cloth.step(dt)
    return cloth.sim.last_pcg_iterations()


@pytest.mark.parametrize("inner", [127, 255])
def test_bf16_refinement_at_a_multiple_of_256_exchanges(gpu, inner):
    """After 127 inner iterations the refinement's rows are sent 256 exchanges
    after the set-up's, after 255 512.  The warm start is one for which the
    recursive residual has a new minimum at that iteration, and the tolerance
    lies between it and the last minimum, so that the refinement comes right
    there.  The solve does the streaming one's operations, so its true residual
    is that one's but for the rounding of alpha and beta: by a factor of two at
    most, more than an iteration changes it by."""
    from chysx import scenes

    a, b = (scenes.DeviceCloth(_spec(64, 61, 0)) for _ in range(2))
    for c in (a, b):
        c.sim.set_bf16_blocks(True)
    b.sim.set_lds_staging(False)  # the streaming solve
    start = a.pos.clone()
    for seed in range(32):
        warm = np.random.default_rng(seed).normal(0.0, 0.01, (a.spec.n, 3)).astype(np.float32)
        history = []
        for cap in (inner, *range(inner - 1, inner - 40, -1)):
            assert _solve_from_rest(a, start, warm, cap, 0.0) == cap
            history.append(a.sim.last_relative_residual())
            if cap < inner and history[0] > 0.98 * history[-1]:
                break
        else:
            break
    else:
        pytest.fail("no warm start with a new minimum there")
    tol = (history[0] * min(history[1:])) ** 0.5
    its = [_solve_from_rest(c, start, warm, inner + 200, tol) for c in (a, b)]
    res = [_true_residual(c) for c in (a, b)]
    print(f"seed {seed}, tolerance {tol:.2e}: {its} iterations, true residuals {res}", flush=True)
    assert inner < its[0] <= inner + 200 and a.sim.last_relative_residual() <= tol
    assert res[0] <= 2.0 * res[1]


@pytest.mark.parametrize("nx,ny,shuffle", [(32, 32, False), (64, 61, False), (40, 39, True)])
def test_more_iterations_than_a_tag_counts(gpu, nx, ny, shuffle):
    """600 FP32 iterations: the tags' exchange numbers go round twice.  With a
    step of a second the solve is far from converged then, so a wrong halo row
    would show in its residual."""
    from chysx import scenes

    a, b = (scenes.DeviceCloth(_spec(nx, ny, nx, shuffle)) for _ in range(2))
    b.sim.set_lds_staging(False)
    start = a.pos.clone()
    for cap in (255, 256, 257, 600):
        for c in (a, b):
            assert _solve_from_rest(c, start, np.zeros((nx * ny, 3), np.float32), cap, 0.0, dt=1.0) == cap
        res = [_true_residual(c) for c in (a, b)]
        print(f"{nx}x{ny}, {cap} iterations: true residuals {res}", flush=True)
        assert res[0] <= 2.0 * res[1]


def test_rows_solve_with_more_iterations_than_a_tag_counts(gpu):
    import torch

    import chysx
    from test_gpu_resident import _rows_system

    A, b = _rows_system(40)
    out = []
    for lanes in (8, 4):  # four lanes per row: the streaming solve
        x = torch.zeros_like(b)
        S = chysx.PCGSolver()
        S.solve(A, b.data_ptr(), x.data_ptr(), max_iterations=300, lanes_per_row=lanes)
        assert S.last_iterations() == 300
        out.append(x.cpu().numpy())
    # both at the FP32 floor of this diagonally dominant system
    assert np.abs(out[0] - out[1]).max() <= 1e-5 * np.abs(out[1]).max()


@pytest.mark.parametrize("calls", ["assemble and solve", "streaming steps between"])
def test_launch_numbers_start_over_at_any_reset(gpu, calls):
    """An assembly by itself and a streaming solve count as launches too, so
    the numbers start over at calls after which the resident kernel does not
    run; the next one that does clears the old tags.  Solves of two states in
    turn give each its first bits; what carries the same number from before
    they started over is of the other state."""
    import torch

    import chysx
    from chysx import scenes

    cloths = [scenes.DeviceCloth(_spec(n, n + 1, n)) for n in (40, 33)]
    batch = chysx.ClothBatch()
    for c in cloths:
        c.sim.set_pcg_iterations(4)
        c.sim.set_pcg_tolerance(0.0)
        batch.add_instance(c.sim)
    dt = cloths[0].spec.dt
    starts = [[c.pos + k * 1.0e-2 * torch.sin(9.0 * c.pos) for c in cloths] for k in range(2)]
    first = {}

    def solve(k):
        for c, start in zip(cloths, starts[k % 2]):
            c.pos.copy_(start)
            c.vel.zero_()
            c.sim.debug_set_warm_start(np.zeros((c.spec.n, 3), np.float32))
        torch.cuda.synchronize()
        if calls == "assemble and solve":
            batch.assemble(dt)
            batch.assemble(dt)  # three launches a solve: number 3 comes again after 255
            batch.solve()
        else:
            batch.step(dt)
        got = [c.state()[0] for c in cloths]
        want = first.setdefault(k % 2, got)
        assert all(np.array_equal(g, w) for g, w in zip(got, want)), k

    if calls == "assemble and solve":
        for k in range(300):
            solve(k)
    else:
        for k in range(16):
            solve(k)
            if k < 9:
                continue
            batch.set_lds_staging(False)
            for _ in range(254):
                batch.step(dt)
            batch.set_lds_staging(True)


def _disk(valence, rings, seed=0):
    """A round cloth: a centre with `valence` neighbours (2 * valence blocks in
    its row, with the opposite vertices of its bending elements) and rings."""
    from chysx import scenes

    a = 2.0 * np.pi * np.arange(valence) / valence
    ring = np.stack([np.cos(a), np.zeros(valence), np.sin(a)], 1)
    pos = np.concatenate([np.zeros((1, 3))] + [ring * (r + 1.0) / rings for r in range(rings)])
    pos = (0.5 * pos + [0.0, 1.0, 0.0] + np.random.default_rng(seed).normal(0.0, 1.0e-4, pos.shape)).astype(np.float32)
    at = lambda r, k: 1 + r * valence + k % valence
    tris = [(0, at(0, k + 1), at(0, k)) for k in range(valence)]
    for r in range(rings - 1):
        for k in range(valence):
            tris += [(at(r, k), at(r, k + 1), at(r + 1, k)), (at(r, k + 1), at(r + 1, k + 1), at(r + 1, k))]
    start = pos.copy()
    start[:, 1] += 0.02 * np.sin(7.0 * pos[:, 0] + 4.0 * pos[:, 2])
    return scenes.ClothSpec(pos=pos, tris=np.array(tris, np.int32), pins=np.array([at(rings - 1, 0)], np.int32),
                            k_stretch=100.0, k_shear=100.0, k_bend=1.0e-4, k_pin=1.0e6, density=0.2, dt=1.0 / 600.0,
                            max_iter=60, tol=1.0e-6, pos_start=start)


def test_a_batch_reports_the_solve_that_it_runs(gpu):
    """Settings and cloths that leave the resident solve, and those that do not."""
    import chysx
    from chysx import scenes

    cloths = [scenes.DeviceCloth(_spec(n, n + 1, n)) for n in (40, 33)]
    wide, narrow = (scenes.DeviceCloth(_disk(v, 40)) for v in (9, 8))
    batch = chysx.ClothBatch()
    assert not batch.resident()
    for c in cloths + [narrow]:
        batch.add_instance(c.sim)
    dt = cloths[0].spec.dt

    def runs():
        batch.step(dt)
        return batch.resident()

    assert runs()
    batch.set_lds_staging(False)
    assert not runs()
    batch.set_lds_staging(True)
    batch.set_pcg_form(1)
    assert not runs()
    batch.set_pcg_form(0)
    batch.set_grid_blocks(4)  # the 40x41 cloth has 7 parts
    assert not runs()
    batch.set_grid_blocks(0)
    assert runs()
    batch.add_instance(wide.sim)  # one row of 18 blocks: no plan
    assert not runs()
    batch.remove_instance(wide.sim)
    assert runs()
    wide.step()
    narrow.step()
    assert narrow.sim.resident() and not wide.sim.resident()


def test_a_grid_limit_set_while_a_stream_is_captured(gpu):
    """The limit is host state of the next launch: a graph captured with one
    replays the streaming solve, without one the resident one."""
    import torch

    from chysx import scenes

    cloth, eager = (scenes.DeviceCloth(_spec(40, 41, 3)) for _ in range(2))
    dt = cloth.spec.dt
    s = torch.cuda.Stream()
    cloth.step(dt, s.cuda_stream)
    eager.step(dt)
    torch.cuda.synchronize()
    for limit in (3, 0):
        eager.sim.set_grid_blocks(limit)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            cloth.sim.set_grid_blocks(limit)
            cloth.step(dt, torch.cuda.current_stream().cuda_stream)
        assert cloth.sim.resident() == (limit == 0)
        for _ in range(3):
            g.replay()
            torch.cuda.synchronize()
            eager.step(dt)
            assert np.array_equal(cloth.state()[0], eager.state()[0])


def test_a_batch_that_streams_keeps_no_plans_for_its_other_cloths(gpu):
    """One cloth without a plan: the others get none of the batch's part size
    on the device, only the one of their own steps."""
    import chysx
    from chysx import scenes

    batch = chysx.ClothBatch()
    cloths = [scenes.DeviceCloth(_spec(64, 61, k)) for k in range(20)]  # 320 parts of 256 rows
    for c in cloths:
        c.step()  # a plan of its own, 16 parts
    before = [c.sim.device_bytes() for c in cloths]
    wide = scenes.DeviceCloth(_disk(9, 40))
    for c in cloths + [wide]:
        batch.add_instance(c.sim)
    batch.step(cloths[0].spec.dt)
    assert not batch.resident() and [c.sim.device_bytes() for c in cloths] == before
    batch.remove_instance(wide.sim)
    batch.step(cloths[0].spec.dt)
    assert batch.resident() and all(c.sim.device_bytes() > b for c, b in zip(cloths, before))


@pytest.mark.parametrize("shuffle", [False, True])
@pytest.mark.parametrize("tile_rows", [256, 512, 1024])
def test_streaming_solve_below_a_grid_limit(gpu, tile_rows, shuffle):
    """A grid limit below the cloth's parts leaves its solve to the staged
    single-barrier kernel: 16-bit and 32-bit entries, tiles of several sizes,
    against the resident solve of the same cloth (the tolerances of
    test_gpu_resident.py, for its reasons)."""
    import helpers
    from chysx import scenes

    a, b = (scenes.DeviceCloth(_spec(52, 51, 5, shuffle)) for _ in range(2))  # 11 parts of 256 rows; 6 of 512
    b.sim.set_tile_rows(tile_rows)
    b.sim.set_grid_blocks(3)
    for _ in range(3):
        a.step()
        b.step()
        assert a.sim.resident() and not b.sim.resident() and b.sim.debug_entries16() != shuffle
        assert abs(a.sim.last_pcg_iterations() - b.sim.last_pcg_iterations()) <= 1
        assert helpers.rel_maxnorm(a.state()[0], b.state()[0]) <= 1e-6


def test_a_cloth_without_a_plan_against_the_oracle(gpu):
    """Valence 9: a row of 18 blocks, wider than a plan's."""
    import helpers
    from chysx import scenes

    spec = _disk(9, 40)
    cloth, oracle = scenes.DeviceCloth(spec), helpers.oracle_from_spec(spec)
    for _ in range(3):
        cloth.step()
        oracle.step(spec.dt)
    assert not cloth.sim.resident()
    assert helpers.rel_maxnorm(cloth.state()[0], oracle.state()[0]) <= 1e-5


def test_a_batch_with_a_cloth_without_a_plan(gpu):
    """The whole batch streams then: every cloth as alone but for the order of
    FP64 sums (the tolerances of test_gpu_resident.py); the one that streams
    alone too, bit for bit."""
    import chysx
    import helpers
    from chysx import scenes

    specs = [_spec(40, 41, 1), _disk(9, 40), _spec(12, 13, 2), _spec(27, 19, 3, True)]
    alone, mixed = ([scenes.DeviceCloth(s) for s in specs] for _ in range(2))
    batch = chysx.ClothBatch()
    for c in mixed:
        batch.add_instance(c.sim)
    for _ in range(3):
        batch.step(specs[0].dt)
        for c in alone:
            c.step()
        assert not batch.resident()
        for k, (a, i) in enumerate(zip(alone, batch.last_pcg_iterations())):
            assert abs(a.sim.last_pcg_iterations() - i) <= 1, k
    for k, (a, m) in enumerate(zip(alone, mixed)):
        assert helpers.rel_maxnorm(m.state()[0], a.state()[0]) <= 1e-6, k
    assert np.array_equal(alone[1].state()[0], mixed[1].state()[0])


@pytest.mark.parametrize("nx,ny,shuffle", [(16, 32, False), (27, 19, False), (64, 64, False), (27, 19, True)])
def test_bf16_velocities_and_residuals_are_the_streaming_solves(gpu, nx, ny, shuffle):
    """Velocities are the solution over the time step, so they show what
    positions of a metre hide.  Same operations but for the rounding of alpha
    and beta (6e-8 each, over at most 60 iterations of a preconditioned system
    whose condition is well below 1e4): 1e-3 of the largest velocity; the
    residual by less than an iteration changes it."""
    import helpers
    from chysx import scenes

    a, b = (scenes.DeviceCloth(_spec(nx, ny, 100 * nx + ny, shuffle)) for _ in range(2))
    for c in (a, b):
        c.sim.set_bf16_blocks(True)
    b.sim.set_lds_staging(False)  # the streaming solve
    for _ in range(4):
        a.step()
        b.step()
        assert a.sim.resident() and not b.sim.resident()
        assert helpers.rel_maxnorm(a.state()[1], b.state()[1]) <= 1e-3
        ra, rb = a.sim.last_relative_residual(), b.sim.last_relative_residual()
        assert ra <= 2.0 * rb and (a.sim.last_pcg_iterations() == 60 or ra <= 1e-6)


@pytest.mark.parametrize("grid", [0, 16, 13])
@pytest.mark.parametrize("count", [6, 1030])
def test_streaming_batches_are_their_cloths_alone(gpu, grid, count):
    """A batch that a wide cloth leaves to the staged streaming kernel: every
    cloth bit for bit as streamed alone (global gathers, the same sums in the
    same order).  1030 instances are more than the compacted tile list holds."""
    import chysx
    from chysx import scenes

    specs = scenes.batched(seed=15, count=count, lo=4, hi=48 if count < 1000 else 7)
    dt = specs[0].dt
    specs.append(_disk(9, 40))
    alone, mixed = ([scenes.DeviceCloth(s) for s in specs] for _ in range(2))
    batch = chysx.ClothBatch()
    for c in mixed:
        batch.add_instance(c.sim)
    batch.set_grid_blocks(grid)
    for c in alone:
        c.sim.set_lds_staging(False)
    for _ in range(2):
        batch.step(dt)
        for c in alone:
            c.step(dt)
        assert not batch.resident()
        assert batch.last_pcg_iterations() == [c.sim.last_pcg_iterations() for c in alone]
    for a, m in zip(alone, mixed):
        assert all(np.array_equal(p, q) for p, q in zip(a.state(), m.state()))


def test_a_batch_whose_waits_are_given_up(gpu):
    """A wait bound of one tick, set by the host: every workgroup of the
    resident solve leaves normally, pos and vel stay, the next step reports it,
    and the steps after that are those of a batch that never gave up."""
    import torch

    import chysx
    from chysx import scenes

    specs = [_spec(n, n + 1, n) for n in (40, 33, 64, 12)]
    sets = [[scenes.DeviceCloth(s) for s in specs] for _ in range(2)]
    batches = [chysx.ClothBatch() for _ in sets]
    for batch, cloths in zip(batches, sets):
        for c in cloths:
            batch.add_instance(c.sim)
        batch.step(specs[0].dt)
        assert batch.resident()
    before = [c.state() for c in sets[0]]
    batches[0].set_barrier_timeout_ticks(1)
    batches[0].step(specs[0].dt)
    torch.cuda.synchronize()
    batches[0].set_barrier_timeout_ticks(0)
    with pytest.raises(RuntimeError, match="timed out"):
        batches[0].step(specs[0].dt)
    for c, (pos, vel) in zip(sets[0], before):
        assert np.array_equal(c.state()[0], pos) and np.array_equal(c.state()[1], vel)
    for cloths in sets:
        for c in cloths:
            c.sim.debug_set_warm_start(np.zeros((c.spec.n, 3), np.float32))
    for _ in range(3):
        for batch in batches:
            batch.step(specs[0].dt)
    for a, b in zip(*sets):
        assert np.array_equal(a.state()[0], b.state()[0]) and np.array_equal(a.state()[1], b.state()[1])
