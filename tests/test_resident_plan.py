"""The resident solve's plan (host, integer): one product by the plan's
lists -- own upper blocks, their transposes through the product slots, ghost
blocks, halo rows -- gives the CSR matrix-vector product, with every index
inside the kernel's arrays."""
import numpy as np
import pytest

import chysx
from chysx import scenes

LEAF, PART, HELD, HALO, GHOST, NONE = 64, 1024, 6, 512, 512, 0xFFFFFFFF


def _pattern(nx, ny):
    _, tris = scenes.cloth_grid(nx, ny)
    d = chysx.topology.cloth_system(nx * ny, tris, np.zeros(0, np.int32))
    return d["row_offsets"], d["col_indices"]


def _slots(n, ro, ci):
    """Value slot of every CSR block: a number of its own per upper block."""
    bs, seen, at = np.zeros(len(ci), np.int64), {}, 0
    for i in range(n):
        for k in range(ro[i], ro[i + 1]):
            j = int(ci[k])
            if j > i:
                seen[i, j] = at
                bs[k] = at
                at += 1
    for i in range(n):
        for k in range(ro[i], ro[i + 1]):
            if ci[k] < i:
                bs[k] = -1 - seen[int(ci[k]), i]
    return bs.astype(np.int32), at


@pytest.mark.parametrize("nx,ny", [(2, 2), (5, 3), (8, 8), (33, 31), (40, 57), (128, 9), (65, 66)])
@pytest.mark.parametrize("part_rows", [256, 512, 1024])
def test_plan_product_is_the_matrix_product(nx, ny, part_rows):
    n = nx * ny
    ro, ci = _pattern(nx, ny)
    bs, n_values = _slots(n, ro, ci)
    plan = chysx.topology.resident_plan(n, ro, ci, bs, part_rows)
    order, blob, parts = plan["order"], plan["blob"].astype(np.int64), plan["parts"]
    assert sorted(order) == list(range(n)) and parts == -(-n // part_rows)
    rng = np.random.default_rng(n + part_rows)
    val, x = rng.integers(1, 50, n_values), rng.integers(-50, 50, n)  # scalar blocks, exact sums
    want = np.zeros(n, np.int64)
    rows = np.repeat(np.arange(n), np.diff(ro))
    np.add.at(want, rows, val[np.where(bs < 0, -1 - bs, bs)] * x[ci])
    rows_at, meta_at, exp_at, held_at = 8 * parts, 8 * parts + n, 8 * parts + 2 * n, 8 * parts + 3 * n
    export_row = {}
    for k in range(n):
        e = blob[exp_at + k]
        if e != NONE:
            assert 0 <= e < plan["exports"] and e not in export_row
            export_row[int(e)] = int(order[k])
    assert len(export_row) == plan["exports"]
    got = np.zeros(n, np.int64)
    for q in range(parts):
        own, halo, halo_at, ghost, ghost_at = blob[8 * q:8 * q + 5]
        a = q * part_rows
        assert own == min(part_rows, n - a) and halo <= HALO and ghost <= GHOST
        halo_rows = blob[halo_at:halo_at + 2 * halo].reshape(-1, 2)
        assert all(export_row[int(e)] == r for r, e in halo_rows)
        p = np.zeros(PART + HALO, np.int64)
        p[:own] = x[order[a:a + own]]
        p[PART:PART + halo] = x[halo_rows[:, 0]]
        prod, filled = np.zeros(HELD * PART, np.int64), np.zeros(HELD * PART, bool)

        def put(slot, v):
            assert not filled[slot]
            filled[slot], prod[slot] = True, v

        for g in blob[ghost_at:ghost_at + 2 * ghost].reshape(-1, 2):
            src = g[1] & 0xFFFF
            assert PART <= src < PART + halo and g[0] < n_values
            put(g[1] >> 16, val[g[0]] * p[src])
        for k in range(own):
            i = int(blob[rows_at + a + k])
            assert i == order[a + k]
            nl, nh = blob[meta_at + a + k] & 15, blob[meta_at + a + k] >> 4
            assert nl <= HELD and nh <= HELD and nl + nh == ro[i + 1] - ro[i]
            for u in range(nh):
                w = blob[held_at + u * n + a + k]
                col, v = w & 0xFFFF, val[bs[ro[i] + nl + u]]
                assert col < own or PART <= col < PART + halo
                got[i] += v * p[col]
                if w >> 16 != 0xFFFF:
                    assert col < own and (w >> 16) % PART == col
                    put(w >> 16, v * p[k])
        for k in range(own):
            i, nl = int(order[a + k]), blob[meta_at + a + k] & 15
            at = np.arange(HELD) * PART + k
            assert filled[at[:nl]].all() and not filled[at[nl:]].any()
            got[i] += prod[at[:nl]].sum()
            # column order: slot l holds the product with the l-th lower column
            lower = ci[ro[i]:ro[i] + nl]
            assert (prod[at[:nl]] == val[-1 - bs[ro[i]:ro[i] + nl]] * x[lower]).all()
    assert (got == want).all()


def test_pattern_outside_the_limits_has_no_plan():
    """A vertex coupled to more rows than a thread holds: no plan."""
    n = 40
    rows = np.r_[np.zeros(n - 1, np.int32), np.arange(1, n, dtype=np.int32)]
    cols = np.r_[np.arange(1, n, dtype=np.int32), np.zeros(n - 1, np.int32)]
    ro, ci = chysx.topology.build_pattern(n, rows, cols)
    bs, _ = _slots(n, ro, ci)
    assert chysx.topology.resident_plan(n, ro, ci, bs, 256) is None
