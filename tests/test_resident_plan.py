"""The resident solve's plan (host, integer): one product by the plan's
lists -- own upper blocks, their transposes through the product slots, ghost
blocks, halo rows -- gives the CSR matrix-vector product, with every index
inside the kernel's arrays."""
import numpy as np
import pytest

import chysx
from chysx import scenes

PART, HELD, HALO, GHOST, NONE = 1024, 6, 512, 512, 0xFFFFFFFF
GEN_PART, GEN_HELD, GEN_WIDTH = 512, 8, 16


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
            nl, nh = blob[meta_at + a + k] & 255, blob[meta_at + a + k] >> 8
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
            i, nl = int(order[a + k]), blob[meta_at + a + k] & 255
            at = np.arange(HELD) * PART + k
            assert filled[at[:nl]].all() and not filled[at[nl:]].any()
            got[i] += prod[at[:nl]].sum()
            # column order: slot l holds the product with the l-th lower column
            lower = ci[ro[i]:ro[i] + nl]
            assert (prod[at[:nl]] == val[-1 - bs[ro[i]:ro[i] + nl]] * x[lower]).all()
    assert (got == want).all()


@pytest.mark.parametrize("nx,ny,shuffle", [(2, 2, False), (16, 16, True), (33, 31, False), (33, 31, True), (65, 40, True)])
@pytest.mark.parametrize("part_rows", [256, 512])
def test_general_plan_product_is_the_matrix_product(nx, ny, shuffle, part_rows):
    """Any numbering: every pair's block is held once (or is a ghost of the
    other part), every product lands at its place in the column order of its
    row, with the transpose marked where the stored block is the other
    row's."""
    n = nx * ny
    _, tris = scenes.cloth_grid(nx, ny)
    if shuffle:
        tris = np.random.default_rng(n).permutation(n).astype(np.int32)[tris]
    d = chysx.topology.cloth_system(n, tris, np.zeros(0, np.int32))
    ro, ci = d["row_offsets"], d["col_indices"]
    bs, n_values = _slots(n, ro, ci)
    plan = chysx.topology.resident_plan(n, ro, ci, bs, part_rows, general=True)
    order, blob, parts = plan["order"], plan["blob"].astype(np.int64), plan["parts"]
    assert sorted(order) == list(range(n)) and parts == -(-n // part_rows)
    rows_at, meta_at, exp_at, held_at = 8 * parts, 8 * parts + n, 8 * parts + 2 * n, 8 * parts + 3 * n
    export_row = {int(blob[exp_at + k]): int(order[k]) for k in range(n) if blob[exp_at + k] != NONE}
    assert sorted(export_row) == list(range(plan["exports"]))
    for q in range(parts):
        own, halo, halo_at, ghost, ghost_at, widest = blob[8 * q:8 * q + 6]
        a = q * part_rows
        assert own == min(part_rows, n - a) and halo <= HALO and ghost <= GHOST
        halo_rows = blob[halo_at:halo_at + 2 * halo].reshape(-1, 2)
        assert all(export_row[int(e)] == r for r, e in halo_rows)
        row_of = {k: int(order[a + k]) for k in range(own)}
        row_of.update({GEN_PART + h: int(halo_rows[h, 0]) for h in range(halo)})
        got = {}  # product slot -> (row, column, value slot, as stored)

        def put(slot, *what):
            assert slot not in got and slot < GEN_WIDTH * GEN_PART
            got[slot] = what

        for value, w in blob[ghost_at:ghost_at + 2 * ghost].reshape(-1, 2):
            i, j = row_of[(w >> 16) % GEN_PART], row_of[w & 0xFFFF]
            # the kernel transposes a ghost block unless its mark is set
            put(w >> 16, i, j, value & 0x7FFFFFFF, bool(value >> 31))
        for k in range(own):
            i, meta = row_of[k], blob[meta_at + a + k]
            assert blob[rows_at + a + k] == i and meta & 255 == ro[i + 1] - ro[i] <= widest and meta >> 8 <= GEN_HELD
            for u in range(meta >> 8):
                w, value = blob[held_at + u * n + a + k], blob[held_at + (GEN_HELD + u) * n + a + k]
                j, flip = row_of[w & 0x3FF], bool(value >> 31)
                put((w >> 24) * GEN_PART + k, i, j, value & 0x7FFFFFFF, not flip)
                t = (w >> 10) & 0x3FFF
                assert (t == 0x3FFF) == ((w & 0x3FF) >= GEN_PART)
                if t != 0x3FFF:
                    assert t % GEN_PART == w & 0x3FF
                    put(t, j, i, value & 0x7FFFFFFF, flip)
        want = {}
        for k in range(own):
            i = row_of[k]
            for t, c in enumerate(range(ro[i], ro[i + 1])):
                j = int(ci[c])
                want[t * GEN_PART + k] = (i, j, bs[c] if j > i else -1 - bs[c], j > i)
        assert got == want


def test_pattern_outside_the_limits_has_no_plan():
    """A vertex coupled to more rows than a thread holds: no plan."""
    n = 40
    rows = np.r_[np.zeros(n - 1, np.int32), np.arange(1, n, dtype=np.int32)]
    cols = np.r_[np.arange(1, n, dtype=np.int32), np.zeros(n - 1, np.int32)]
    ro, ci = chysx.topology.build_pattern(n, rows, cols)
    bs, _ = _slots(n, ro, ci)
    assert chysx.topology.resident_plan(n, ro, ci, bs, 256) is None
    assert chysx.topology.resident_plan(n, ro, ci, bs, 256, general=True) is None


@pytest.mark.parametrize("nx,ny", [(2, 2), (8, 8), (23, 22), (33, 31), (65, 66)])
@pytest.mark.parametrize("part_rows", [256, 512])
def test_half_sheet_is_the_sheet_with_smaller_numbers(nx, ny, part_rows):
    """At a capacity of 512 rows a plan is the one at 1024 rows with local
    indices and product slots numbered by the smaller capacity."""
    n, half = nx * ny, 512
    ro, ci = _pattern(nx, ny)
    bs, _ = _slots(n, ro, ci)
    full = chysx.topology.resident_plan(n, ro, ci, bs, part_rows)
    got = chysx.topology.resident_plan(n, ro, ci, bs, part_rows, capacity=half)
    assert (got["order"] == full["order"]).all() and got["parts"] == full["parts"] and got["exports"] == full["exports"]
    want, blob, parts = full["blob"].astype(np.int64), got["blob"].astype(np.int64), full["parts"]

    def renumber(w):
        local, slot = w & 0xFFFF, w >> 16
        local = np.where(local >= PART, local - PART + half, local)
        return local | np.where(slot == 0xFFFF, slot, slot // PART * half + slot % PART) << 16

    # held words of the blocks that are there, and the second words of the ghost lists
    held_at, meta = 8 * parts + 3 * n, want[8 * parts + n:8 * parts + 2 * n]
    for u in range(HELD):
        at = held_at + u * n + np.flatnonzero(meta >> 8 > u)
        want[at] = renumber(want[at])
    for q in range(parts):
        g, at = want[8 * q + 3:8 * q + 5]
        want[at + 1:at + 2 * g:2] = renumber(want[at + 1:at + 2 * g:2])
    assert (blob == want).all()


def test_an_awaited_tag_is_never_the_old_one():
    """Slots keep what was last written: until a word of an exchange arrives,
    its reader finds an older one there, whose tag has to differ.  The
    two-reduction solver sends halo rows with the set-up's residual, with
    every iteration's sigma (not with its rho) and, after `inner` iterations,
    with the refinement's x and residual; tags repeat after 256 numbers."""
    for inner in [*range(520), 5118, 5119, 5120]:
        with_rows = [True] + [True, False] * inner + [True, True] + [True, False] * 3
        words = {}
        for exchange in chysx.topology.resident_exchanges(9, with_rows):
            for kind, word in zip(("sums", "rows"), exchange):
                if word is not None:
                    slot, tag = word
                    assert slot in (0, 1) and tag >> 8 == 9
                    assert words.get((kind, slot)) != tag, (inner, kind)
                    words[kind, slot] = tag


def _resets(case, rng):
    """Whether the resident kernel runs after each reset of the control words."""
    if case == "steps":
        return [True] * 1200
    if case == "assemble and solve":
        return [False, True] * 600 + [False, False, True] * 400
    if case == "streaming steps between":
        return [True] * 10 + ([False] * 254 + [True]) * 5 + ([False] * 600 + [True]) * 3
    return [bool(x) for x in rng.random(5000) < rng.choice([0.01, 0.3, 0.9])]


@pytest.mark.parametrize("case", ["steps", "assemble and solve", "streaming steps between", *range(12)])
def test_a_launch_number_comes_again_only_after_a_clear(case):
    """No launch of the resident kernel finds words of an earlier one under
    its own number, in whatever order assemblies, streaming solves and
    resident solves reset the control words."""
    runs = _resets(case, np.random.default_rng(0 if isinstance(case, str) else case))
    used = set()
    for resident, (number, clears) in zip(runs, chysx.topology.resident_launches(runs)):
        assert 1 <= number <= 255
        if resident:
            if clears:
                used.clear()
            assert number not in used
            used.add(number)
