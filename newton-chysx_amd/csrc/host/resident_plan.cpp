#include "resident_plan.h"

#include <algorithm>
#include <numeric>

#include "chysx_hip.h"

namespace chysx {
namespace engine {

namespace {

// Breadth-first distances over the pattern from `seed`; components that it
// does not reach follow behind it, each from its lowest row.
std::vector<int> distances(const topology::Pattern& p, int seed) {
    std::vector<int> d(static_cast<std::size_t>(p.n), -1), q;
    q.reserve(static_cast<std::size_t>(p.n));
    int base = 0, next = 0;
    for (std::size_t head = 0; static_cast<int>(q.size()) < p.n;) {
        d[seed] = base;
        q.push_back(seed);
        for (; head < q.size(); ++head) {
            const int r = q[head];
            for (int k = p.row_offsets[r]; k < p.row_offsets[r + 1]; ++k)
                if (d[p.col_indices[k]] < 0) {
                    d[p.col_indices[k]] = d[r] + 1;
                    q.push_back(p.col_indices[k]);
                }
        }
        base = d[q.back()] + 1;
        while (next < p.n && d[next] >= 0) ++next;
        seed = next;
    }
    return d;
}

// Two coordinates of every row.  A sheet numbered row by row (the first row
// without a block to its successor ends a mesh row, and so does every
// width-th one) has its grid coordinates; any other pattern the
// graph distances from two far-apart rows.
void coordinates(const topology::Pattern& p, std::vector<int>& x, std::vector<int>& y) {
    const int n = p.n;
    const auto linked = [&](int r) {
        const auto b = p.col_indices.begin() + p.row_offsets[r], e = p.col_indices.begin() + p.row_offsets[r + 1];
        return r + 1 < n && std::binary_search(b, e, r + 1);
    };
    int w = 0;
    while (w < n && linked(w)) ++w;
    ++w;
    bool sheet = w > 1 && n % w == 0;
    for (int r = 0; r < n && sheet; ++r) sheet = linked(r) == (r % w != w - 1);
    x.resize(static_cast<std::size_t>(n));
    y.resize(static_cast<std::size_t>(n));
    if (sheet) {
        for (int r = 0; r < n; ++r) {
            x[r] = r % w;
            y[r] = r / w;
        }
        return;
    }
    const auto far = [](const std::vector<int>& d) {
        return static_cast<int>(std::max_element(d.begin(), d.end()) - d.begin());
    };
    const int a = far(distances(p, 0));
    x = distances(p, a);
    const std::vector<int> c = distances(p, far(x));
    std::vector<int> s(static_cast<std::size_t>(n));
    for (int r = 0; r < n; ++r) s[r] = x[r] + c[r] - std::abs(x[r] - c[r]);
    y = distances(p, far(s));
}

}  // namespace

std::vector<int> resident_order(const topology::Pattern& p) {
    std::vector<int> order(static_cast<std::size_t>(p.n)), x, y;
    std::iota(order.begin(), order.end(), 0);
    if (p.n <= CHX_RES_LEAF) return order;
    coordinates(p, x, y);
    constexpr int kMost = CHX_RES_PART_MAX / CHX_RES_LEAF;  // leaves of the largest part
    struct Range {
        int b, e;
    };
    std::vector<Range> todo{{0, p.n}};
    while (!todo.empty()) {
        const Range r = todo.back();
        todo.pop_back();
        const int leaves = (r.e - r.b + CHX_RES_LEAF - 1) / CHX_RES_LEAF;
        if (leaves <= 1) {
            std::sort(order.begin() + r.b, order.begin() + r.e);  // rows in memory order: coalesced loads
            continue;
        }
        // left half in whole largest parts, or below that in a power of two
        // of leaves, so parts of every size are runs of whole subtrees
        int left;
        if (leaves > kMost) {
            left = ((leaves + kMost - 1) / kMost / 2) * kMost;
        } else {
            left = 1;
            while (2 * left < leaves) left *= 2;
        }
        int x0 = x[order[r.b]], x1 = x0, y0 = y[order[r.b]], y1 = y0;
        for (int k = r.b; k < r.e; ++k) {
            const int i = order[k];
            x0 = std::min(x0, x[i]);
            x1 = std::max(x1, x[i]);
            y0 = std::min(y0, y[i]);
            y1 = std::max(y1, y[i]);
        }
        const std::vector<int>&major = x1 - x0 > y1 - y0 ? x : y, &minor = x1 - x0 > y1 - y0 ? y : x;
        const int mid = r.b + left * CHX_RES_LEAF;
        std::nth_element(order.begin() + r.b, order.begin() + mid, order.begin() + r.e, [&](int i, int j) {
            if (major[i] != major[j]) return major[i] < major[j];
            if (minor[i] != minor[j]) return minor[i] < minor[j];
            return i < j;
        });
        todo.push_back({r.b, mid});
        todo.push_back({mid, r.e});
    }
    return order;
}

namespace {

// Halo rows, ghost blocks and exports of both forms.  Planes: words per
// position behind the first three (row, meta, export).  For every part,
// row(k, i) writes position k's planes and meta, and may add ghost blocks.
struct Builder {
    const topology::Pattern& p;
    const std::vector<int>& order;
    int part_rows, capacity, planes;
    std::vector<int> pos, local;
    std::vector<std::uint32_t> blob, halos, ghosts;
    std::size_t N, rows_at, meta_at, exp_at, held_at;
    int parts, exports = 0;
    int a = 0, b = 0, widest = 0;  // the part at hand

    Builder(const topology::Pattern& pat, const std::vector<int>& ord, int rows, int cap, int n_planes)
        : p(pat), order(ord), part_rows(rows), capacity(cap), planes(n_planes), N(static_cast<std::size_t>(pat.n)) {
        parts = (p.n + rows - 1) / rows;
        pos.resize(N);
        local.assign(N, 0);
        for (int k = 0; k < p.n; ++k) pos[order[k]] = k;
        rows_at = 8u * static_cast<std::size_t>(parts);
        meta_at = rows_at + N;
        exp_at = meta_at + N;
        held_at = exp_at + N;
        blob.assign(held_at + static_cast<std::size_t>(planes) * N, 0u);
    }
    bool own(int j) const { return pos[j] >= a && pos[j] < b; }
    std::uint32_t local_of(int j) const { return static_cast<std::uint32_t>(own(j) ? pos[j] - a : local[j]); }
    std::uint32_t& plane(int u, int k) {
        return blob[held_at + static_cast<std::size_t>(u) * N + static_cast<std::size_t>(k)];
    }
    void ghost(std::uint32_t value, std::uint32_t word) {
        ghosts.push_back(value);
        ghosts.push_back(word);
    }
    template <class Row>
    bool build(Row row) {
        const auto& ro = p.row_offsets;
        const auto& ci = p.col_indices;
        // exported rows, numbered part by part in canonical order
        std::vector<std::uint32_t> exp(N, CHX_RES_NONE);
        for (int k = 0; k < p.n; ++k)
            for (int c = ro[order[k]]; c < ro[order[k] + 1]; ++c)
                if (pos[ci[c]] / part_rows != k / part_rows) exp[ci[c]] = 0u;
        for (int k = 0; k < p.n; ++k)
            if (exp[order[k]] == 0u) exp[order[k]] = static_cast<std::uint32_t>(exports++);
        std::vector<int> stamp(N, -1), halo;
        for (int q = 0; q < parts; ++q) {
            a = q * part_rows;
            b = std::min(p.n, a + part_rows);
            widest = 0;
            halo.clear();
            for (int k = a; k < b; ++k) {
                const int i = order[k];
                widest = std::max(widest, ro[i + 1] - ro[i]);
                for (int c = ro[i]; c < ro[i + 1]; ++c)
                    if (!own(ci[c]) && stamp[ci[c]] != q) {
                        stamp[ci[c]] = q;
                        halo.push_back(ci[c]);
                    }
            }
            if (halo.size() > CHX_RES_HALO_MAX) return false;
            std::sort(halo.begin(), halo.end(), [&](int i, int j) { return pos[i] < pos[j]; });
            for (std::size_t h = 0; h < halo.size(); ++h) local[halo[h]] = capacity + static_cast<int>(h);
            const std::size_t ghost0 = ghosts.size() / 2;
            for (int k = a; k < b; ++k) {
                const int i = order[k];
                blob[rows_at + static_cast<std::size_t>(k)] = static_cast<std::uint32_t>(i);
                blob[exp_at + static_cast<std::size_t>(k)] = exp[i];
                blob[meta_at + static_cast<std::size_t>(k)] = row(k, i);
            }
            const std::size_t n_ghosts = ghosts.size() / 2 - ghost0;
            if (n_ghosts > CHX_RES_GHOST_MAX) return false;
            std::uint32_t* H = blob.data() + 8 * static_cast<std::size_t>(q);
            H[0] = static_cast<std::uint32_t>(b - a);
            H[1] = static_cast<std::uint32_t>(halo.size());
            H[2] = static_cast<std::uint32_t>(halos.size());
            H[3] = static_cast<std::uint32_t>(n_ghosts);
            H[4] = static_cast<std::uint32_t>(2 * ghost0);
            H[5] = static_cast<std::uint32_t>(widest);
            for (int j : halo) {
                halos.push_back(static_cast<std::uint32_t>(j));
                halos.push_back(exp[j]);
            }
        }
        // the lists behind the planes, at absolute word offsets
        const std::size_t halo_at = blob.size(), ghost_at = halo_at + halos.size();
        if (ghost_at + ghosts.size() >= (std::size_t(1) << 30)) return false;
        for (int q = 0; q < parts; ++q) {
            blob[8 * static_cast<std::size_t>(q) + 2] += static_cast<std::uint32_t>(halo_at);
            blob[8 * static_cast<std::size_t>(q) + 4] += static_cast<std::uint32_t>(ghost_at);
        }
        blob.insert(blob.end(), halos.begin(), halos.end());
        blob.insert(blob.end(), ghosts.begin(), ghosts.end());
        return true;
    }
    ResidentPlan take() {
        ResidentPlan out;
        out.part_rows = part_rows;
        out.parts = parts;
        out.exports = exports;
        out.blob = std::move(blob);
        return out;
    }
};

}  // namespace

ResidentPlan resident_plan(const topology::Pattern& p, const std::vector<int>& block_slots,
                           const std::vector<int>& order, int part_rows, int capacity) {
    const int n = p.n;
    if (n <= 0 || part_rows > capacity || capacity > CHX_RES_PART_MAX) return {};
    const auto& ro = p.row_offsets;
    const auto& ci = p.col_indices;
    // lower[k]: place of upper block (i, j)'s transpose among row j's lower blocks
    std::vector<std::uint8_t> lower(ci.size(), 0), nl(static_cast<std::size_t>(n), 0);
    std::vector<int> up0(static_cast<std::size_t>(n));
    for (int i = 0; i < n; ++i) {
        int k = ro[i];
        while (k < ro[i + 1] && ci[k] < i) ++k;
        up0[i] = k;
        if (ro[i + 1] - k > CHX_RES_HELD || k - ro[i] > CHX_RES_HELD) return {};
        for (; k < ro[i + 1]; ++k) lower[k] = nl[ci[k]]++;
    }
    Builder B(p, order, part_rows, capacity, CHX_RES_HELD);
    const bool ok = B.build([&](int k, int i) {
        for (int c = ro[i]; c < up0[i]; ++c)  // blocks another part holds
            if (!B.own(ci[c]))
                B.ghost(static_cast<std::uint32_t>(-1 - block_slots[c]),
                        B.local_of(ci[c]) |
                            (static_cast<std::uint32_t>((c - ro[i]) * capacity + (k - B.a)) << 16));
        for (int c = up0[i]; c < ro[i + 1]; ++c) {
            const std::uint32_t lj = B.local_of(ci[c]);
            const std::uint32_t target =
                B.own(ci[c]) ? static_cast<std::uint32_t>(lower[c] * capacity) + lj : 0xffffu;
            B.plane(c - up0[i], k) = lj | (target << 16);
        }
        return static_cast<std::uint32_t>((up0[i] - ro[i]) | ((ro[i + 1] - up0[i]) << 8));
    });
    return ok ? B.take() : ResidentPlan{};
}

ResidentPlan resident_plan_general(const topology::Pattern& p, const std::vector<int>& block_slots,
                                   const std::vector<int>& order, int part_rows) {
    const int n = p.n;
    if (n <= 0 || part_rows > CHX_RES_GEN_PART) return {};
    const auto& ro = p.row_offsets;
    const auto& ci = p.col_indices;
    // mirror[k]: CSR index of block k's transpose
    std::vector<int> mirror(ci.size()), at(ro.begin(), ro.end() - 1);
    for (int i = 0; i < n; ++i) {
        if (ro[i + 1] - ro[i] > CHX_RES_GEN_WIDTH) return {};
        for (int k = ro[i]; k < ro[i + 1]; ++k) mirror[k] = at[ci[k]]++;
    }
    // Every pair's block is held by one of its rows, half of a row's blocks
    // (rounded up at most): walk trails over unused pairs, each held by the
    // row the trail leaves.  Trails from rows with an odd number of pairs
    // first: they end at such rows, and the rest close.
    std::vector<std::uint8_t> held(ci.size(), 0), used(ci.size(), 0);
    std::vector<int> next(ro.begin(), ro.end() - 1);
    const auto walk = [&](int i) {
        for (;;) {
            int& k = next[i];
            while (k < ro[i + 1] && used[k]) ++k;
            if (k == ro[i + 1]) return;
            held[k] = used[k] = used[mirror[k]] = 1;
            i = ci[k];
        }
    };
    for (int i = 0; i < n; ++i)
        if ((ro[i + 1] - ro[i]) % 2 != 0) {
            int unused = 0;
            for (int k = ro[i]; k < ro[i + 1]; ++k) unused += used[k] ? 0 : 1;
            if (unused % 2 != 0) walk(i);
        }
    for (int i = 0; i < n; ++i) walk(i);
    static_assert(CHX_RES_GEN_HELD * 2 >= CHX_RES_GEN_WIDTH, "half of the widest row");
    Builder B(p, order, part_rows, CHX_RES_GEN_PART, 2 * CHX_RES_GEN_HELD);
    const bool ok = B.build([&](int k, int i) {
        int u = 0;
        for (int c = ro[i]; c < ro[i + 1]; ++c) {
            const int j = ci[c];
            const std::uint32_t value = static_cast<std::uint32_t>(block_slots[c] < 0 ? -1 - block_slots[c] : block_slots[c]);
            const std::uint32_t place = static_cast<std::uint32_t>(c - ro[i]);
            if (held[c]) {
                const std::uint32_t lj = B.local_of(j);
                const std::uint32_t target =
                    B.own(j) ? static_cast<std::uint32_t>(mirror[c] - ro[j]) * CHX_RES_GEN_PART + lj : 0x3fffu;
                B.plane(u, k) = lj | (target << 10) | (place << 24);
                B.plane(CHX_RES_GEN_HELD + u, k) = value | (j < i ? 0x80000000u : 0u);
                ++u;
            } else if (!B.own(j)) {
                B.ghost(value | (j > i ? 0x80000000u : 0u),
                        B.local_of(j) | ((place * CHX_RES_GEN_PART + static_cast<std::uint32_t>(k - B.a)) << 16));
            }
        }
        return static_cast<std::uint32_t>((ro[i + 1] - ro[i]) | (u << 8));
    });
    return ok ? B.take() : ResidentPlan{};
}

ResidentPlan resident_plan_rows(const topology::Pattern& p, const std::vector<int>& order, int part_rows) {
    if (p.n <= 0 || part_rows > CHX_RES_GEN_PART) return {};
    const auto& ro = p.row_offsets;
    for (int i = 0; i < p.n; ++i)
        if (ro[i + 1] - ro[i] > CHX_RES_ROW_WIDTH) return {};
    Builder B(p, order, part_rows, CHX_RES_GEN_PART, CHX_RES_ROW_WIDTH);
    const bool ok = B.build([&](int k, int i) {
        for (int c = ro[i]; c < ro[i + 1]; ++c) B.plane(c - ro[i], k) = B.local_of(p.col_indices[c]);
        return static_cast<std::uint32_t>((ro[i + 1] - ro[i]) << 8);
    });
    return ok ? B.take() : ResidentPlan{};
}

int resident_part_rows(const std::vector<int>& rows, int largest) {
    constexpr long kWorkgroups = 256;
    for (int pr = 256; pr <= largest; pr *= 2) {
        long parts = 0, most = 0;
        for (int n : rows) {
            const long q = n <= largest ? 1 : (n + pr - 1) / pr;
            parts += q;
            most = std::max(most, q);
        }
        if (parts <= kWorkgroups) return rows.size() == 1 && rows[0] <= largest ? largest : pr;
        if (pr == largest && most <= kWorkgroups) return pr;
    }
    return 0;
}

std::vector<ResidentChoice> resident_choices(const std::vector<int>& rows, bool bf16) {
    std::vector<ResidentChoice> out;
    const int half = resident_part_rows(rows, CHX_RES_GEN_PART), full = resident_part_rows(rows, CHX_RES_PART_MAX);
    if (bf16 && half > 0) out.push_back({CHX_RES_FORM_HALF, half});
    if (!bf16 && full > 0) out.push_back({CHX_RES_FORM_SHEET, full});
    if (half > 0) out.push_back({CHX_RES_FORM_GENERAL, half});
    return out;
}

}  // namespace engine
}  // namespace chysx
