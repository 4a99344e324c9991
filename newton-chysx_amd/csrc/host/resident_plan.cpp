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

ResidentPlan resident_plan(const topology::Pattern& p, const std::vector<int>& block_slots,
                           const std::vector<int>& order, int part_rows) {
    ResidentPlan out;
    const int n = p.n;
    if (n <= 0) return out;
    const auto& ro = p.row_offsets;
    const auto& ci = p.col_indices;
    const int parts = (n + part_rows - 1) / part_rows;
    std::vector<int> pos(static_cast<std::size_t>(n));
    for (int k = 0; k < n; ++k) pos[order[k]] = k;
    // lower[k]: place of upper block (i, j)'s transpose among row j's lower blocks
    std::vector<std::uint8_t> lower(ci.size(), 0), nl(static_cast<std::size_t>(n), 0);
    std::vector<int> up0(static_cast<std::size_t>(n));
    for (int i = 0; i < n; ++i) {
        int k = ro[i];
        while (k < ro[i + 1] && ci[k] < i) ++k;
        up0[i] = k;
        if (ro[i + 1] - k > CHX_RES_HELD || k - ro[i] > CHX_RES_HELD) return out;
        for (; k < ro[i + 1]; ++k) lower[k] = nl[ci[k]]++;
    }
    const std::size_t N = static_cast<std::size_t>(n);
    const std::size_t rows_at = 8u * static_cast<std::size_t>(parts), meta_at = rows_at + N, exp_at = meta_at + N,
                      held_at = exp_at + N, lists_at = held_at + CHX_RES_HELD * N;
    std::vector<std::uint32_t> B(lists_at, 0u);
    std::vector<std::uint32_t> halo_all, ghost_all;
    std::vector<int> stamp(N, -1), local(N, 0);
    // exported rows, numbered part by part in canonical order
    std::vector<std::uint8_t> shared(N, 0);
    for (int i = 0; i < n; ++i)
        for (int k = up0[i]; k < ro[i + 1]; ++k)
            if (pos[i] / part_rows != pos[ci[k]] / part_rows) shared[i] = shared[ci[k]] = 1;
    std::vector<std::uint32_t> exp(N, CHX_RES_NONE);
    int exports = 0;
    for (int k = 0; k < n; ++k)
        if (shared[order[k]]) exp[order[k]] = static_cast<std::uint32_t>(exports++);
    std::vector<int> halo;
    for (int q = 0; q < parts; ++q) {
        const int a = q * part_rows, b = std::min(n, a + part_rows);
        halo.clear();
        for (int k = a; k < b; ++k) {
            const int i = order[k];
            for (int c = ro[i]; c < ro[i + 1]; ++c) {
                const int j = ci[c];
                if (pos[j] >= a && pos[j] < b) continue;
                if (stamp[j] != q) {
                    stamp[j] = q;
                    halo.push_back(j);
                }
            }
        }
        std::sort(halo.begin(), halo.end(), [&](int i, int j) { return pos[i] < pos[j]; });
        if (halo.size() > CHX_RES_HALO_MAX) return out;
        for (std::size_t h = 0; h < halo.size(); ++h) local[halo[h]] = CHX_RES_PART_MAX + static_cast<int>(h);
        const std::size_t ghost0 = ghost_all.size() / 2;
        for (int k = a; k < b; ++k) {
            const int i = order[k];
            const std::size_t K = static_cast<std::size_t>(k);
            B[rows_at + K] = static_cast<std::uint32_t>(i);
            B[meta_at + K] = static_cast<std::uint32_t>((up0[i] - ro[i]) | ((ro[i + 1] - up0[i]) << 4));
            B[exp_at + K] = exp[i];
            for (int c = ro[i]; c < up0[i]; ++c) {  // blocks another part holds
                const int j = ci[c];
                if (pos[j] >= a && pos[j] < b) continue;
                ghost_all.push_back(static_cast<std::uint32_t>(-1 - block_slots[c]));
                ghost_all.push_back(static_cast<std::uint32_t>(local[j]) |
                                    (static_cast<std::uint32_t>((c - ro[i]) * CHX_RES_PART_MAX + (k - a)) << 16));
            }
            for (int c = up0[i]; c < ro[i + 1]; ++c) {
                const int j = ci[c];
                const bool own = pos[j] >= a && pos[j] < b;
                const std::uint32_t lj = static_cast<std::uint32_t>(own ? pos[j] - a : local[j]);
                const std::uint32_t target =
                    own ? static_cast<std::uint32_t>(lower[c]) * CHX_RES_PART_MAX + lj : 0xffffu;
                B[held_at + static_cast<std::size_t>(c - up0[i]) * N + K] = lj | (target << 16);
            }
        }
        const std::size_t ghosts = ghost_all.size() / 2 - ghost0;
        if (ghosts > CHX_RES_GHOST_MAX) return out;
        std::uint32_t* H = B.data() + 8 * static_cast<std::size_t>(q);
        H[0] = static_cast<std::uint32_t>(b - a);
        H[1] = static_cast<std::uint32_t>(halo.size());
        H[2] = static_cast<std::uint32_t>(halo_all.size() / 2);
        H[3] = static_cast<std::uint32_t>(ghosts);
        H[4] = static_cast<std::uint32_t>(ghost0);
        for (int j : halo) {
            halo_all.push_back(static_cast<std::uint32_t>(j));
            halo_all.push_back(exp[j]);
        }
    }
    // absolute word offsets of the lists
    const std::size_t halo_at = lists_at, ghost_at = halo_at + halo_all.size();
    if (ghost_at + ghost_all.size() >= (std::size_t(1) << 30)) return out;
    for (int q = 0; q < parts; ++q) {
        std::uint32_t* H = B.data() + 8 * static_cast<std::size_t>(q);
        H[2] = static_cast<std::uint32_t>(halo_at + 2 * H[2]);
        H[4] = static_cast<std::uint32_t>(ghost_at + 2 * H[4]);
    }
    B.insert(B.end(), halo_all.begin(), halo_all.end());
    B.insert(B.end(), ghost_all.begin(), ghost_all.end());
    out.part_rows = part_rows;
    out.parts = parts;
    out.exports = exports;
    out.blob = std::move(B);
    return out;
}

}  // namespace engine
}  // namespace chysx
