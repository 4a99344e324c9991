// Resident block-Jacobi PCG of the FP32 cloth instances: a workgroup keeps
// its part of an instance's matrix in registers and its vectors in registers
// and LDS from the first product to the last, so an iteration reads no
// matrix from memory.  What crosses workgroups in an iteration is the halo
// rows of q = A p and five partial sums, in one hop.
//
// Why: streaming the matrix every iteration cost 20.5 ms per solve of the
// 512-cloth batch (2.08 M rows, 66 iterations on average), set by the
// L1-L2 stream, and 19 us per iteration of one 256x256 cloth, set by the
// grid barrier's cache write-backs.  A CU has 512 KB of registers: 1024 rows
// of a sheet's matrix (six upper blocks a row) take 221 KB, so 256 CUs hold
// 262,144 rows, and the instances of a batch are independent: they are
// solved one after another by gangs of ceil(rows / 1024) workgroups.
//
// Arithmetic: the single-barrier recurrence of pcg1_kernel (chx_step.hip),
// operation for operation; every row sums its diagonal product, its lower
// blocks and its upper blocks in column order.  A row's upper blocks are in
// its thread's registers: it forms A_ij p_j for itself and A_ij^T p_i for
// row j, which it leaves in row j's product slot in LDS.  Blocks between
// parts are held by both (the second copy is a "ghost block").  Halo rows'
// r, z and p are kept by every part that reads them, updated from the
// published q with the same operations as by their owner.
//
// Inner products: FP64, one sum per 64-row leaf (a wavefront), combined over
// the leaves of the instance by a fixed binary tree that does not depend on
// how many leaves a part has: the same bits for every part size and gang.
//
// Exchange: 64-bit words {value, tag}, the tag naming launch and phase, so a
// reader needs no ordering between words and no cache maintenance: it reads
// a word until its tag is the awaited one.  Words alternate between two
// slots; slot t is rewritten in phase t + 2, which its writer enters only
// after every part's sums of phase t + 1, sent after their reads of phase t.
#include <algorithm>
#include <mutex>

#include "chx_pcg.h"
#include "chx_resident.h"

namespace chx {
namespace {

constexpr int kThreads = 512;  // two waves per SIMD with 256 VGPRs each
constexpr int kWaves = kThreads / kWave;
constexpr int kLeaves = CHX_RES_PART_MAX / CHX_RES_LEAF;
// The two forms of a plan (chysx_hip.h).  Sheet: a row's lower blocks come
// through product slots and are summed before the upper ones that its thread
// holds, which is column order.  General: all of a row's products go through
// its slots, in column order; twice the slots and wider rows, so half the
// rows.
template <bool GEN>
struct Form {
    static constexpr unsigned kRows = GEN ? CHX_RES_GEN_PART : CHX_RES_PART_MAX;
    static constexpr int kSlots = kRows / kThreads;  // own rows per thread
    static constexpr int kHeld = GEN ? CHX_RES_GEN_HELD : CHX_RES_HELD;
    static constexpr unsigned kPlaces = GEN ? CHX_RES_GEN_WIDTH : CHX_RES_HELD;  // product slots per row
    static constexpr unsigned kNoSlot = GEN ? 0x3fffu : 0xffffu;
    static constexpr unsigned kSpare = kPlaces * kRows;  // first of the unread product slots
    // fields of a held block's word
    static __device__ __forceinline__ unsigned src(unsigned w) { return w & (GEN ? 0x3ffu : 0xffffu); }
    static __device__ __forceinline__ unsigned slot(unsigned w) { return GEN ? (w >> 10) & 0x3fffu : w >> 16; }
    static __device__ __forceinline__ unsigned word(unsigned s, unsigned t) { return s | (t << (GEN ? 10 : 16)); }
};
static_assert(Form<true>::kSpare + kWave <= Form<true>::kNoSlot && Form<false>::kSpare + kWave <= Form<false>::kNoSlot &&
                  Form<true>::kRows + CHX_RES_HALO_MAX <= 1024,
              "word fields");
constexpr int kSums = 5;  // rho, sigma, delta, gamma, ||r||^2 (set-up: ||b||^2 in place of sigma)
constexpr int kMaxParts = 256;
constexpr unsigned kFan = 16;    // parts per group and groups, above 64 parts
constexpr unsigned kCopies = 16;  // copies of the groups' sums
static_assert(kFan * kFan >= kMaxParts && 2 * kCopies <= 64, "two levels");
constexpr unsigned kExit = 0xffffffu;  // mailbox item: nothing left
static_assert(CHX_RES_LEAF == kWave && Form<false>::kSlots == 2 && Form<true>::kSlots == 1 && kLeaves == 2 * kWaves,
              "a leaf per wave and slot");
static_assert(CHX_RES_HALO_MAX <= kThreads && CHX_RES_GHOST_MAX <= kThreads, "one halo row and ghost block a thread");

typedef unsigned long long u64;

__device__ __forceinline__ u64 ld64(const u64* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st64(u64* p, u64 v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 tagged(unsigned v, unsigned tag) { return (u64(tag) << 32) | v; }

// LDS triples as one 96-bit access.
typedef float v3f __attribute__((ext_vector_type(3), aligned(4)));
__device__ __forceinline__ f3 lds_ld(const f3* p) {
    const v3f v = *reinterpret_cast<const v3f*>(p);
    return {v.x, v.y, v.z};
}
__device__ __forceinline__ void lds_st(f3* p, f3 v) {
    v3f w;
    w.x = v.x;
    w.y = v.y;
    w.z = v.z;
    *reinterpret_cast<v3f*>(p) = w;
}
// Keeps a value that the loop does not change from being re-derived ahead of
// the loop (addresses and masks of every block would not fit the registers).
__device__ __forceinline__ unsigned opaque(unsigned v) {
    asm volatile("" : "+v"(v));
    return v;
}

template <bool GEN>
struct ResLds {
    // products by target row, then one unread slot per lane for blocks
    // without a target
    f3 prod[Form<GEN>::kSpare + kWave];
    f3 p[Form<GEN>::kRows + CHX_RES_HALO_MAX];     // source vector: own rows, halo rows
    float diag[6][Form<GEN>::kRows];
    f3 x[Form<GEN>::kRows];
    float ghost[9][CHX_RES_GHOST_MAX];
    double leaf[kLeaves][kSums];
    double tot[8];
    int bad;         // a wait gave up
    unsigned mail;   // mailbox word of the workgroup
};

// Bounded wait of one lane: true while it may go on.  After the bound the
// solve is aborted for every workgroup (the report of grid_sync).
struct Watch {
    const Barrier& bar;
    u64 t0;
    unsigned polls = 0;
    __device__ explicit Watch(const Barrier& b) : bar(b), t0(__builtin_amdgcn_s_memrealtime()) {}
    __device__ bool again(u64* progress, unsigned& seen) {
        unsigned* sync = bar.sync;
        if ((++polls & 15u) == 0u && ld_relaxed(&sync[SYNC_ABORT]) != 0u) return false;
        if (__builtin_amdgcn_s_memrealtime() - t0 <= bar.ticks) return true;
        if (progress != nullptr) {
            const unsigned now = unsigned(ld64(progress));
            if (now != seen) {
                seen = now;
                t0 = __builtin_amdgcn_s_memrealtime();
                return true;
            }
        }
        st_relaxed(&sync[SYNC_SEEN], 0u);
        st_relaxed(&sync[SYNC_WAITING], 1u);
        st_relaxed(&sync[SYNC_GRID], gridDim.x);
        st_relaxed(&sync[SYNC_ABORT], 1u);
        st_relaxed(&sync[SYNC_STATUS], 1u);
        if (bar.status_host != nullptr)
            __hip_atomic_store(bar.status_host, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        return false;
    }
};

// N tagged words from p on, read until every tag is the awaited one; false:
// the wait was given up.
template <int N>
__device__ __forceinline__ bool await(const u64* p, unsigned tag, unsigned (&v)[N], const Barrier& bar) {
    u64 w[N];
    auto read = [&] {
        bool ok = true;
#pragma unroll
        for (int k = 0; k < N; ++k) w[k] = ld64(p + k);
#pragma unroll
        for (int k = 0; k < N; ++k) ok = ok && unsigned(w[k] >> 32) == tag;
        return ok;
    };
    if (!read()) {
        Watch watch(bar);
        unsigned seen = 0;
        do {
            if (!watch.again(nullptr, seen)) return false;
        } while (!read());
    }
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = unsigned(w[k]);
    return true;
}
__device__ __forceinline__ void transpose9(float (&m)[9]) {
    const float a = m[1], b = m[2], c = m[5];
    m[1] = m[3];
    m[2] = m[6];
    m[5] = m[7];
    m[3] = a;
    m[6] = b;
    m[7] = c;
}
__device__ __forceinline__ f3 mv9t(const float (&m)[9], f3 v) {
    const float b[9] = {m[0], m[3], m[6], m[1], m[4], m[7], m[2], m[5], m[8]};
    return mv9(b, v);
}
__device__ __forceinline__ f3 mv_sym(const float (&u)[6], f3 v) {
    const float a[9] = {u[0], u[1], u[2], u[1], u[3], u[4], u[2], u[4], u[5]};
    return mv9(a, v);
}
__device__ __forceinline__ void inverse_sym(const float (&u)[6], float (&mi)[6], float (&full)[9]) {
    const float a[9] = {u[0], u[1], u[2], u[1], u[3], u[4], u[2], u[4], u[5]};
    inverse9(a, full);
#pragma unroll
    for (unsigned q = 0; q < 6; ++q) mi[q] = full[sym6_pos(q)];
}
__device__ __forceinline__ void ld6u(gp<const float> m, unsigned i, float (&u)[6]) {
#pragma unroll
    for (unsigned q = 0; q < 6; q += 2) ld_pair(m, bp6(q, i), u[q], u[q + 1]);
}
__device__ __forceinline__ f3 axpy(float a, f3 x, f3 y) { return mk(fmaf(a, x.x, y.x), fmaf(a, x.y, y.y), fmaf(a, x.z, y.z)); }

// The wave's two leaf sums of kSums values into S.leaf.  Halving butterfly:
// each step adds lane pairs and packs two values into the two halves of the
// pairs, so five values of two leaves take 14 FP64 adds instead of 60.
template <int CTRL>
__device__ __forceinline__ double dpp64(double v) {
    const u64 b = u64(__double_as_longlong(v));
    const unsigned lo = unsigned(__builtin_amdgcn_mov_dpp(int(unsigned(b)), CTRL, 0xf, 0xf, true));
    const unsigned hi = unsigned(__builtin_amdgcn_mov_dpp(int(unsigned(b >> 32)), CTRL, 0xf, 0xf, true));
    return __longlong_as_double((long long)((u64(hi) << 32) | lo));
}
constexpr int kRor8 = 0x128, kHalfMirror = 0x141, kXor2 = 0x4e, kXor1 = 0xb1;  // DPP controls
typedef unsigned v2u __attribute__((ext_vector_type(2)));
// lanes of half 0: a summed over the pairs; of half 1: b
__device__ __forceinline__ double fold32(double a, double b) {
    const u64 x = u64(__double_as_longlong(a)), y = u64(__double_as_longlong(b));
    const v2u lo = __builtin_amdgcn_permlane32_swap(unsigned(x), unsigned(y), false, false);
    const v2u hi = __builtin_amdgcn_permlane32_swap(unsigned(x >> 32), unsigned(y >> 32), false, false);
    return __longlong_as_double((long long)((u64(hi.x) << 32) | lo.x)) +
           __longlong_as_double((long long)((u64(hi.y) << 32) | lo.y));
}
__device__ __forceinline__ double fold16(double a, double b) {
    const u64 x = u64(__double_as_longlong(a)), y = u64(__double_as_longlong(b));
    const v2u lo = __builtin_amdgcn_permlane16_swap(unsigned(x), unsigned(y), false, false);
    const v2u hi = __builtin_amdgcn_permlane16_swap(unsigned(x >> 32), unsigned(y >> 32), false, false);
    return __longlong_as_double((long long)((u64(hi.x) << 32) | lo.x)) +
           __longlong_as_double((long long)((u64(hi.y) << 32) | lo.y));
}
__device__ __forceinline__ double fold8(double a, double b, unsigned lane) {
    const bool up = (lane & 8u) != 0u;
    return (up ? b : a) + dpp64<kRor8>(up ? a : b);
}
__device__ __forceinline__ void leaf_sums(const double (&a)[kSums], const double (&b)[kSums],
                                          double (&leaf)[kLeaves][kSums], unsigned wave, unsigned lane) {
    double v[kSums];
#pragma unroll
    for (int k = 0; k < kSums; ++k) v[k] = fold32(a[k], b[k]);  // half h: leaf of slot h
    // rows (16 lanes) 2h, 2h + 1 of half h: values 0 | 1, 2 | 3, 4 | 4
    const double x = fold16(v[0], v[1]), y = fold16(v[2], v[3]), z = fold16(v[4], v[4]);
    double w0 = fold8(x, y, lane);             // half-rows: values 0 2 | 1 3
    double w1 = z + dpp64<kRor8>(z);           // value 4 everywhere
    w0 += dpp64<kHalfMirror>(w0);
    w1 += dpp64<kHalfMirror>(w1);
    w0 += dpp64<kXor2>(w0);
    w1 += dpp64<kXor2>(w1);
    w0 += dpp64<kXor1>(w0);
    w1 += dpp64<kXor1>(w1);
    double(&out)[kSums] = leaf[(lane >> 5) * kWaves + wave];
    const unsigned place = lane & 31u;
    if ((place & 7u) == 0u) out[(place >> 4) + ((place & 8u) >> 2)] = w0;
    if (place == 1u) out[4] = w1;
}

// Solves instance `inst` together with the workgroups that hold its other
// parts; this one holds part `part`.  False: aborted.
template <bool GEN>
__device__ __forceinline__ bool solve_part(const chx_cloth_batch& B, const Inst& I, int inst, int part, unsigned epoch,
                                           ResLds<GEN>& S, const Barrier& bar, int& trace_e) {
    using F = Form<GEN>;
    constexpr int kSlots = F::kSlots, kHeld = F::kHeld;
    constexpr unsigned kPart = F::kRows;
    const unsigned tid = threadIdx.x, lane = tid & (kWave - 1);
    const unsigned wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const gp<const unsigned> plan = I.res_plan;
    const unsigned n = unsigned(I.n_rows), parts = unsigned(I.res_parts);
    const gp<const unsigned> hdr = plan + 8 * part;
    const unsigned n_own = hdr[0], n_halo = hdr[1], halo_at = hdr[2], n_ghost = hdr[3], ghost_at = hdr[4], widest = hdr[5];
    const unsigned pos0 = unsigned(part) * unsigned(I.res_part_rows);
    const unsigned rows_at = 8u * parts, meta_at = rows_at + n, exp_at = meta_at + n, held_at = exp_at + n;
    // exchange areas: [2][kSums][parts] pairs of words, then [2][exports] rows of 3
    u64* const xsum = B.xbuf + I.res_xbase;
    u64* const xgroup = xsum + 4u * kSums * parts;  // [2][kCopies][kSums][kFan] pairs
    u64* const xrow = xgroup + (parts > unsigned(kWave) ? 4u * kCopies * kSums * kFan : 0u);
    const unsigned exports = unsigned(I.res_exports);
    auto tag_of = [&](int t) { return (epoch << 8) | (unsigned(t) & 255u); };
    auto sum_words = [&](int t, unsigned v, unsigned q) {
        return xsum + 2u * (((unsigned(t) & 1u) * kSums + v) * parts + q);
    };
    auto group_words = [&](int t, unsigned copy, unsigned v, unsigned g) {
        return xgroup + 2u * ((((unsigned(t) & 1u) * kCopies + copy) * kSums + v) * kFan + g);
    };
    auto row_words = [&](int t, unsigned e) { return xrow + 3ull * ((unsigned(t) & 1u) * exports + e); };

    auto send_row = [&](int t, unsigned e, f3 v) {
        u64* const w = row_words(t, e);
        st64(w, tagged(__float_as_uint(v.x), tag_of(t)));
        st64(w + 1, tagged(__float_as_uint(v.y), tag_of(t)));
        st64(w + 2, tagged(__float_as_uint(v.z), tag_of(t)));
    };

    // ---- load: own rows, ghost block, halo row ----
    unsigned lp[kSlots], ex[kSlots], holds[kSlots], word[kSlots][kHeld];
    bool live[kSlots], on[kSlots];  // this lane's row exists; this wave has a row
    float V[kSlots][kHeld][9], M[kSlots][6];
    f3 r[kSlots], p[kSlots], q[kSlots];
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
        lp[s] = (unsigned(s) * kWaves + wave) * kWave + lane;
        on[s] = (unsigned(s) * kWaves + wave) * kWave < n_own;
        live[s] = lp[s] < n_own;
        const unsigned K = pos0 + (live[s] ? lp[s] : 0u);
        ex[s] = CHX_RES_NONE;
        holds[s] = 0u;
        r[s] = p[s] = q[s] = mk(0.f, 0.f, 0.f);
        if (on[s]) {
            unsigned ns = 0u, nh = 0u;
            const unsigned row = ldx(plan, rows_at + K);
            const unsigned meta = ldx(plan, meta_at + K);
            if (live[s]) {
                ns = meta & 255u;
                nh = meta >> 8;
                ex[s] = ldx(plan, exp_at + K);
            }
            holds[s] = nh;
            const unsigned vs = unsigned(ldx(I.upper_offsets, row / CHX_SLICE_ROWS)) + row % CHX_SLICE_ROWS;
#pragma unroll
            for (int u = 0; u < kHeld; ++u) {
                // a block that is not there is zero, of the row itself
                const bool has = unsigned(u) < nh;
                unsigned w = has ? ldx(plan, held_at + unsigned(u) * n + K) : F::word(lp[s], F::kNoSlot);
                if (F::slot(w) == F::kNoSlot) w = (w & ~F::word(0u, F::kNoSlot)) | F::word(0u, F::kSpare + lane);
                word[s][u] = w;
#pragma unroll
                for (int c = 0; c < 9; ++c) V[s][u][c] = 0.0f;
                if (has) {
                    unsigned v = vs + unsigned(u) * CHX_SLICE_ROWS;
                    if (GEN) v = ldx(plan, held_at + unsigned(kHeld + u) * n + K);
                    ld9p(gp<const float>(I.values), v & 0x7fffffffu, V[s][u]);
                    if (GEN && (v >> 31) != 0u) transpose9(V[s][u]);
                }
            }
            // product slots that no block fills stay zero and are added like
            // the others
#pragma unroll
            for (unsigned u = 0; u < F::kPlaces; ++u)
                if (u >= ns) S.prod[u * kPart + lp[s]] = mk(0.f, 0.f, 0.f);
            float d[6], full[9];
            ld6u(gp<const float>(I.diag), row, d);
#pragma unroll
            for (int c = 0; c < 6; ++c) S.diag[c][lp[s]] = d[c];
            inverse_sym(d, M[s], full);
            if (live[s]) p[s] = ld3g(I.x, row);
            S.x[lp[s]] = p[s];
            S.p[lp[s]] = p[s];
        }
    }
    // ghost blocks and halo rows from the last thread down: in a small part
    // the first waves have the rows
    const unsigned rtid = unsigned(kThreads - 1) - tid;
    unsigned gword = 0;
    if (rtid < n_ghost) {
        const unsigned vs = ldx(plan, ghost_at + 2u * rtid);
        gword = ldx(plan, ghost_at + 2u * rtid + 1u);
        float g[9];
        ld9p(gp<const float>(I.values), vs & 0x7fffffffu, g);
        if (GEN && (vs >> 31) != 0u) transpose9(g);
#pragma unroll
        for (int c = 0; c < 9; ++c) S.ghost[c][rtid] = g[c];
    }
    float hM[6];
    f3 hr = mk(0.f, 0.f, 0.f);
    unsigned hex = 0;
    if (rtid < n_halo) {
        const unsigned hrow = ldx(plan, halo_at + 2u * rtid);
        hex = ldx(plan, halo_at + 2u * rtid + 1u);
        float d[6], full[9];
        ld6u(gp<const float>(I.diag), hrow, d);
        inverse_sym(d, hM, full);
        S.p[kPart + rtid] = ld3g(I.x, hrow);
    }
    if (tid == 0) S.bad = 0;
    if (tid < kLeaves * kSums) S.leaf[tid / kSums][tid % kSums] = 0.0;

    // A times the vector in S.p (own rows also in v); S.p and
    // S.prod are read until the next workgroup barrier.
    auto apply = [&](const f3 (&v)[kSlots], f3 (&out)[kSlots]) {
#pragma unroll
        for (int s = 0; s < kSlots; ++s)
            if (on[s]) {
#pragma unroll
                for (int u = 0; u < kHeld; ++u) lds_st(&S.prod[F::slot(opaque(word[s][u]))], mv9t(V[s][u], v[s]));
            }
        __syncthreads();
        if (rtid < n_ghost) {
            float g[9];
#pragma unroll
            for (int c = 0; c < 9; ++c) g[c] = S.ghost[c][rtid];
            lds_st(&S.prod[gword >> 16], mv9t(g, lds_ld(&S.p[gword & 0xffffu])));
        }
        if (GEN && on[0]) {
            f3 src[kHeld];
#pragma unroll
            for (int u = 0; u < kHeld; ++u) src[u] = lds_ld(&S.p[F::src(opaque(word[0][u]))]);
#pragma unroll
            for (int u = 0; u < kHeld; ++u)
                if (unsigned(u) < opaque(holds[0]))
                    lds_st(&S.prod[(opaque(word[0][u]) >> 24) * kPart + lp[0]], mv9(V[0][u], src[u]));
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < kSlots; ++s)
            if (on[s]) {
                float d[6];
#pragma unroll
                for (int c = 0; c < 6; ++c) d[c] = S.diag[c][lp[s]];
                if (GEN) {
                    f3 sum = mv_sym(d, v[s]);
#pragma unroll
                    for (unsigned t = 0; t < F::kPlaces; t += 4)
                        if (t < widest) {
                            f3 y[4];
#pragma unroll
                            for (unsigned u = 0; u < 4; ++u) y[u] = lds_ld(&S.prod[(t + u) * kPart + lp[s]]);
#pragma unroll
                            for (unsigned u = 0; u < 4; ++u) sum = add(sum, y[u]);
                        }
                    out[s] = sum;
                } else {
                    f3 low[kHeld], src[kHeld];
#pragma unroll
                    for (int u = 0; u < kHeld; ++u) src[u] = lds_ld(&S.p[F::src(opaque(word[s][u]))]);
#pragma unroll
                    for (int l = 0; l < kHeld; ++l) low[l] = lds_ld(&S.prod[unsigned(l) * kPart + lp[s]]);
                    f3 sum = mv_sym(d, v[s]);
#pragma unroll
                    for (int l = 0; l < kHeld; ++l) sum = add(sum, low[l]);
#pragma unroll
                    for (int u = 0; u < kHeld; ++u) sum = add(sum, mv9(V[s][u], src[u]));
                    out[s] = sum;
                }
            }
    };
    // Sums of phase t: per leaf, then over the part's leaves, sent to the gang.
    auto send_sums = [&](int t, double (&acc)[kSlots][kSums]) {
        const double none[kSums] = {0.0, 0.0, 0.0, 0.0, 0.0};
        if constexpr (kSlots == 2) leaf_sums(acc[0], acc[1], S.leaf, wave, lane);
        else leaf_sums(acc[0], none, S.leaf, wave, lane);
        __syncthreads();
        if (tid < 8 * kSums) {
            const unsigned v = tid >> 3, i = tid & 7u;
            double w = S.leaf[2 * i][v] + S.leaf[2 * i + 1][v];
            w += __shfl_xor(w, 1);
            w += __shfl_xor(w, 2);
            w += __shfl_xor(w, 4);
            if (i == 0) {
                if (parts == 1) {
                    S.tot[v] = w;
                } else {
                    const u64 b = u64(__double_as_longlong(w));
                    u64* const w2 = sum_words(t, v, unsigned(part));
                    st64(w2, tagged(unsigned(b), tag_of(t)));
                    st64(w2 + 1, tagged(unsigned(b >> 32), tag_of(t)));
                }
            }
        }
    };
    // The instance's sums of phase t into S.tot: a tree over the parts, read
    // by everyone up to 64 parts; above, the first part of every 16 sums them
    // up and sends the result to kCopies places, each read by some of the
    // parts (256 readers of 256 parts' words took 20 us a phase).
    auto take_sums = [&](int t) -> bool {
        if (parts > 1 && wave < kSums) {
            auto fetch = [&](const u64* at, bool mine, double& w) {
                unsigned b[2];
                w = 0.0;
                if (!mine) return true;
                if (!await<2>(at, tag_of(t), b, bar)) return false;
                w = __longlong_as_double((long long)((u64(b[1]) << 32) | b[0]));
                return true;
            };
            double w;
            bool ok = true;
            if (parts <= unsigned(kWave)) {
                ok = fetch(sum_words(t, wave, lane), lane < parts, w);
#pragma unroll
                for (int m = 1; m < kWave; m <<= 1) w += __shfl_xor(w, m);
            } else {
                if ((unsigned(part) % kFan) == 0u) {
                    ok = fetch(sum_words(t, wave, unsigned(part) + lane), lane < kFan && unsigned(part) + lane < parts, w);
#pragma unroll
                    for (unsigned m = 1; m < kFan; m <<= 1) w += __shfl_xor(w, int(m));
                    w = __shfl(w, 0);
                    const u64 b = u64(__double_as_longlong(w));
                    if (ok && lane < 2u * kCopies)
                        st64(group_words(t, lane >> 1, wave, unsigned(part) / kFan) + (lane & 1u),
                             tagged((lane & 1u) != 0u ? unsigned(b >> 32) : unsigned(b), tag_of(t)));
                }
                ok = __ballot(!ok) == 0ull &&
                     fetch(group_words(t, unsigned(part) % kCopies, wave, lane), lane < (parts + kFan - 1u) / kFan, w);
#pragma unroll
                for (unsigned m = 1; m < kFan; m <<= 1) w += __shfl_xor(w, int(m));
            }
            if (lane == 0) S.tot[wave] = w;
            if (!ok) S.bad = 1;
        }
        __syncthreads();
        return S.bad == 0;
    };

    // ---- set-up: r_0 = b - A x, z_0 = p_0 = M^-1 r_0 ----
    apply(p, q);
    {
    double acc[kSlots][kSums];
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
#pragma unroll
        for (int v = 0; v < kSums; ++v) acc[s][v] = 0.0;
        if (on[s] && live[s]) {
            const f3 b = ld3g(I.rhs, ldx(plan, rows_at + pos0 + lp[s]));
            r[s] = sub(b, q[s]);
            p[s] = mv_sym(M[s], r[s]);
            if (ex[s] != CHX_RES_NONE) send_row(0, ex[s], r[s]);
            acc[s][0] = dot64(r[s], p[s]);
            acc[s][1] = dot64(b, b);
            acc[s][4] = dot64(r[s], r[s]);
        }
    }
    send_sums(0, acc);
    }
    double bb = 0.0;
    for (int k = 0;; ++k) {
        const bool last = k > 0 && k >= I.max_iter;  // at the cap: the last update only
        // The halo rows' q_{k-1} (set-up: r_0), sent before the sums: waiting
        // for them first hides their way behind the sums'.
        f3 h = mk(0.f, 0.f, 0.f);
        if (rtid < n_halo && !last) {
            unsigned w[3];
            if (await<3>(row_words(k, hex), tag_of(k), w, bar))
                h = mk(__uint_as_float(w[0]), __uint_as_float(w[1]), __uint_as_float(w[2]));
            else
                S.bad = 1;
        }
        if (!take_sums(k)) return false;
        const double rho = S.tot[0], sig = S.tot[1], del = S.tot[2], gam = S.tot[3], rr = S.tot[4];
        if (k == 0) bb = sig;
        if (B.trace != nullptr) {
            trace_point(B, trace_e, unsigned(B.n_instances) - unsigned(ld64(&B.xbuf[RES_DONE])));
            ++trace_e;
        }
        const int its = k > 0 ? k - 1 : 0;  // updates of x so far
        if (its >= I.max_iter || (I.tol > 0.0 && rr <= I.tol * I.tol * bb)) {
            if (part == 0 && tid == 0) {
                B.inst_iters[inst] = its;
                B.inst_rr[inst] = rr;
                B.inst_bb[inst] = bb;
                if (B.inst_rho != nullptr) B.inst_rho[inst] = rho;
                (void)__hip_atomic_fetch_add(&B.xbuf[RES_DONE], 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            break;
        }
        if (part == 0 && tid == 0 && (k & 7) == 0)
            (void)__hip_atomic_fetch_add(&B.xbuf[RES_PROGRESS], 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        float alpha = 0.0f, beta = 0.0f;
        if (k > 0) merged_scalars(rho, sig, del, gam, alpha, beta);
        // halo rows: r_k, z_k, p_k as their owners form them
        if (rtid < n_halo && !last) {
            if (k == 0) {
                hr = h;
                lds_st(&S.p[kPart + rtid], mv_sym(hM, hr));
            } else {
                hr = axpy(-alpha, h, hr);
                lds_st(&S.p[kPart + rtid], axpy(beta, lds_ld(&S.p[kPart + rtid]), mv_sym(hM, hr)));
            }
        }
#pragma unroll
        for (int s = 0; s < kSlots; ++s)
            if (on[s]) {
                if (k > 0) {
                    r[s] = axpy(-alpha, q[s], r[s]);
                    S.x[lp[s]] = axpy(alpha, p[s], S.x[lp[s]]);
                    p[s] = axpy(beta, p[s], mv_sym(M[s], r[s]));
                }
                S.p[lp[s]] = p[s];
            }
        if (!last) apply(p, q);
        double acc[kSlots][kSums];
#pragma unroll
        for (int s = 0; s < kSlots; ++s) {
#pragma unroll
            for (int v = 0; v < kSums; ++v) acc[s][v] = 0.0;
            if (on[s] && live[s]) {
                if (!last && ex[s] != CHX_RES_NONE) send_row(k + 1, ex[s], q[s]);
                const f3 z = mv_sym(M[s], r[s]);
                acc[s][0] = dot64(r[s], z);
                acc[s][4] = dot64(r[s], r[s]);
                if (!last) {
                    acc[s][1] = dot64(p[s], q[s]);
                    acc[s][2] = dot64(q[s], z);
                    acc[s][3] = dot64(q[s], mv_sym(M[s], q[s]));
                }
            }
        }
        send_sums(k + 1, acc);
    }
#pragma unroll
    for (int s = 0; s < kSlots; ++s)
        if (live[s]) st3g(I.x, ldx(plan, rows_at + pos0 + lp[s]), S.x[lp[s]]);
    return true;
}

// The workgroup's next (item, part), or kExit: it reports itself idle, hands
// list items to the idle workgroups of its group while the next one fits,
// and waits for its own.  Items come by falling number of parts, so what a
// finished gang frees always holds the next one; with no gang left running
// every workgroup of the group is idle and any item of the list fits.
__device__ unsigned next_item(const chx_cloth_batch& B, unsigned group, unsigned first, unsigned stride, unsigned idx,
                              unsigned epoch, unsigned had, unsigned& out, const Barrier& bar) {
    __syncthreads();  // its readers are done
    if (threadIdx.x == 0) {
        u64* const idle = &B.xbuf[RES_IDLE + 16 * group];
        u64* const next = &B.xbuf[RES_NEXT];
        const gp<const int> items = glb(B.res_items);
        const unsigned n_items = unsigned(B.res_n_items - B.res_n_big);
        auto mail = [&](unsigned i) { return &B.xbuf[RES_MAIL + 16ull * (first + stride * i)]; };
        auto add_idle = [&](unsigned m) {
            return unsigned(__hip_atomic_fetch_or(idle, u64(m), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) | m;
        };
        auto send = [&](unsigned gang, unsigned item) {
            unsigned part = 0;
            for (unsigned m = gang; m != 0u; m &= m - 1u, ++part)
                st64(mail(unsigned(__ffs(int(m))) - 1u), tagged((item << 8) | (item == kExit ? 0u : part), epoch));
        };
        unsigned have = add_idle(1u << idx);
        unsigned i = unsigned(ld64(next));
        for (;;) {
            if (i >= n_items) {  // nothing left: everyone idle leaves
                const unsigned m = unsigned(__hip_atomic_exchange(idle, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                send(m, kExit);
                break;
            }
            const unsigned need = unsigned(items[4 * (unsigned(B.res_n_big) + i) + 1]);
            if (unsigned(__popc(have)) < need) break;
            unsigned gang = 0, m = have;
            for (unsigned c = 0; c < need; ++c, m &= m - 1u) gang |= m & (0u - m);
            u64 expect = have;
            if (!__hip_atomic_compare_exchange_strong(idle, &expect, u64(have & ~gang), __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT)) {
                have = unsigned(expect);
                i = unsigned(ld64(next));
                continue;
            }
            u64 at = i;
            if (__hip_atomic_compare_exchange_strong(next, &at, u64(i + 1u), __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT)) {
                send(gang, unsigned(B.res_n_big) + i);
                have = unsigned(ld64(idle));
                i = unsigned(ld64(next));
            } else {
                have = add_idle(gang);
                i = unsigned(at);
            }
        }
        // wait for this workgroup's own word
        const u64* const mine = mail(idx);
        Watch watch(bar);
        unsigned seen = unsigned(ld64(&B.xbuf[RES_PROGRESS])), level = 0, got = kExit << 8;
        for (;;) {
            const u64 w = ld64(mine);
            if (unsigned(w >> 32) == epoch && unsigned(w) != had) {
                got = unsigned(w);
                break;
            }
            if (!watch.again(&B.xbuf[RES_PROGRESS], seen)) {
                got = kExit << 8 | 1u;  // aborted
                break;
            }
            backoff(level);
        }
        out = got;
    }
    __syncthreads();
    return out;
}

template <bool GEN>
__global__ __launch_bounds__(kThreads, 2) void resident_kernel(chx_cloth_batch B, int finalize) {
    __shared__ ResLds<GEN> S;
    const int G = int(gridDim.x);
    const Barrier bar = make_barrier(B);
    unsigned* const progress = reinterpret_cast<unsigned*>(&B.xbuf[RES_PROGRESS]);
    const unsigned epoch = unsigned(ld64(&B.xbuf[RES_EPOCH]));
    if (blockIdx.x == 0 && B.trace != nullptr)
        for (int e = threadIdx.x; e < 2 * B.trace_entries; e += blockDim.x) glb(B.trace)[e] = 0ull;
    if (ld64(&B.xbuf[RES_CLEAR]) != 0ull) {
        // the launch numbers start over: no word may keep an old tag
        for (u64 k = RES_MAIL + u64(blockIdx.x) * kThreads + threadIdx.x; k < B.res_xwords; k += u64(G) * kThreads)
            st64(&B.xbuf[k], 0ull);
        if (!grid_sync(bar, unsigned(G))) return;
    }
    __syncthreads();
    // groups: workgroups b = x (mod 8), which the dispatcher places on one
    // XCD, or all of them
    const unsigned groups = unsigned(B.res_groups), group = blockIdx.x % groups, idx = blockIdx.x / groups;
    const unsigned rank = group * (unsigned(G) / groups) + idx;
    int trace_e = 0;
    // the workgroup's work: the single instance's part, or the leading large
    // items that use its rank, then items dealt to its group
    const gp<const int> items = glb(B.res_items);
    int big = 0;
    unsigned had = 0xffffffffu;
    bool ok = true;
    for (;;) {
        int inst = 0, part = -1;
        if (B.inst == nullptr) {
            if (big++ > 0 || rank >= unsigned(B.single.res_parts)) break;
            part = int(rank);
        } else if (big < B.res_n_big) {
            const int base = items[4 * big + 2], parts = items[4 * big + 1];
            inst = items[4 * big];
            ++big;
            if (int(rank) < base || int(rank) >= base + parts) continue;
            part = int(rank) - base;
            __syncthreads();  // the previous solve's readers of S are done
        } else {
            if (B.res_n_items == B.res_n_big) break;
            had = next_item(B, group, group, groups, idx, epoch, had, S.mail, bar);
            if ((had >> 8) == kExit) {
                ok = (had & 255u) == 0u;
                break;
            }
            inst = __builtin_amdgcn_readfirstlane(items[4 * (had >> 8)]);
            part = int(__builtin_amdgcn_readfirstlane(had & 255u));
        }
        const Inst I = inst_at(B, inst);
        ok = solve_part<GEN>(B, I, inst, part, epoch, S, bar, trace_e);
        if (!ok) break;
    }
    // pos and vel change only when every instance was solved
    if (!ok) return;
    if (G > 1 && !grid_sync(bar, unsigned(G), -1, nullptr, progress)) return;
    if (finalize) finalize_tiles(B, G);
}

using ResFn = void (*)(chx_cloth_batch, int);
ResFn resident_fn(bool general) { return general ? resident_kernel<true> : resident_kernel<false>; }

std::mutex g_mu;
int g_limit[16] = {0};

}  // namespace

int resident_grid_limit() {
    int dev = 0;
    hip_check(hipGetDevice(&dev), "hipGetDevice");
    std::lock_guard<std::mutex> lk(g_mu);
    int& l = g_limit[dev & 15];
    if (l == 0) {
        hipDeviceProp_t prop;
        hip_check(hipGetDeviceProperties(&prop, dev), "hipGetDeviceProperties");
        bool fits = true;
        for (bool general : {false, true}) {
            int per_cu = 0;
            hip_check(hipOccupancyMaxActiveBlocksPerMultiprocessor(
                          &per_cu, reinterpret_cast<const void*>(resident_fn(general)), kThreads, 0),
                      "hipOccupancyMaxActiveBlocksPerMultiprocessor");
            fits = fits && per_cu >= 1;
        }
        l = fits ? std::min(kMaxParts, prop.multiProcessorCount) : -1;
    }
    return std::max(l, 0);
}

void launch_resident(const chx_cloth_batch& B, int finalize, hipStream_t stream) {
    if (B.res_grid == 1) {
        // nothing waits for another workgroup: an ordinary launch, without the
        // ~11 us before and after that a cooperative one takes
        resident_fn(B.res_general != 0)<<<1, kThreads, 0, stream>>>(B, finalize);
        hip_check(hipGetLastError(), "resident_kernel launch");
        return;
    }
    chx_cloth_batch arg = B;
    int fin = finalize;
    void* args[] = {&arg, &fin};
    hip_check(hipLaunchCooperativeKernel(reinterpret_cast<const void*>(resident_fn(B.res_general != 0)),
                                         dim3(B.res_grid), dim3(kThreads), args, 0, stream),
              "hipLaunchCooperativeKernel(resident pcg)");
}

}  // namespace chx

using namespace chx;

extern "C" int chx_resident_grid_limit(int* max_blocks) {
    return guarded([&] {
        require(max_blocks != nullptr, "chx_resident_grid_limit: null output");
        *max_blocks = resident_grid_limit();
    });
}
