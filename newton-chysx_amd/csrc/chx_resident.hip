// Resident block-Jacobi PCG: a workgroup keeps its part of a matrix in
// registers and its vectors in registers and LDS from the first product to
// the last, so an iteration reads no matrix from memory.  What crosses
// workgroups in an iteration is the halo rows of q = A p and a few partial
// sums.
//
// Why: streaming the matrix every iteration cost 20.5 ms per solve of the
// 512-cloth batch (2.08 M rows, 66 iterations on average), set by the
// L1-L2 stream, and 19 us per iteration of one 256x256 cloth, set by the
// grid barrier's cache write-backs.  A CU has 512 KB of registers: 1024 rows
// of a sheet's matrix (six upper blocks a row) take 221 KB, so 256 CUs hold
// 262,144 rows, and the instances of a batch are independent: they are
// solved one after another by gangs of ceil(rows / 1024) workgroups.
//
// Two solvers, operation for operation those of chx_step.hip: the merged
// recurrence of pcg1_kernel (one exchange an iteration: halo rows of q and
// five sums), and the two-reduction one of pcg_kernel (BF16 mode and caller's
// row-major systems: halo rows of q and sigma, then rho and ||r||^2).  Every
// row sums its products in the order of those kernels.
//
// Products: a thread's held block serves its own row (A_ij p_j) and, through
// a product slot in LDS, the row of its transpose (A_ij^T p_i).  Blocks
// between parts are held by both (the second copy is a "ghost block").
// Halo rows' r, z and p are kept by every part that reads them, updated from
// the sent q with the same operations as by their owner.
//
// Inner products: FP64, one sum per 64-row leaf (a wavefront), combined over
// the leaves of the instance by a fixed binary tree that does not depend on
// how many leaves a part has: the same bits for every part size and gang.
//
// Exchange: 64-bit words of values and a tag that names launch and exchange,
// so a reader needs no ordering between words and no cache maintenance: it
// reads a word until its tag is the awaited one.  Words alternate between two
// slots; a slot is rewritten two exchanges later at the earliest, which its
// writer enters only after every part's sums of the exchange between, sent
// after their reads of the slot.  Sums and rows are numbered apart
// (chx_exchange.h): iterations of the two-reduction solver send rows in every
// second exchange.
//
// Every part has a 128-byte line for its sums, which all parts read, 16 bytes
// a lane.  What costs is lines with several writers: with the parts' words
// side by side an all-to-all of five sums took 1.8 us between 16 workgroups,
// 2.1 between 32 and 2.4 between 64; with a line each 1.3, 1.3 and 1.4, and
// 2.9 between 256.  Two levels of any group size (3.3 to 5.3 us for 64 to 256)
// and copies per reader lose to that, and so does more than one read in
// flight: the floor of one store and one load is 1.0 to 1.2 us.
// A halo row is 16 bytes: three floats and the tag's 16 bits in both words.
#include <algorithm>
#include <cstddef>
#include <mutex>

#include "chx_pcg.h"
#include "chx_resident.h"

namespace chx {
namespace {

constexpr int kThreads = 512;  // two waves per SIMD with 256 VGPRs each
constexpr int kWaves = kThreads / kWave;
constexpr int kLeaves = CHX_RES_PART_MAX / CHX_RES_LEAF;
// Keeps a value that the loop does not change from being re-derived ahead of
// the loop (addresses and masks of every block would not fit the registers).
__device__ __forceinline__ unsigned opaque(unsigned v) {
    asm volatile("" : "+v"(v));
    return v;
}
// The thread index for addresses and masks of one use.  What the loop derives
// from it is derived again: kept over the loop those values went to scratch,
// and a reload waits for every store in flight, the halo rows just sent among
// them (32 spilled registers: 6.8 us an iteration of a 256x256 cloth, 5.8 without).
__device__ __forceinline__ unsigned tid_here() { return opaque(threadIdx.x); }
// Four times the low (0) or high (1) half of a word, in one instruction and
// anew at every use.
template <int HALF>
__device__ __forceinline__ unsigned lds_bytes(unsigned w) {
    unsigned r;
    if constexpr (HALF == 0)
        asm volatile("v_lshlrev_b32_sdwa %0, %2, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0"
                     : "=v"(r) : "v"(w), "s"(2u));
    else
        asm volatile("v_lshlrev_b32_sdwa %0, %2, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1"
                     : "=v"(r) : "v"(w), "s"(2u));
    return r;
}

// The forms of a plan (chysx_hip.h).  Sheet: a row's lower blocks come
// through product slots and are summed before the upper ones that its thread
// holds, which is column order.  General: all of a row's products go through
// its slots, in column order; twice the slots and wider rows, so half the
// rows.  Rows: a caller's matrix, every row holding all of its own blocks.
// Half sheet: a sheet's plan for 512 rows, one row a thread, which leaves
// registers for the two-reduction solver (at 1024 rows it would spill 430).
// BF16 mode, four substeps of a 128x128 cloth: 2.30 ms, on a general plan with
// its longer rows of product slots 2.56.  For FP32 solves of small parts it is
// no faster than the sheet kernel with half its threads' rows idle.
enum { SHEET = CHX_RES_FORM_SHEET, GENERAL = CHX_RES_FORM_GENERAL, ROWS = CHX_RES_FORM_ROWS, HALF = CHX_RES_FORM_HALF };
template <int FORM>
struct Form {
    static constexpr bool kSheet = FORM == SHEET || FORM == HALF;
    static constexpr unsigned kRows = FORM == SHEET ? CHX_RES_PART_MAX : CHX_RES_GEN_PART;
    static constexpr int kSlots = kRows / kThreads;  // own rows per thread
    static constexpr int kHeld = kSheet ? CHX_RES_HELD : (FORM == GENERAL ? CHX_RES_GEN_HELD : CHX_RES_ROW_WIDTH);
    // product slots per row
    static constexpr unsigned kPlaces = kSheet ? CHX_RES_HELD : (FORM == GENERAL ? CHX_RES_GEN_WIDTH : 0);
    static constexpr unsigned kSpare = kPlaces * kRows;  // first of the unread product slots
    static constexpr unsigned kSource = 3 * (kSpare + kWave);  // LDS word of the source vector, behind the products
    // A held block's word in the plan, and here: the LDS words of its source
    // vector entry and of its product slot, and its place in the row.
    static __device__ __forceinline__ unsigned unpack(unsigned w, unsigned lane) {
        if (FORM == ROWS) return kSource + 3u * w;
        const unsigned src = kSheet ? w & 0xffffu : w & 0x3ffu;
        unsigned slot = kSheet ? w >> 16 : (w >> 10) & 0x3fffu;
        if (slot == (kSheet ? 0xffffu : 0x3fffu)) slot = kSpare + lane;
        return kSheet ? (kSource + 3u * src) | (3u * slot) << 16 : 3u * src | (3u * slot) << 12 | (w >> 24) << 27;
    }
    // LDS byte offsets, formed at every use
    static __device__ __forceinline__ unsigned src(unsigned w) {
        return FORM == GENERAL ? 4u * (kSource + (opaque(w) & 0xfffu)) : lds_bytes<0>(w);
    }
    static __device__ __forceinline__ unsigned slot(unsigned w) {
        return kSheet ? lds_bytes<1>(w) : 4u * ((opaque(w) >> 12) & 0x7fffu);
    }
    static __device__ __forceinline__ unsigned place(unsigned w) { return w >> 27; }
};
static_assert(Form<SHEET>::kSource + 3 * (Form<SHEET>::kRows + CHX_RES_HALO_MAX) < (1u << 16) &&
                  3 * (Form<GENERAL>::kSpare + kWave) < (1u << 15) &&
                  3 * (Form<GENERAL>::kRows + CHX_RES_HALO_MAX) <= (1u << 12) && CHX_RES_GEN_WIDTH <= 16,
              "word fields");
// Sums of an exchange: merged solver rho, sigma, delta, gamma, ||r||^2
// (set-up: ||b||^2 in place of sigma); two-reduction solver sigma, or rho and
// ||r||^2 (set-up: and ||b||^2).
constexpr int kSums = 5;
constexpr int kMaxParts = 256;
constexpr unsigned kLine = 16;  // words of a part's line
static_assert(2 * kSums <= kLine, "a part's sums in one line");
constexpr unsigned kExit = 0xffffffu;  // mailbox item: nothing left
static_assert(CHX_RES_LEAF == kWave && Form<SHEET>::kSlots == 2 && Form<GENERAL>::kSlots == 1 && kLeaves == 2 * kWaves,
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

// 16-byte accesses of the exchange area at agent scope (byte offsets).  The
// two 64-bit words of one may be of different age: both carry the tag.  A
// word itself arrives whole: an aligned 64-bit atomic load or store is the
// same memory instruction, two dwords wide, so an aligned half of a wider
// access of the same scope is no less whole.  Measured: 64 lanes each of 128
// workgroups storing without a pause, 128 workgroups on other dies reading,
// 1.6e9 reads, 4.9e8 of them of a new value, no half torn.
typedef unsigned v4u __attribute__((ext_vector_type(4)));
using Area = __amdgpu_buffer_rsrc_t;
constexpr int kAgent = 1 << 4;  // sc1
__device__ __forceinline__ Area exchange_area(const chx_cloth_batch& B) {
    return __builtin_amdgcn_make_buffer_rsrc(B.xbuf, 0, int(B.res_xwords * 8ull), 0x00020000);
}
__device__ __forceinline__ v4u ld128(Area a, unsigned at) { return __builtin_amdgcn_raw_buffer_load_b128(a, at, 0, kAgent); }
__device__ __forceinline__ void st128(Area a, unsigned at, v4u v) { __builtin_amdgcn_raw_buffer_store_b128(v, a, at, 0, kAgent); }

// Triples in LDS, by the byte offset of their first word in the struct that
// starts with them, or by its index.
template <class Lds>
__device__ __forceinline__ f3 lds_at(const Lds& S, unsigned at) {
    const float* const m = reinterpret_cast<const float*>(reinterpret_cast<const char*>(&S) + at);
    return {m[0], m[1], m[2]};
}
template <class Lds>
__device__ __forceinline__ void lds_put(Lds& S, unsigned at, f3 v) {
    float* const m = reinterpret_cast<float*>(reinterpret_cast<char*>(&S) + at);
    m[0] = v.x;
    m[1] = v.y;
    m[2] = v.z;
}
__device__ __forceinline__ f3 lds_ld(const float* m, unsigned i) { return {m[i], m[i + 1u], m[i + 2u]}; }
__device__ __forceinline__ void lds_st(float* m, unsigned i, f3 v) {
    m[i] = v.x;
    m[i + 1u] = v.y;
    m[i + 2u] = v.z;
}
template <int FORM, bool FULL>
struct ResLds {
    // products by target row, then one unread slot per lane for blocks
    // without a target
    float prod[3 * (Form<FORM>::kSpare + kWave)];
    float p[3 * (Form<FORM>::kRows + CHX_RES_HALO_MAX)];  // source vector: own rows, halo rows
    float diag[FULL ? 9 : 6][Form<FORM>::kRows];
    float x[3 * Form<FORM>::kRows];
    float ghost[FORM == ROWS ? 1 : 9][CHX_RES_GHOST_MAX];
    float hminv[FORM == SHEET ? 6 : 1][CHX_RES_HALO_MAX];  // halo rows' inverses (other forms: registers)
    double bb;       // ||b||^2
    double leaf[kLeaves][kSums];
    double tot[8];
    double wsum[kWaves][8];
    int bad;         // a wait gave up
    unsigned mail;   // mailbox word of the workgroup
};

using SheetLds = ResLds<SHEET, false>;
using HalfLds = ResLds<HALF, true>;
using GeneralLds = ResLds<GENERAL, false>;
using RowsLds = ResLds<ROWS, true>;
static_assert(offsetof(SheetLds, p) == 4 * Form<SHEET>::kSource && offsetof(HalfLds, p) == 4 * Form<HALF>::kSource &&
                  offsetof(GeneralLds, p) == 4 * Form<GENERAL>::kSource && offsetof(RowsLds, p) == 4 * Form<ROWS>::kSource,
              "the source vector follows the products");

// Bounded wait of one lane: true while it may go on.  After the bound the
// solve is aborted for every workgroup (the report of grid_sync).
struct Watch {
    const Barrier& bar;
    u64 t0 = 0;
    unsigned polls = 0;
    __device__ explicit Watch(const Barrier& b) : bar(b) {}
    __device__ bool again(u64* progress, unsigned& seen) {
        unsigned* sync = bar.sync;
        if (polls == 0u) t0 = __builtin_amdgcn_s_memrealtime();
        if ((++polls & 15u) == 0u && ld_relaxed(&sync[SYNC_ABORT]) != 0u) return false;
        if (__builtin_amdgcn_s_memrealtime() - t0 <= bar.ticks) return true;
        const unsigned now = unsigned(ld64(progress));
        if (now != seen) {
            seen = now;
            t0 = __builtin_amdgcn_s_memrealtime();
            return true;
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

// The 16 bytes at at(j) for j < N, read until `mine` accepts them all; false:
// the wait was given up.  A peer may still be busy with an earlier large item
// of the list, so the wait goes on as long as any gang iterates.
template <int N, class At, class Mine>
__device__ __forceinline__ bool await(Area area, At at, Mine mine, v4u (&w)[N], u64* progress, const Barrier& bar) {
    Watch watch(bar);
    unsigned seen = 0;
    for (;;) {
        asm volatile("" ::: "memory");  // the loads read again
        bool ok = true;
#pragma unroll
        for (int j = 0; j < N; ++j) w[j] = ld128(area, at(j));
#pragma unroll
        for (int j = 0; j < N; ++j) ok = ok && mine(w[j]);
        if (ok) return true;
        if (!watch.again(progress, seen)) return false;
    }
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
// The wave's two leaf sums of five values into `leaf`.  Halving butterfly:
// each step adds lane pairs and packs two values into the two halves of the
// pairs, so five values of two leaves take 14 FP64 adds instead of 60.
__device__ __forceinline__ void leaf_sums(const double (&a)[5], const double (&b)[5], double (&leaf)[kLeaves][kSums],
                                          unsigned wave) {
    const unsigned lane = tid_here() & unsigned(kWave - 1);
    double v[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) v[k] = fold32(a[k], b[k]);  // half h: leaf of slot h
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
// The same for up to three values (the second and third in one row each).
template <int N>
__device__ __forceinline__ void leaf_sums(const double (&a)[N], const double (&b)[N], double (&leaf)[kLeaves][kSums],
                                          unsigned wave) {
    static_assert(N >= 1 && N <= 3, "values");
    const unsigned lane = tid_here() & unsigned(kWave - 1);
    double w = fold16(fold32(a[0], b[0]), N > 1 ? fold32(a[N > 1 ? 1 : 0], b[N > 1 ? 1 : 0]) : 0.0);
    double y = 0.0;
    if constexpr (N == 3) {
        y = fold32(a[2], b[2]);
        y = fold16(y, y);
    }
    w = fold8(w, y, lane);
    w += dpp64<kHalfMirror>(w);
    w += dpp64<kXor2>(w);
    w += dpp64<kXor1>(w);
    double(&out)[kSums] = leaf[(lane >> 5) * kWaves + wave];
    const unsigned place = lane & 31u;
    if (place == 0u) out[0] = w;
    if (N > 1 && place == 16u) out[1] = w;
    if (N > 2 && place == 8u) out[2] = w;
}

// Solves instance `inst` together with the workgroups that hold its other
// parts; this one holds part `part`.  TWO: the two-reduction solver (with
// B.bf16_blocks on the BF16 matrix).  False: aborted.
template <int FORM, bool TWO>
__device__ __forceinline__ bool solve_part(const chx_cloth_batch& B, const Inst& I, int inst, int part, unsigned epoch,
                                           ResLds<FORM, TWO>& S, const Barrier& bar, int& trace_e) {
    using F = Form<FORM>;
    constexpr int kSlots = F::kSlots, kHeld = F::kHeld;
    constexpr unsigned kPart = F::kRows;
    constexpr int kDiag = TWO ? 9 : 6;       // words of a diagonal block in LDS
    constexpr int kMinv = FORM == ROWS ? 9 : 6;  // words of an inverse
    const unsigned tid = threadIdx.x, lane = tid & (kWave - 1);
    const unsigned wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const gp<const unsigned> plan = I.res_plan;
    const unsigned n = unsigned(I.n_rows), parts = unsigned(I.res_parts);
    const gp<const unsigned> hdr = plan + 8 * part;
    const unsigned n_own = hdr[0], n_halo = hdr[1], halo_at = hdr[2], n_ghost = hdr[3], ghost_at = hdr[4], widest = hdr[5];
    const unsigned pos0 = unsigned(part) * unsigned(I.res_part_rows);
    const unsigned rows_at = 8u * parts, meta_at = rows_at + n, exp_at = meta_at + n, held_at = exp_at + n;
    // exchange area (byte offsets): [2][parts] lines, then [2][exports] rows
    const Area area = exchange_area(B);
    const unsigned xsum = 8u * I.res_xbase, xrow = xsum + 2u * 8u * kLine * parts;
    const unsigned exports = unsigned(I.res_exports);
    // numbers of exchanges: t of the sums, u of the rows
    auto tag_of = [&](unsigned number) { return exchange_tag(epoch, number); };
    auto line = [&](unsigned t, unsigned q) { return xsum + 8u * kLine * (exchange_slot(t) * parts + q); };
    auto row_bytes = [&](unsigned u, unsigned e) { return xrow + 16u * (exchange_slot(u) * exports + e); };
    auto send_row = [&](unsigned u, unsigned e, f3 v) {
        const unsigned x = __float_as_uint(v.x), y = __float_as_uint(v.y), z = __float_as_uint(v.z);
        const unsigned tag = tag_of(u) << 16;
        st128(area, row_bytes(u, e), v4u{x, (y & 0xffffu) | tag, z, (y >> 16) | tag});
    };

    // ---- load: own rows, ghost block, halo row ----
    unsigned ex[kSlots], holds[kSlots], word[kSlots][kHeld];
    bool on[kSlots];  // this wave has a row
    auto row_at = [&](int s) { return unsigned(s) * kThreads + tid_here(); };  // this lane's row of slot s
    auto live = [&](int s) { return row_at(s) < n_own; };
    float V[kSlots][kHeld][9], M[kSlots][kMinv];
    f3 r[kSlots], p[kSlots], q[kSlots];
    // ghost blocks and halo rows from the last thread down: in a small part
    // the first waves have the rows
    auto rtid_here = [] { return unsigned(kThreads - 1) - tid_here(); };
    auto halo_slot = [&] { return 3u * (kPart + rtid_here()); };
    auto is_halo = [&] { return rtid_here() < n_halo; };
    auto is_ghost = [&] { return FORM != ROWS && rtid_here() < n_ghost; };
    auto position = [&](int s) { return pos0 + (live(s) ? row_at(s) : 0u); };
    // Where the blocks of a row are (one slot per block in the general form).
    struct Where {
        unsigned row, first, slot[FORM == GENERAL ? kHeld : 1];
    };
    auto locate = [&](Where (&w)[kSlots], unsigned& ghost) {
#pragma unroll
        for (int s = 0; s < kSlots; ++s) {
            const unsigned K = position(s);
            w[s].row = ldx(plan, rows_at + K);
            if constexpr (FORM == GENERAL) {
#pragma unroll
                for (int u = 0; u < kHeld; ++u) w[s].slot[u] = ldx(plan, held_at + unsigned(kHeld + u) * n + K);
            }
        }
        ghost = is_ghost() ? ldx(plan, ghost_at + 2u * rtid_here()) : 0u;
    };
    auto find_first = [&](Where (&w)[kSlots]) {
        if constexpr (FORM != GENERAL)
#pragma unroll
            for (int s = 0; s < kSlots; ++s)
                w[s].first = FORM == ROWS ? unsigned(ldx(I.row_offsets, w[s].row))
                                          : unsigned(ldx(I.upper_offsets, w[s].row / CHX_SLICE_ROWS)) +
                                                w[s].row % CHX_SLICE_ROWS;
    };
    // the matrix blocks: FP32, or the BF16 copies and compensated diagonal
    auto load_blocks = [&](bool half, const Where (&w)[kSlots], unsigned ghost) {
        auto block = [&](unsigned v, float (&m)[9]) {
            if (FORM == ROWS) {
                const gp<const float> b = rec_at(gp<const float>(I.values), v, 9u);
#pragma unroll
                for (int c = 0; c < 9; ++c) m[c] = b[c];
            } else if (TWO && half) {
                ld9p(gp<const uint16_t>(I.values16), v & 0x7fffffffu, m);
            } else {
                ld9p(gp<const float>(I.values), v & 0x7fffffffu, m);
            }
            if (FORM == GENERAL && (v >> 31) != 0u) transpose9(m);
        };
#pragma unroll
        for (int s = 0; s < kSlots; ++s)
            if (on[s]) {
#pragma unroll
                for (int u = 0; u < kHeld; ++u) {
#pragma unroll
                    for (int c = 0; c < 9; ++c) V[s][u][c] = 0.0f;
                    if (unsigned(u) < holds[s]) {
                        if constexpr (FORM == GENERAL) block(w[s].slot[u], V[s][u]);
                        else block(w[s].first + unsigned(u) * (FORM == ROWS ? 1u : unsigned(CHX_SLICE_ROWS)), V[s][u]);
                    }
                }
            }
        if (is_ghost()) {
            float g[9];
            block(ghost, g);
            const unsigned rtid = rtid_here();
#pragma unroll
            for (int c = 0; c < 9; ++c) S.ghost[c][rtid] = g[c];
        }
    };
    auto load_diag = [&](bool half, unsigned row, float (&d)[9]) {
        if (FORM == ROWS) {
            const gp<const float> b = rec_at(gp<const float>(I.diag), row, 9u);
#pragma unroll
            for (int c = 0; c < 9; ++c) d[c] = b[c];
        } else if (TWO && half) {
            ld9p(gp<const float>(I.diag_c), row, d);
        } else {
            ld6p(gp<const float>(I.diag), row, d);
        }
    };
    auto keep_diag = [&](int s, const float (&d)[9]) {
        const unsigned lp = row_at(s);
#pragma unroll
        for (unsigned c = 0; c < unsigned(kDiag); ++c) S.diag[c][lp] = d[kDiag == 9 ? c : sym6_pos(c)];
    };
    auto apply_minv = [&](const float (&m)[kMinv], f3 v) {
        if constexpr (FORM == ROWS) return mv9(m, v);
        else return mv_sym(m, v);
    };
    auto invert = [&](const float (&d)[9], float (&m)[kMinv]) {
        float full[9];
        inverse9(d, full);
#pragma unroll
        for (unsigned c = 0; c < unsigned(kMinv); ++c) m[c] = full[kMinv == 9 ? c : sym6_pos(c)];
    };
    // The set-up is a chain of round trips to memory, so each link's loads are
    // issued together: the plan's words of the rows, halo rows and ghost
    // blocks; then diagonals, vectors and block offsets; then the blocks.
    Where where[kSlots];
    unsigned ghost, meta[kSlots], gword = 0, hrow = 0, hex = 0;
    locate(where, ghost);
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
        on[s] = (unsigned(s) * kWaves + wave) * kWave < n_own;
        const unsigned K = position(s);
        meta[s] = ldx(plan, meta_at + K);
        ex[s] = ldx(plan, exp_at + K);
#pragma unroll
        for (int u = 0; u < kHeld; ++u) word[s][u] = ldx(plan, held_at + unsigned(u) * n + K);
    }
    if (is_ghost()) gword = ldx(plan, ghost_at + 2u * rtid_here() + 1u);  // its source and product slot
    if (is_halo()) {
        hrow = ldx(plan, halo_at + 2u * rtid_here());
        hex = ldx(plan, halo_at + 2u * rtid_here() + 1u);
    }
    constexpr bool kHaloInLds = FORM == SHEET;
    float hM[kMinv];
    f3 hr = mk(0.f, 0.f, 0.f);
    {
        find_first(where);
        float d[kSlots][9], hd[9];
        f3 hx = hr;
#pragma unroll
        for (int s = 0; s < kSlots; ++s) {
            load_diag(false, where[s].row, d[s]);
            p[s] = ld3g(I.x, where[s].row);
            r[s] = ld3g(I.rhs, where[s].row);
        }
        if (is_halo()) {
            load_diag(false, hrow, hd);
            hx = ld3g(I.x, hrow);
        }
#pragma unroll
        for (int s = 0; s < kSlots; ++s) {
            const bool has = live(s);
            const unsigned lp = row_at(s), ns = has ? meta[s] & 255u : 0u;
            holds[s] = has ? meta[s] >> 8 : 0u;
            if (!has) {
                ex[s] = CHX_RES_NONE;
                r[s] = p[s] = mk(0.f, 0.f, 0.f);
            }
            q[s] = mk(0.f, 0.f, 0.f);
#pragma unroll
            for (int u = 0; u < kHeld; ++u) {
                // a block that is not there is zero, of the row itself
                const unsigned none = F::kSheet ? (0xffffu << 16) | lp : (FORM == GENERAL ? (0x3fffu << 10) | lp : lp);
                word[s][u] = F::unpack(unsigned(u) < holds[s] ? word[s][u] : none, lane);
            }
            if (on[s]) {
                // product slots that no block fills stay zero and are added
                // like the others
#pragma unroll
                for (unsigned u = 0; u < F::kPlaces; ++u)
                    if (u >= ns) lds_st(S.prod, 3u * (u * kPart + lp), mk(0.f, 0.f, 0.f));
                keep_diag(s, d[s]);
                lds_st(S.x, 3u * lp, p[s]);
                lds_st(S.p, 3u * lp, p[s]);
            }
            invert(d[s], M[s]);
        }
        if (is_halo()) {
            invert(hd, hM);
            if constexpr (kHaloInLds) {
                const unsigned rtid = rtid_here();
#pragma unroll
                for (int c = 0; c < kMinv; ++c) S.hminv[c][rtid] = hM[c];
            }
            lds_st(S.p, halo_slot(), hx);
        }
    }
    load_blocks(false, where, ghost);
    // vmcnt(0): with no load pending at its entry the loop waits for none (and
    // so for none of its stores) where it uses what was loaded here
    __builtin_amdgcn_s_waitcnt(0x0f70);
    auto halo_minv = [&](f3 v) {
        if constexpr (kHaloInLds) {
            const unsigned rtid = rtid_here();
            float m[kMinv];
#pragma unroll
            for (int c = 0; c < kMinv; ++c) m[c] = S.hminv[c][rtid];
            return apply_minv(m, v);
        } else {
            return apply_minv(hM, v);
        }
    };
    if (tid == 0) S.bad = 0;
    if (tid < kLeaves * kSums) S.leaf[tid / kSums][tid % kSums] = 0.0;

    // A times the vector in S.p (own rows also in v); S.p and S.prod are read
    // until the next workgroup barrier.
    auto apply = [&](const f3 (&v)[kSlots], f3 (&out)[kSlots]) {
        if constexpr (FORM != ROWS) {
#pragma unroll
            for (int s = 0; s < kSlots; ++s)
                if (on[s]) {
#pragma unroll
                    for (int u = 0; u < kHeld; ++u) lds_put(S, F::slot(word[s][u]), mv9t(V[s][u], v[s]));
                }
        }
        __syncthreads();
        if constexpr (FORM != ROWS) {
            if (is_ghost()) {
                const unsigned rtid = rtid_here();
                float g[9];
#pragma unroll
                for (int c = 0; c < 9; ++c) g[c] = S.ghost[c][rtid];
                const unsigned w = opaque(gword);
                lds_st(S.prod, 3u * (w >> 16), mv9t(g, lds_ld(S.p, 3u * (w & 0xffffu))));
            }
        }
        if constexpr (FORM == GENERAL) {
            if (on[0]) {
                const unsigned lp = row_at(0);
                f3 src[kHeld];
#pragma unroll
                for (int u = 0; u < kHeld; ++u) src[u] = lds_at(S, F::src(word[0][u]));
#pragma unroll
                for (int u = 0; u < kHeld; ++u)
                    if (unsigned(u) < opaque(holds[0]))
                        lds_st(S.prod, 3u * (F::place(opaque(word[0][u])) * kPart + lp), mv9(V[0][u], src[u]));
            }
        }
        // a sheet's part without ghost blocks has all its products already
        if (FORM == GENERAL || (F::kSheet && n_ghost > 0u)) __syncthreads();
#pragma unroll
        for (int s = 0; s < kSlots; ++s)
            if (on[s]) {
                const unsigned lp = row_at(s);
                f3 src[kHeld], low[kHeld];
                float d[9];
                if constexpr (FORM != GENERAL) {
#pragma unroll
                    for (int u = 0; u < kHeld; ++u) src[u] = lds_at(S, F::src(word[s][u]));
                }
#pragma unroll
                for (int c = 0; c < kDiag; ++c) d[kDiag == 9 ? unsigned(c) : sym6_pos(unsigned(c))] = S.diag[c][lp];
                if constexpr (kDiag == 6) {
                    d[3] = d[1];
                    d[6] = d[2];
                    d[7] = d[5];
                }
                f3 sum;
                if constexpr (F::kSheet) {
#pragma unroll
                    for (int l = 0; l < kHeld; ++l) low[l] = lds_ld(S.prod, 3u * (unsigned(l) * kPart + lp));
                    sum = mv9(d, v[s]);
#pragma unroll
                    for (int l = 0; l < kHeld; ++l) sum = add(sum, low[l]);
#pragma unroll
                    for (int u = 0; u < kHeld; ++u) sum = add(sum, mv9(V[s][u], src[u]));
                } else if constexpr (FORM == GENERAL) {
                    sum = mv9(d, v[s]);
#pragma unroll
                    for (unsigned t = 0; t < F::kPlaces; t += 4)
                        if (t < widest) {
                            f3 y[4];
#pragma unroll
                            for (unsigned u = 0; u < 4; ++u) y[u] = lds_ld(S.prod, 3u * ((t + u) * kPart + lp));
#pragma unroll
                            for (unsigned u = 0; u < 4; ++u) sum = add(sum, y[u]);
                        }
                } else {
                    // the order of spmv_core<8>: lane l's diag (l = 0) and
                    // blocks l, l + 8, then the lanes' butterfly
                    static_assert(kHeld > 8 && kHeld <= 16, "two rounds of eight");
                    f3 w[8];
#pragma unroll
                    for (int l = 0; l < 8; ++l) {
                        w[l] = mv9(V[s][l], src[l]);
                        if (l == 0) w[0] = add(mv9(d, v[s]), w[0]);
                        if (l + 8 < kHeld) w[l] = add(w[l], mv9(V[s][l + 8 < kHeld ? l + 8 : l], src[l + 8 < kHeld ? l + 8 : l]));
                    }
#pragma unroll
                    for (int m = 4; m > 0; m >>= 1)
#pragma unroll
                        for (int l = 0; l < m; ++l) w[l] = add(w[l], w[l + m]);
                    sum = w[0];
                }
                out[s] = sum;
            }
    };
    // The sums of exchange t: per leaf, then over the part's leaves, sent to
    // the gang.
    auto tree8 = [](double w) {  // over eight lanes
        w += dpp64<kXor1>(w);
        w += dpp64<kXor2>(w);
        return w + dpp64<kHalfMirror>(w);
    };
    auto send_sums = [&](unsigned t, auto& acc) {
        constexpr int N = int(sizeof(acc[0]) / sizeof(double));
        double none[N] = {};
        leaf_sums(acc[0], kSlots == 2 ? acc[kSlots - 1] : none, S.leaf, wave);
        __syncthreads();
        const unsigned me = tid_here();
        if (me < 8u * N) {
            const unsigned v = me >> 3, i = me & 7u;
            const double w = tree8(S.leaf[2 * i][v] + S.leaf[2 * i + 1][v]);
            const u64 b = u64(__double_as_longlong(w));
            if (i == 0 && parts == 1) S.tot[v] = w;
            if (i == 0 && parts > 1)
                st128(area, line(t, unsigned(part)) + 16u * v, v4u{unsigned(b), tag_of(t), unsigned(b >> 32), tag_of(t)});
        }
    };
    // The instance's N sums of exchange t into tot: a tree over the parts.
    // Up to 64 parts a wave reads one sum of every part (1.47 us for an
    // exchange of 64 parts in a loop of its own, 1.94 the other way).  Above,
    // that is 1280 reads of 16 bytes for 256 parts (2.9 us): there eight lanes
    // read a part's line together and a wave 32 lines (2.6 us), and the waves'
    // sums meet in LDS, where every wave adds them up by itself.
    double tot[kSums];
    auto take_sums = [&](unsigned t, unsigned N) -> bool {
        const unsigned lane = tid_here() & unsigned(kWave - 1), tag = tag_of(t);
        u64* const progress = &B.xbuf[RES_PROGRESS];
        auto mine = [&](v4u w) { return w.y == tag && w.w == tag; };
        auto value = [](v4u w) { return __longlong_as_double((long long)((u64(w.z) << 32) | w.x)); };
        const bool wide = parts > unsigned(kWave);
        if (parts == 1) {
        } else if (!wide) {
            if (wave < N) {
                v4u b[1];
                const bool has = lane < parts;
                // lanes without a part read the first one's
                if (!await<1>(area, [&](int) { return line(t, has ? lane : 0u) + 16u * wave; }, mine, b, progress, bar))
                    S.bad = 1;
                double w = tree8(has ? value(b[0]) : 0.0);
                w += dpp64<kRor8>(w);
                if (parts > 16u) {
                    w = fold16(w, w);
                    w = fold32(w, w);
                }
                if (lane == 0) S.tot[wave] = w;
            }
        } else {
            constexpr int kReads = kMaxParts / (8 * kWaves);
            double sum = 0.0;
            if (8u * kReads * wave < parts) {
                const unsigned first = 8u * kReads * wave + (lane >> 3);
                const unsigned word = (lane & 7u) < N ? lane & 7u : N - 1u;
                auto has = [&](int j) { return first + 8u * unsigned(j) < parts; };
                v4u b[kReads];
                if (!await<kReads>(
                        area, [&](int j) { return line(t, has(j) ? first + 8u * unsigned(j) : 0u) + 16u * word; }, mine, b,
                        progress, bar))
                    S.bad = 1;
                double w[kReads];
#pragma unroll
                for (int j = 0; j < kReads; ++j) {
                    w[j] = has(j) ? value(b[j]) : 0.0;
                    w[j] += dpp64<kRor8>(w[j]);
                    w[j] = fold16(w[j], w[j]);
                    w[j] = fold32(w[j], w[j]);
                }
                static_assert(kReads == 4, "a tree over a wave's reads");
                sum = (w[0] + w[1]) + (w[2] + w[3]);
            }
            if (lane < N) S.wsum[wave][lane] = sum;
        }
        __syncthreads();
        if (S.bad != 0) return false;
        if (!wide) {
#pragma unroll
            for (unsigned v = 0; v < unsigned(kSums); ++v)
                if (v < N) tot[v] = S.tot[v];
        } else {
            double w = 0.0;
            if (lane < 8u * N) w = S.wsum[lane & 7u][lane >> 3];
            w = tree8(w);
            const u64 b = u64(__double_as_longlong(w));
#pragma unroll
            for (unsigned v = 0; v < unsigned(kSums); ++v)
                if (v < N) {
                    const unsigned lo = __builtin_amdgcn_readlane(unsigned(b), 8 * v);
                    const unsigned hi = __builtin_amdgcn_readlane(unsigned(b >> 32), 8 * v);
                    tot[v] = __longlong_as_double((long long)((u64(hi) << 32) | lo));
                }
        }
        return true;
    };
    // The halo row's triple of number u (sent before its exchange's sums:
    // waiting for it first hides its way behind the sums').
    auto take_halo = [&](unsigned u) {
        f3 h = mk(0.f, 0.f, 0.f);
        if (is_halo()) {
            const unsigned tag = tag_of(u) & 0xffffu;
            v4u w[1];
            if (await<1>(
                    area, [&](int) { return row_bytes(u, hex); },
                    [&](v4u v) { return v.y >> 16 == tag && v.w >> 16 == tag; }, w, &B.xbuf[RES_PROGRESS], bar))
                h = mk(__uint_as_float(w[0].x), __uint_as_float((w[0].y & 0xffffu) | w[0].w << 16),
                       __uint_as_float(w[0].z));
            else
                S.bad = 1;
        }
        return h;
    };
    auto mark_trace = [&] {
        if (B.trace != nullptr) {
            trace_point(B, trace_e, unsigned(B.n_instances) - unsigned(ld64(&B.xbuf[RES_DONE])));
            ++trace_e;
            __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0), so that the loop has no load pending to wait for
        }
    };
    auto stop = [&](int its, double rr, double bb, double rho) {
        if (part == 0 && tid_here() == 0) {
            const unsigned i = opaque(unsigned(inst));
            stx(glb(B.inst_iters), i, its);
            stx(glb(B.inst_rr), i, rr);
            stx(glb(B.inst_bb), i, bb);
            if (B.inst_rho != nullptr) stx(glb(B.inst_rho), i, rho);
            (void)__hip_atomic_fetch_add(&B.xbuf[RES_DONE], 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    };
    auto alive = [&](int k) {
        if (part == 0 && tid == 0 && (k & 7) == 0)
            (void)__hip_atomic_fetch_add(&B.xbuf[RES_PROGRESS], 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    // r = b - A x (A x in q) and its sums; the exported rows of r are sent.
    auto residual = [&](unsigned t, unsigned u) {
        double acc[kSlots][3];  // rho, ||b||^2, ||r||^2
#pragma unroll
        for (int s = 0; s < kSlots; ++s) {
            acc[s][0] = acc[s][1] = acc[s][2] = 0.0;
            if (on[s] && live(s)) {
                // at the set-up r holds b
                const f3 b = t > 0u ? ld3g(I.rhs, ldx(plan, rows_at + pos0 + row_at(s))) : r[s];
                r[s] = sub(b, q[s]);
                if (ex[s] != CHX_RES_NONE) send_row(u, ex[s], r[s]);
                acc[s][0] = dot64(r[s], apply_minv(M[s], r[s]));
                acc[s][1] = dot64(b, b);
                acc[s][2] = dot64(r[s], r[s]);
            }
        }
        send_sums(t, acc);
    };

    if constexpr (!TWO) {
        // ---- set-up: r_0 = b - A x, z_0 = p_0 = M^-1 r_0 ----
        apply(p, q);
        residual(0u, 0u);  // every exchange has rows: one number for both
        hr = take_halo(0u);
        if (!take_sums(0u, 3)) return false;
        double rho = tot[0], rr = tot[2];
        S.bb = tot[1];  // every thread the same
        mark_trace();
        double sig = 0.0, del = 0.0, gam = 0.0;
        for (int k = 0;; ++k) {
            const bool last = k > 0 && k >= I.max_iter;  // at the cap: the last update only
            f3 h = mk(0.f, 0.f, 0.f);
            if (k > 0) {
                if (!last) h = take_halo(k);
                if (!take_sums(k, 5)) return false;
                rho = tot[0];
                sig = tot[1];
                del = tot[2];
                gam = tot[3];
                rr = tot[4];
                mark_trace();
            }
            const int its = k > 0 ? k - 1 : 0;  // updates of x so far
            const double bb = S.bb;
            if (its >= I.max_iter || (I.tol > 0.0 && rr <= I.tol * I.tol * bb)) {
                stop(its, rr, bb, rho);
                break;
            }
            alive(k);
            float alpha = 0.0f, beta = 0.0f;
            if (k > 0) merged_scalars(rho, sig, del, gam, alpha, beta);
            // r_k, z_k, p_k (k = 0: both factors are zero), halo rows as their
            // owners form them
            if (is_halo() && !last) {
                hr = axpy(-alpha, h, hr);
                const unsigned at = halo_slot();
                lds_st(S.p, at, axpy(beta, lds_ld(S.p, at), halo_minv(hr)));
            }
#pragma unroll
            for (int s = 0; s < kSlots; ++s)
                if (on[s]) {
                    r[s] = axpy(-alpha, q[s], r[s]);
                    const unsigned at = 3u * row_at(s);
                    lds_st(S.x, at, axpy(alpha, p[s], lds_ld(S.x, at)));
                    p[s] = axpy(beta, p[s], apply_minv(M[s], r[s]));
                    lds_st(S.p, at, p[s]);
                }
            if (!last) apply(p, q);
            double acc[kSlots][5];
#pragma unroll
            for (int s = 0; s < kSlots; ++s) {
#pragma unroll
                for (int v = 0; v < 5; ++v) acc[s][v] = 0.0;
                if (on[s]) {  // lanes without a row add zeros
                    if (!last && ex[s] != CHX_RES_NONE) send_row(k + 1, ex[s], q[s]);
                    const f3 z = apply_minv(M[s], r[s]);
                    acc[s][0] = dot64(r[s], z);
                    acc[s][4] = dot64(r[s], r[s]);
                    if (!last) {
                        acc[s][1] = dot64(p[s], q[s]);
                        acc[s][2] = dot64(q[s], z);
                        acc[s][3] = dot64(q[s], apply_minv(M[s], q[s]));
                    }
                }
            }
            send_sums(k + 1, acc);
        }
    } else {
        // With B.bf16_blocks the inner iterations run on the BF16 matrix and
        // test the recursive residual; when it meets the tolerance one slot
        // computes the true residual with the FP32 blocks: the solve stops on
        // that, or CG restarts from it (pcg_kernel, instance_slot).
        const bool half = FORM != ROWS && B.bf16_blocks != 0;
        constexpr int kMaxRefine = 1;
        double rho = 0.0, rr = 0.0, bb = 0.0;
        float beta = 0.0f;
        bool residual_step = true;        // set-up, then refinement: r = b - A x, x in p and S.p
        bool exact = true, fresh = true;  // rr is of b - A x; p starts from z
        int k = 0, refines = -1;
        Exchange at;                      // the last exchange
        int blocks = 0;                   // which matrix V holds
        for (;;) {
            if (!residual_step) {
                const bool met = I.tol > 0.0 && rr <= I.tol * I.tol * bb;
                if (k >= I.max_iter || (met && (!half || exact || refines >= kMaxRefine))) {
                    stop(k, rr, bb, rho);
                    break;
                }
                alive(k);
                if (met) {
                    // this slot computes the true residual: halo rows of x first
                    residual_step = true;
                    ++k;
                    at.next(true);
                    double zero[kSlots][1] = {};
#pragma unroll
                    for (int s = 0; s < kSlots; ++s)
                        if (on[s]) {
                            p[s] = lds_ld(S.x, 3u * row_at(s));
                            if (ex[s] != CHX_RES_NONE) send_row(at.rows, ex[s], p[s]);
                        }
                    send_sums(at.sums, zero);
                    const f3 hx = take_halo(at.rows);
                    if (!take_sums(at.sums, 1)) return false;
                    if (is_halo()) lds_st(S.p, halo_slot(), hx);
                } else {
                    if (is_halo()) {
                        const f3 z = halo_minv(hr);
                        lds_st(S.p, halo_slot(), fresh ? z : axpy(beta, lds_ld(S.p, halo_slot()), z));
                    }
#pragma unroll
                    for (int s = 0; s < kSlots; ++s)
                        if (on[s]) {
                            const f3 z = apply_minv(M[s], r[s]);
                            p[s] = fresh ? z : axpy(beta, p[s], z);
                        }
                }
#pragma unroll
                for (int s = 0; s < kSlots; ++s)
                    if (on[s]) lds_st(S.p, 3u * row_at(s), p[s]);
            }
            const int want = half && !residual_step ? 1 : 0;
            if (want != blocks) {
                Where w[kSlots];
                unsigned g;
                locate(w, g);
                find_first(w);
                load_blocks(want != 0, w, g);
#pragma unroll
                for (int s = 0; s < kSlots; ++s)
                    if (on[s]) {
                        float d[9];
                        load_diag(want != 0, w[s].row, d);
                        keep_diag(s, d);
                    }
                __builtin_amdgcn_s_waitcnt(0x0f70);
                blocks = want;
            }
            apply(p, q);
            if (residual_step) {
                at.next(true);
                residual(at.sums, at.rows);
                hr = take_halo(at.rows);
                if (!take_sums(at.sums, 3)) return false;
                rho = tot[0];
                bb = tot[1];
                rr = tot[2];
                residual_step = false;
                exact = fresh = true;
                ++refines;
                mark_trace();
                continue;
            }
            at.next(true);
            double sum[kSlots][1];
#pragma unroll
            for (int s = 0; s < kSlots; ++s) {
                sum[s][0] = 0.0;
                if (on[s]) {
                    if (ex[s] != CHX_RES_NONE) send_row(at.rows, ex[s], q[s]);
                    sum[s][0] = dot64(p[s], q[s]);
                }
            }
            send_sums(at.sums, sum);
            const f3 h = take_halo(at.rows);
            if (!take_sums(at.sums, 1)) return false;
            const float alpha = guarded_div(rho, tot[0]);
            mark_trace();
            if (is_halo()) hr = axpy(-alpha, h, hr);
            at.next(false);
            double acc[kSlots][2];
#pragma unroll
            for (int s = 0; s < kSlots; ++s) {
                acc[s][0] = acc[s][1] = 0.0;
                if (on[s]) {
                    const unsigned xi = 3u * row_at(s);
                    lds_st(S.x, xi, axpy(alpha, p[s], lds_ld(S.x, xi)));
                    r[s] = axpy(-alpha, q[s], r[s]);
                    acc[s][0] = dot64(r[s], apply_minv(M[s], r[s]));
                    acc[s][1] = dot64(r[s], r[s]);
                }
            }
            send_sums(at.sums, acc);
            if (!take_sums(at.sums, 2)) return false;
            beta = guarded_div(tot[0], rho);
            rho = tot[0];
            rr = tot[1];
            exact = fresh = false;
            mark_trace();
            ++k;
        }
    }
#pragma unroll
    for (int s = 0; s < kSlots; ++s)
        if (live(s)) st3g(I.x, ldx(plan, rows_at + pos0 + row_at(s)), lds_ld(S.x, 3u * row_at(s)));
    // x is stored in the plan's row order and the finalize reads it in row
    // order: rows of other waves, with no grid barrier in between when the
    // launch has one workgroup
    __syncthreads();
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
        auto add_idle = [&](u64 m) {
            return u64(__hip_atomic_fetch_or(idle, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) | m;
        };
        auto send = [&](u64 gang, unsigned item) {
            unsigned part = 0;
            for (u64 m = gang; m != 0ull; m &= m - 1ull, ++part)
                st64(mail(unsigned(__ffsll((long long)m)) - 1u), tagged((item << 8) | (item == kExit ? 0u : part), epoch));
        };
        u64 have = add_idle(1ull << idx);
        unsigned i = unsigned(ld64(next));
        for (;;) {
            if (i >= n_items) {  // nothing left: everyone idle leaves
                send(__hip_atomic_exchange(idle, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), kExit);
                break;
            }
            const unsigned need = unsigned(items[4 * (unsigned(B.res_n_big) + i) + 1]);
            if (unsigned(__popcll(have)) < need) break;
            u64 gang = 0, m = have;
            for (unsigned c = 0; c < need; ++c, m &= m - 1ull) gang |= m & (0ull - m);
            u64 expect = have;
            if (!__hip_atomic_compare_exchange_strong(idle, &expect, have & ~gang, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT)) {
                have = expect;
                i = unsigned(ld64(next));
                continue;
            }
            u64 at = i;
            if (__hip_atomic_compare_exchange_strong(next, &at, u64(i + 1u), __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT)) {
                send(gang, unsigned(B.res_n_big) + i);
                have = ld64(idle);
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

template <int FORM, bool TWO>
__global__ __launch_bounds__(kThreads, 2) void resident_kernel(chx_cloth_batch B, int finalize) {
    __shared__ ResLds<FORM, TWO> S;
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
    // groups: workgroups b = x (mod groups); with eight, the dispatcher places
    // a group on one XCD
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
        ok = solve_part<FORM, TWO>(B, I, inst, part, epoch, S, bar, trace_e);
        if (!ok) break;
    }
    // pos and vel change only when every instance was solved
    if (!ok) return;
    if (G > 1 && !grid_sync(bar, unsigned(G), -1, nullptr, progress)) return;
    if (finalize) finalize_tiles(B, G);
}

using ResFn = void (*)(chx_cloth_batch, int);
// form: a plan's; two: the two-reduction solver (always for a caller's rows)
ResFn resident_fn(int form, bool two) {
    if (form == ROWS) return resident_kernel<ROWS, true>;
    if (form == HALF) return resident_kernel<HALF, true>;
    if (form == GENERAL) return two ? resident_kernel<GENERAL, true> : resident_kernel<GENERAL, false>;
    return resident_kernel<SHEET, false>;
}
ResFn resident_fn(const chx_cloth_batch& B) { return resident_fn(B.res_form, B.bf16_blocks != 0); }

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
        for (int form : {SHEET, HALF, GENERAL, ROWS})
            for (bool two : {false, true}) {
                int per_cu = 0;
                hip_check(hipOccupancyMaxActiveBlocksPerMultiprocessor(
                              &per_cu, reinterpret_cast<const void*>(resident_fn(form, two)), kThreads, 0),
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
        resident_fn(B)<<<1, kThreads, 0, stream>>>(B, finalize);
        hip_check(hipGetLastError(), "resident_kernel launch");
        return;
    }
    chx_cloth_batch arg = B;
    int fin = finalize;
    void* args[] = {&arg, &fin};
    hip_check(hipLaunchCooperativeKernel(reinterpret_cast<const void*>(resident_fn(B)),
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
