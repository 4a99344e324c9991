// Device helpers shared by the streaming and the resident PCG kernels.
#pragma once

#include "chx_device.h"
#include "chx_exchange.h"

namespace chx {

// Divide guard |den| > 1e-37 (ChysX/src/solver/pcg_solver.cu:122-127), with
// the FP64 inner products rounded to FP32 once.
__device__ __forceinline__ float guarded_div(double a, double b) {
    return (b > 1e-37 || b < -1e-37) ? float(a / b) : 0.0f;
}

// Optional solver trace (workgroup 0, thread 0): real-time stamp and
// active-instance count at barrier e.
__device__ __forceinline__ void trace_point(const chx_cloth_batch& B, int e, unsigned active) {
    if (B.trace != nullptr && blockIdx.x == 0 && threadIdx.x == 0 && e < B.trace_entries) {
        const gp<unsigned long long> t = glb(B.trace);
        t[2 * e] = __builtin_amdgcn_s_memrealtime();
        t[2 * e + 1] = active;
    }
}

// Finalize of every tile (cloth_simulator.cu:222-244): pos = x_n + dx,
// vel = dx / dt, times exp(-damping dt) when damping > 0.
__device__ __forceinline__ void finalize_tiles(const chx_cloth_batch& B, int G) {
    for (int t = blockIdx.x; t < B.n_tiles; t += G) {
        int inst, rb, re;
        get_tile(B, t, inst, rb, re);
        const Inst I = inst_at(B, inst);
        const float inv_dt = 1.0f / I.dt;
        const float decay = (I.damping > 0.0f) ? expf(-I.damping * I.dt) : 1.0f;
        for (unsigned row = unsigned(rb) + threadIdx.x; row < unsigned(re); row += blockDim.x) {
            const f3 d = ld3g(I.x, row);
            const f3 p = ld3g(I.pos, row);
            st3g(I.pos, row, add(p, d));
            f3 v = mul(d, inv_dt);
            if (I.damping > 0.0f) v = mul(v, decay);
            st3g(I.vel, row, v);
        }
    }
}

// The single-barrier iteration's scalars (chx_step.hip, pcg1_kernel) from
// the previous phase's exact sums: alpha, and beta from the identity
//   <r_k, z_k> = rho - 2 alpha delta + alpha^2 gamma.
// Its terms carry the FP32 rounding of the stored vectors, a few units of
// 2^-24 of their size.  Above 1e-5 of them (~100 such units) rho_k, and so
// beta, is resolved to about 1%; below, the direction restarts from z_k
// (beta = 0) instead of taking a rounding-noise beta.  A tighter cut (1e-3)
// restarts on ordinary fast-converging iterations and costs the Krylov
// acceleration: 13 iterations instead of 9 on a pin-driven substep of the
// 32x32 cloth.
__device__ __forceinline__ void merged_scalars(double rho, double sig, double del, double gam, float& alpha,
                                               float& beta) {
    alpha = guarded_div(rho, sig);
    const double ad = double(alpha);
    const double t1 = 2.0 * ad * del, t2 = ad * ad * gam;
    const double rho_k = rho - t1 + t2;
    const bool resolved = rho_k > 1.0e-5 * (fabs(rho) + fabs(t1) + fabs(t2));
    beta = resolved ? guarded_div(rho_k, rho) : 0.0f;
}

// ---- control words of the resident PCG (first words of chx_cloth_batch::xbuf)
enum : int {
    RES_EPOCH = 0,      // launch number, 1 .. kResEpochs: the tag of everything exchanged
    RES_CLEAR = 1,      // the numbers started over: the next resident launch clears old tags first
    RES_NEXT = 16,      // next item of the list
    RES_PROGRESS = 32,  // changes while any gang iterates (idle workgroups wait as long as it does)
    RES_DONE = 48,      // instances finished
    RES_IDLE = 64,      // per group (16 words apart): its idle workgroups
    RES_MAIL = 256      // per workgroup (16 words apart): its next item and part
};
constexpr int kResGroups = 8;
static_assert(RES_MAIL + 16 * 256 <= CHX_RES_CONTROL_WORDS && RES_IDLE + 16 * kResGroups <= RES_MAIL, "control words");

// New launch number and an empty work list, before each PCG launch (same
// stream, an earlier kernel).
__device__ __forceinline__ void reset_resident(unsigned long long* xbuf) {
    if (xbuf == nullptr) return;
    if (threadIdx.x < kResGroups) xbuf[RES_IDLE + 16 * threadIdx.x] = 0ull;
    if (threadIdx.x == 0) {
        const Launch next = next_launch({xbuf[RES_EPOCH], xbuf[RES_CLEAR]}, xbuf[RES_DONE]);
        xbuf[RES_NEXT] = 0ull;
        xbuf[RES_DONE] = 0ull;
        xbuf[RES_EPOCH] = next.number;
        xbuf[RES_CLEAR] = next.clear;
    }
}

}  // namespace chx
