// vh_keyswitch.hip -- key-switch inner product fused into the forward row pass of the
// ModUp digits (FP64 path, N = 2^13 .. 2^16, at most two output components).
#include "vh_device.h"
#include "vh_kernels.h"

// ---------------------------------------------------------------------------
// The column pass has left the lifted digit rows, transformed over their first
// logn - 8 stages, in jb.modup; this kernel finishes the last 8 stages of every digit
// for one tile of 8 rows of 256 elements and accumulates
//     out_c = -+ sum_d NTT(digit_d) * key[d][c]      (the mul_subto of gadget.c:22-37)
// in registers, so the transformed digits never return to memory.
//
// A row has 32 threads with 8 values each, in three register phases:
//   1  stages 0..2   k = t + 32 m                    (256-byte runs of the digit row)
//   2  stages 3..5   k = 32 (t >> 2) + 4 m + (t & 3)
//   3  stages 6..7   k = 128 (m >> 2) + 4 t + (m & 3)
// with two exchanges through LDS inside the wave (row slices of 36 doubles per 32: the
// reads of phase 2 touch every bank once).  Phase 3 leaves four adjacent elements per
// lane, so the key rows, the pass-through rows and the output move as 16-byte words of
// one contiguous kilobyte per 32 lanes.  (16 values per thread ending in 16 contiguous
// elements made every key load touch 64 separate 128-byte lines.)
// The row's 255 twiddles do not depend on the digit: they are formed once per workgroup
// (table head times row factor, centred, as in k_ntt16p) into LDS.
// 8 values and two accumulators per thread leave room to load a digit's key words and the
// next digit before the butterflies within 128 VGPRs: four workgroups per CU.
// Measured for 32 ciphertexts at N = 2^16, 24 + 4 limbs (11.7 GB to read and write, 2.2 ms of
// FP64 issue): 5.54 ms with 16 values per thread and contiguous key reads, 4.75 ms with those
// values regrouped before the key reads, 3.80 ms in this form (3.1 TB/s).
// Bounds: every twiddle is paired with w * RN(1/q), so a multiplied operand must stay
// below 4q (see k_ntt16p): inputs are centred, four stages add at most 4q with the
// multiplied operand of the fourth below 3.5q, then every value is centred again.
//
// Grid: x = ciphertext, y = tile, z = extended limb.  A key block is (y, z).
// Consecutive workgroups are dealt round-robin over the 8 XCDs, so with `xcd` set the
// workgroup index is remapped to put all ciphertexts of one key block on one XCD, one after
// another: each XCD's L2 then fetches a key block once instead of every XCD fetching it.
// Spreading a job's digits over several workgroups (partial sums added by a second kernel) was
// measured on launches of 60 to 300 workgroups and gained nothing: the digit loop keeps its loads
// in flight, and the partials' traffic costs what the extra workgroups save.
// ---------------------------------------------------------------------------
constexpr int VH_RM_PITCH = 288;   // doubles of one row's exchange slice (256 + 4 per 32)

template <int C>
__global__ void __launch_bounds__(256, 4)
k_row_mac(const vh_mac_job *__restrict__ jobs, const vh_limb *__restrict__ limbs,
          const uint64_t *const *__restrict__ kptr, int logn, int xcd)
{
    constexpr int ROWS = 8, S = 256, T = 32;
    __shared__ double lds[ROWS * VH_RM_PITCH];
    __shared__ double tws[ROWS][S];
    unsigned bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
    if (xcd) {   // bijective when gridDim.y * gridDim.z is a multiple of 8 (checked at launch)
        const unsigned lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
        const unsigned slot = lin >> 3, kb = (slot / gridDim.x) * 8 + (lin & 7);
        bx = slot % gridDim.x;
        by = kb % gridDim.y;
        bz = kb / gridDim.y;
    }
    const vh_mac_job &jb = jobs[bx];
    const int ti = (int)bz;
    if (ti >= jb.next) return;   // jobs of a batch may have fewer extended limbs (whole block)
    const int D = jb.digits;
    const int limb = jb.limb[ti];
    const vh_limb &L = limbs[limb];
    const double q = L.qd, qinv = L.qinv;
    const size_t n = (size_t)1 << logn;
    const int tid = threadIdx.x, g = tid / T, t = tid % T;
    const size_t sub = (size_t)by * ROWS + g;
    {   // the rows' twiddles: entry e of row r = head e times the row's factor of e's stage
        const int e = tid, sp = e ? 31 - __builtin_clz(e) : 0;
        const double h = vh_global(reinterpret_cast<const double *>(L.tw_fwd))[2 * e];
        const VH_GLOBAL double *rf = vh_global(reinterpret_cast<const double *>(L.rowf_fwd)) + ((size_t)by * ROWS * 8 + sp) * 2;
#pragma unroll
        for (int r = 0; r < ROWS; r++)
            tws[r][e] = vh_center(vh_mulmod_tw(h, rf[16 * r], rf[16 * r + 1], q), q, qinv);
        __syncthreads();
    }
    double *xs = lds + g * VH_RM_PITCH;
    const double *tw = tws[g];
    const int ta = t >> 2, tb = t & 3;
    const size_t rowoff = sub * S, x0 = rowoff + 4 * t;
    const VH_GLOBAL uint64_t *dig = vh_global(jb.modup + (size_t)ti * n + rowoff + t);
    const size_t dstep = (size_t)jb.next * n;
    const uint64_t *const *kp = kptr + jb.kptr_off + (size_t)ti * D * C;

    double acc[C][8];
#pragma unroll
    for (int c = 0; c < C; c++)
#pragma unroll
        for (int m = 0; m < 8; m++) acc[c][m] = 0.0;
    auto bf = [&](double &a, double &b, double w) {
        const double x = vh_mulmod_tw(b, w, w * qinv, q);
        b = a - x;
        a = a + x;
    };

    uint64_t raw[8];
    if (D > 0) {
#pragma unroll
        for (int m = 0; m < 8; m++) raw[m] = vh_ld(dig + 32 * m);
    }
    for (int d = 0; d < D; d++, kp += C) {
        double v[8];
#pragma unroll
        for (int m = 0; m < 8; m++) v[m] = __longlong_as_double((long long)raw[m]);
        // this digit's key words, then the next digit: both land during the butterflies
        uint64_t kw[C][8];
#pragma unroll
        for (int c = 0; c < C; c++) {
            const VH_GLOBAL uint64_t *kr = vh_global(kp[c]) + x0;
#pragma unroll
            for (int h = 0; h < 4; h++) vh_ld2(kr + 128 * (h >> 1) + 2 * (h & 1), kw[c][2 * h], kw[c][2 * h + 1]);
        }
        if (d + 1 < D) {
#pragma unroll
            for (int m = 0; m < 8; m++) raw[m] = vh_ld(dig + (size_t)(d + 1) * dstep + 32 * m);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 3; s++) {
            const int hm = 4 >> s;
#pragma unroll
            for (int m = 0; m < 8; m++)
                if (!(m & hm)) bf(v[m], v[m + hm], tw[(1 << s) + (m >> (3 - s))]);
        }
        vh_wave_sync();   // every read of the previous digit's exchange is done
#pragma unroll
        for (int m = 0; m < 8; m++) xs[t + 36 * m] = v[m];
        vh_wave_sync();
#pragma unroll
        for (int m = 0; m < 8; m++) v[m] = xs[36 * ta + 4 * m + tb];
#pragma unroll
        for (int s = 3; s < 6; s++) {
            const int hm = 4 >> (s - 3);
#pragma unroll
            for (int m = 0; m < 8; m++)
                if (!(m & hm)) bf(v[m], v[m + hm], tw[(1 << s) + (ta << (s - 3)) + (m >> (6 - s))]);
            if (s == 3) {
#pragma unroll
                for (int m = 0; m < 8; m++) v[m] = vh_center(v[m], q, qinv);
            }
        }
        // a thread overwrites the slots it read itself
#pragma unroll
        for (int m = 0; m < 8; m++) xs[36 * ta + 4 * m + tb] = v[m];
        vh_wave_sync();
#pragma unroll
        for (int m = 0; m < 8; m++) v[m] = xs[144 * (m >> 2) + 4 * t + 4 * (t >> 3) + (m & 3)];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const double w6 = tw[64 + 32 * h + t];
            bf(v[4 * h], v[4 * h + 2], w6);
            bf(v[4 * h + 1], v[4 * h + 3], w6);
            bf(v[4 * h], v[4 * h + 1], tw[128 + 64 * h + 2 * t]);
            bf(v[4 * h + 2], v[4 * h + 3], tw[128 + 64 * h + 2 * t + 1]);
        }
        const bool fourth = (d & 3) == 3;
#pragma unroll
        for (int m = 0; m < 8; m++) {
            const double a = vh_center(v[m], q, qinv);          // |a| <= q/2 + 1
#pragma unroll
            for (int c = 0; c < C; c++) {
                const double k = vh_u2d(kw[c][m]);
                const double hi = a * k;
                const double lo = __fma_rn(a, k, -hi);
                const double qt = __fma_rn(a, k * qinv, VH_MAGIC) - VH_MAGIC;
                acc[c][m] += __fma_rn(-qt, q, hi) + lo;         // |term| <= q + 2^47
            }
        }
        // centred every 4th digit: |acc| <= q/2 + 4 (q + 2^47) < 2^53 stays exact
        if (fourth) {
#pragma unroll
            for (int c = 0; c < C; c++)
#pragma unroll
                for (int m = 0; m < 8; m++) acc[c][m] = vh_center(acc[c][m], q, qinv);
        }
    }
    const bool fold = (jb.pass_mask >> limb) & 1;
#pragma unroll
    for (int c = 0; c < C; c++) {
        VH_GLOBAL uint64_t *out = vh_global(jb.out[c] + (size_t)limb * n + x0);
        const bool add = fold && jb.pass[c];
        uint64_t w[8];
        if (add) {   // |acc| <= q/2 + 4 (q + 2^47) and |P d| <= 3q/4: the sum stays below 2^53
            const VH_GLOBAL uint64_t *ps = vh_global(jb.pass[c] + (size_t)limb * n + x0);
#pragma unroll
            for (int h = 0; h < 4; h++) vh_ld2(ps + 128 * (h >> 1) + 2 * (h & 1), w[2 * h], w[2 * h + 1]);
        }
        const double2 pm = add ? jb.pmod[limb] : make_double2(0.0, 0.0);
#pragma unroll
        for (int m = 0; m < 8; m++) {
            double y = jb.add ? acc[c][m] : -acc[c][m];
            if (add) y += vh_mulmod_tw(vh_u2d(w[m]), pm.x, pm.y, q);
            w[m] = vh_d2u(vh_canon(y, q, qinv));
        }
#pragma unroll
        for (int h = 0; h < 4; h++) vh_st2(out + 128 * (h >> 1) + 2 * (h & 1), w[2 * h], w[2 * h + 1]);
    }
}

hipError_t vh_launch_row_mac(hipStream_t st, const vh_mac_job *jobs, unsigned njobs, unsigned next,
                             const vh_limb *limbs, const uint64_t *const *kptr, int logn, int comps)
{
    if (logn < 13 || logn > 16 || comps < 1 || comps > 2) return hipErrorInvalidValue;
    const dim3 grid(njobs, 1u << (logn - 11), next);
    const int xcd = (grid.y * grid.z) % 8 == 0;
    if (comps == 1) VH_KL(k_row_mac<1>, grid, dim3(256), 0, st, jobs, limbs, kptr, logn, xcd);
    else VH_KL(k_row_mac<2>, grid, dim3(256), 0, st, jobs, limbs, kptr, logn, xcd);
    return hipGetLastError();
}
