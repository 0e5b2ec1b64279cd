// vh_keyswitch.hip -- key-switch kernels of the FP64 path: the inner product fused into the forward row
// pass of the ModUp digits (N = 2^13 .. 2^16, at most two output components), and the ModDown.
#include "vh_kernels.h"
#include "vh_row8.h"

// ---------------------------------------------------------------------------
// The column pass has left the lifted digit rows, transformed over their first
// logn - 8 stages, in jb.modup; this kernel finishes the last 8 stages of every digit
// for one tile of 8 rows of 256 elements and accumulates
//     out_c = -+ sum_d NTT(digit_d) * key[d][c]      (the mul_subto of gadget.c:22-37)
// in registers, so the transformed digits never return to memory.
//
// Rows run as in vh_row8.h.  Its last phase leaves four adjacent elements per lane, so the key rows,
// the pass-through rows and the output move as 16-byte words of one contiguous kilobyte per 32
// lanes.  (16 values per thread ending in 16 contiguous elements made every key load touch 64
// separate 128-byte lines.)
// 8 values and two accumulators per thread leave room to load a digit's key words and the
// next digit before the butterflies within 128 VGPRs: four workgroups per CU.
// Measured for 32 ciphertexts at N = 2^16, 24 + 4 limbs (11.7 GB to read and write, 2.2 ms of
// FP64 issue): 5.54 ms with 16 values per thread and contiguous key reads, 4.75 ms with those
// values regrouped before the key reads, 3.80 ms in this form (3.1 TB/s).
//
// Grid: x = ciphertext, y = tile, z = extended limb.  A key block is (y, z).
// Consecutive workgroups are dealt round-robin over the 8 XCDs, so with `xcd` set the
// workgroup index is remapped to put all ciphertexts of one key block on one XCD, one after
// another: each XCD's L2 then fetches a key block once instead of every XCD fetching it.
// Spreading a job's digits over several workgroups (partial sums added by a second kernel) was
// measured on launches of 60 to 300 workgroups and gained nothing: the digit loop keeps its loads
// in flight, and the partials' traffic costs what the extra workgroups save.
// ---------------------------------------------------------------------------
template <int C>
__global__ void __launch_bounds__(256, 4)
k_row_mac(const vh_mac_job *__restrict__ jobs, const vh_limb *__restrict__ limbs,
          const uint64_t *const *__restrict__ kptr, int logn, int xcd)
{
    constexpr int ROWS = vh_row8::ROWS, S = vh_row8::S, T = vh_row8::T;
    __shared__ double lds[ROWS * vh_row8::PITCH];
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
    vh_row8::fill(tws, L, [&](int r) { return by * ROWS + r; });
    __syncthreads();
    const vh_row8 row(L, lds, tws);
    const size_t rowoff = sub * S, x0 = rowoff + 4 * t;
    const VH_GLOBAL uint64_t *dig = vh_global(jb.modup + (size_t)ti * n + rowoff + t);
    const size_t dstep = (size_t)jb.next * n;
    const uint64_t *const *kp = kptr + jb.kptr_off + (size_t)ti * D * C;

    double acc[C][8];
#pragma unroll
    for (int c = 0; c < C; c++)
#pragma unroll
        for (int m = 0; m < 8; m++) acc[c][m] = 0.0;
    uint64_t raw[8];
    if (D > 0) {
#pragma unroll
        for (int m = 0; m < 8; m++) raw[m] = vh_ld(dig + 32 * m);
    }
    for (int d = 0; d < D; d++, kp += C) {
        double v[1][8];
#pragma unroll
        for (int m = 0; m < 8; m++) v[0][m] = __longlong_as_double((long long)raw[m]);
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
        row.fwd(v);
        const bool fourth = (d & 3) == 3;
#pragma unroll
        for (int m = 0; m < 8; m++) {
            const double a = row.centre(v[0][m]);                  // |a| <= q/2 + 1
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

// ---------------------------------------------------------------------------
// ModDown of a key-switch output component, with the pass-through add, and with RESC the CKKS
// rescale that follows, on the FP64 path (every limb below 2^50, at most 4 special primes).  The K
// sequential round divisions of the reference (rns_polynomial.c:939-976, ascending special primes,
// then the rescale prime) are affine in the row values and in the carried t_k = (special row k after
// the divisions before it + floor(p_k/2)) mod p_k, so with the products of inverses folded into
// per-limb constants (built on the host, exact):
//   t_k   = canon(v_k G_k + c_k + sum_{j<k} t_j g_kj)                                mod p_k
//   t_r   = canon(x_r X_r + add_r + C_r + sum_k t_k T_rk)                            mod q_r
//   out_i = canon(x_i X_i + add_i A_i + C_i + t_r R_i + sum_k t_k T_ik)              mod q_i
// and without the rescale  out_i = canon(x_i X_i + C_i + sum_k t_k T_ik) + add_i.
// Each product is vh_mulmod_tw against a centred constant ({w, RN(w/q)}): |term| <= 3q/4, so with
// K <= 4 every sum stays below 6q < 2^53 and the result is the reference's, bit for bit.  Constant
// rows (stride VH_MDR_W double2): rows 0..3 the special primes [G, c, g_k0..g_k3], then row 4 +
// limb for every limb of the pool [X, A, C, R, T_0..T_3] (C in .x only).
//
// A thread owns two adjacent coefficients (16-byte accesses).  Bound by HBM at large batches.  A launch of
// few workgroups runs its output limbs one after another and waits for memory at each, so the
// limbs are then divided over gridDim.z slices, each forming the chain t again (64 workgroups for one
// multiply at N = 2^14, 11 + 4 limbs: 16 us in one slice).  With one slice the divided rows are cleared
// here; with more, another slice may still read them and the caller clears them.
// ---------------------------------------------------------------------------
template <bool RESC>
__global__ void __launch_bounds__(256)
k_moddown_fp(const vh_mdr_job *__restrict__ jobs, const vh_limb *__restrict__ limbs, const double2 *__restrict__ cs,
             unsigned n)
{
    constexpr int KMAX = 4, W = VH_MDR_W;
    const vh_mdr_job &jb = jobs[blockIdx.y];
    const unsigned x = (blockIdx.x * 256 + threadIdx.x) * 2;
    if (x >= n) return;
    const int K = jb.K;
    VH_GLOBAL uint64_t *base = vh_global(jb.base);
    const VH_GLOBAL uint64_t *add = jb.add ? vh_global(jb.add) : nullptr;
    auto at = [&](int limb) -> size_t { return (size_t)limb * jb.stride + x; };
    double t[KMAX][2];
#pragma unroll
    for (int k = 0; k < KMAX; k++) {
        if (k >= K) continue;   // (continue, not break: the loop unrolls fully)
        const int lk = jb.div_limb[k];
        const vh_limb &L = limbs[lk];
        const double2 *c = cs + k * W;
        uint64_t v[2];
        vh_ld2(base + at(lk), v[0], v[1]);
#pragma unroll
        for (int e = 0; e < 2; e++) {
            double s = c[1].x + vh_mulmod_tw(vh_u2d(v[e]), c[0].x, c[0].y, L.qd);
#pragma unroll
            for (int j = 0; j < KMAX; j++)
                if (j < k) s += vh_mulmod_tw(t[j][e], c[2 + j].x, c[2 + j].y, L.qd);
            t[k][e] = vh_canon(s, L.qd, L.qinv);
        }
    }
    double tr[2];
    if (RESC) {
        const int lr = jb.resc;
        const vh_limb &L = limbs[lr];
        const double2 *c = cs + (KMAX + lr) * W;
        uint64_t v[2], a[2] = {0, 0};
        vh_ld2(base + at(lr), v[0], v[1]);
        if (add) vh_ld2(add + at(lr), a[0], a[1]);
#pragma unroll
        for (int e = 0; e < 2; e++) {
            double s = c[2].x + vh_mulmod_tw(vh_u2d(v[e]), c[0].x, c[0].y, L.qd) + vh_u2d(a[e]);
#pragma unroll
            for (int k = 0; k < KMAX; k++)
                if (k < K) s += vh_mulmod_tw(t[k][e], c[4 + k].x, c[4 + k].y, L.qd);
            tr[e] = vh_canon(s, L.qd, L.qinv);
        }
    }
    const int per = (jb.nout + (int)gridDim.z - 1) / (int)gridDim.z;
    const int o0 = (int)blockIdx.z * per, o1 = o0 + per < jb.nout ? o0 + per : jb.nout;
    for (int o = o0; o < o1; o++) {
        const int li = jb.out_limb[o];
        const vh_limb &L = limbs[li];
        const double2 *c = cs + (KMAX + li) * W;
        uint64_t v[2], a[2] = {0, 0}, r[2];
        vh_ld2(base + at(li), v[0], v[1]);
        if (add) vh_ld2(add + at(li), a[0], a[1]);
#pragma unroll
        for (int e = 0; e < 2; e++) {
            double s = c[2].x + vh_mulmod_tw(vh_u2d(v[e]), c[0].x, c[0].y, L.qd);
            if (RESC) {
                s += vh_mulmod_tw(tr[e], c[3].x, c[3].y, L.qd);
                if (add) s += vh_mulmod_tw(vh_u2d(a[e]), c[1].x, c[1].y, L.qd);
            }
#pragma unroll
            for (int k = 0; k < KMAX; k++)
                if (k < K) s += vh_mulmod_tw(t[k][e], c[4 + k].x, c[4 + k].y, L.qd);
            r[e] = vh_d2u(vh_canon(s, L.qd, L.qinv));
            if (!RESC && add) r[e] = vh_reduce64(r[e] + a[e], L.q, L.mu64);   // any 64-bit addend, as the elementwise add
        }
        vh_st2(base + at(li), r[0], r[1]);
    }
    if (gridDim.z == 1) {
        for (int k = 0; k < K; k++) vh_st2(base + at(jb.div_limb[k]), 0, 0);
        if (RESC) vh_st2(base + at(jb.resc), 0, 0);
    }
}

// slices: output-limb slices (1: the kernel clears the divided rows).
hipError_t vh_launch_moddown_fp(hipStream_t st, const vh_mdr_job *jobs, unsigned njobs, const vh_limb *limbs,
                                const void *cs, uint64_t n, int resc, unsigned slices)
{
    if (n < 2 || n > (1u << 30) || (n & 1) || slices < 1) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((n + 511) / 512), njobs, slices);
    if (resc) VH_KL(k_moddown_fp<true>, grid, dim3(256), 0, st, jobs, limbs, (const double2 *)cs, (unsigned)n);
    else VH_KL(k_moddown_fp<false>, grid, dim3(256), 0, st, jobs, limbs, (const double2 *)cs, (unsigned)n);
    return hipGetLastError();
}
