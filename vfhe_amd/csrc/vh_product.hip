// vh_product.hip -- the fused product's middle kernel, FP64 path (N = 2^13 .. 2^16).
#include "vh_kernels.h"
#include "vh_row8.h"

// ---------------------------------------------------------------------------
// z = INTT(NTT(x) * NTT(y)): after the forward column passes of x (in it.src) and y (in it.src2), one
// kernel runs the forward row stages of both, the pointwise product and the inverse row stages,
// and writes the input of the inverse column pass to it.dst.  The transformed operands never return
// to memory.
//
// Rows run as in vh_row8.h.  A workgroup takes rows 4 y .. 4 y + 3 and their mirrors at the other end,
// so that the inverse finds its twiddles among the forward ones formed for the partner row: one
// table instead of two, and 78 VGPRs, four workgroups per
// CU, whose loads and butterflies overlap without an explicit prefetch.
// Measured for 64 pairs x 24 limbs of 2^16 (2.4 GB to read and write, 0.48 ms at the rate of a large
// copy; 0.3 ms of FP64 issue): 0.56 .. 0.71 ms, against 0.67 .. 0.83 ms for persistent workgroups
// with 16 values per thread, separate inverse tables and 234 VGPRs.
// Grid: x = tile, y = item.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256, 4)
k_row_mul(const vh_item *__restrict__ items, const vh_limb *__restrict__ limbs, int logn)
{
    constexpr int ROWS = vh_row8::ROWS, S = vh_row8::S, T = vh_row8::T;
    __shared__ double lds[ROWS * vh_row8::PITCH];
    __shared__ double tws[ROWS][S];
    const vh_item &it = items[blockIdx.y];
    const vh_limb &L = limbs[it.limb];
    const int g = threadIdx.x / T, last = (1 << (logn - 8)) - 1, r0 = (int)blockIdx.x * (ROWS / 2);
    auto sub = [&](int r) { return r < ROWS / 2 ? r0 + r : last - (r0 + r - ROWS / 2); };
    const size_t at = (size_t)sub(g) * S + threadIdx.x % T;
    double v[2][8];
    {
        const VH_GLOBAL uint64_t *x = vh_global(it.src) + at, *y = vh_global(it.src2) + at;
#pragma unroll
        for (int m = 0; m < 8; m++) v[0][m] = __longlong_as_double((long long)vh_ld(x + T * m));
#pragma unroll
        for (int m = 0; m < 8; m++) v[1][m] = __longlong_as_double((long long)vh_ld(y + T * m));
    }
    vh_row8::fill(tws, L, sub);
    __syncthreads();
    const vh_row8 row(L, lds, tws);
    const double q = L.qd, qinv = L.qinv;
    row.fwd(v);
    // pointwise product of centred operands (|.| <= q/2 + 1), centred
#pragma unroll
    for (int m = 0; m < 8; m++) {
        const double x = row.centre(v[0][m]), y = row.centre(v[1][m]);
        const double hi = x * y;
        const double lo = __fma_rn(x, y, -hi);
        const double qt = __fma_rn(x, y * qinv, VH_MAGIC) - VH_MAGIC;
        v[0][m] = row.centre(__fma_rn(-qt, q, hi) + lo);
    }
    row.inv(v[0], tws[g ^ (ROWS / 2)]);
    VH_GLOBAL uint64_t *out = vh_global(it.dst) + at;
#pragma unroll
    for (int m = 0; m < 8; m++) vh_st(out + T * m, (uint64_t)__double_as_longlong(row.centre(v[0][m])));
}

hipError_t vh_launch_row_mul(hipStream_t st, const vh_item *items, unsigned nitems, const vh_limb *limbs, int logn)
{
    if (logn < 13 || logn > 16) return hipErrorInvalidValue;
    VH_KL(k_row_mul, dim3(1u << (logn - 11), nitems), dim3(256), 0, st, items, limbs, logn);
    return hipGetLastError();
}
