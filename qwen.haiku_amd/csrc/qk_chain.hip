// qk_chain.hip -- the elementwise links of a decode layer's chain on the
// device (gfx950): residual add + RMSNorm (+ Q8_K of the result), SiLU,
// and SiLU(gate) * up (+ Q8_K), so activations stay in HBM between the
// quantized GEMVs.
//
// Bit-exact restatements of the reference's host code: every float op is
// one IEEE operation with round-to-nearest-even, in the reference's order
// (this file is built with -ffp-contract=off; the only fused multiply-adds
// are the explicit ones inside qk_expf).
#include "qk.h"
#include "qk_dev.h"
#include "qk_expf.h"
#include "qk_kernels.h"

namespace qk {

// v / (1 + expf(-v)): simd_silu_f32's x86 path (simd/simd.c:265-276),
// the same formula as tensor_silu (slm/tensor.c:310-318).
// tab: a copy of qk_expf's table.
__device__ __forceinline__ float silu(float v, const uint64_t *tab) {
    return __fdiv_rn(v, __fadd_rn(1.0f, qk_expf_tab(-v, tab)));
}

// ---- the norm's sequential double sum ----------------------------------
// tensor_rms_norm adds (double)(r_i * r_i) to a double in index order
// (slm/tensor.c:357-360), rounding after every add. The chain of k adds is
// cut into segments of four terms, one per lane. Every segment's start is
// guessed (a scan of the segment sums, whose roundings differ from the
// chain's now and then), every lane runs its own four adds from its guess,
// and the guesses are checked: the first segment's start (0) is right, and
// a segment whose start is right ends right, so when each end equals the
// next start bit for bit the last end is the chain's. At the first end that
// differs, the next start takes it and the later guesses move by the same
// difference; every such step fixes at least one more segment, so the loop
// ends for any input (infinities and NaN included).
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ double dpp64(double v) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROWS, 0xF, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROWS, 0xF, true);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

__device__ __forceinline__ double readlane64(double v, int l) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Inclusive sums over the lanes (lanes past a row boundary get the row
// totals before them by row_bcast). Only the first 16 lanes if `one_row`.
__device__ __forceinline__ double wave_scan64(double v, bool one_row) {
    v = __dadd_rn(v, dpp64<0x111>(v));                // row_shr:1
    v = __dadd_rn(v, dpp64<0x112>(v));                // row_shr:2
    v = __dadd_rn(v, dpp64<0x114>(v));                // row_shr:4
    v = __dadd_rn(v, dpp64<0x118>(v));                // row_shr:8
    if (!one_row) {
        v = __dadd_rn(v, dpp64<0x142, 0xA>(v));       // row_bcast:15 into rows 1 and 3
        v = __dadd_rn(v, dpp64<0x143, 0xC>(v));       // row_bcast:31 into rows 2 and 3
    }
    return v;
}

__device__ __forceinline__ bool same_bits(double a, double b) {
    return __double_as_longlong(a) == __double_as_longlong(b);
}

// The guesses after segment f (lanes above f) once f's end is known.
__device__ __forceinline__ double move_starts(double st, double end, int f, int lane) {
    const double was = readlane64(st, f + 1), by = __dsub_rn(end, was);
    const bool finite = fabs(by) <= 1.0e308;
    const double moved = finite ? __dadd_rn(st, by) : end;
    return lane <= f ? st : (lane == f + 1 ? end : moved);
}

// One wave's block of 256 terms from `start`: lane l adds its terms t0 .. t3
// after lanes 0 .. l - 1. q: the exclusive sums of the lanes before. Returns
// the block's end (of the last lane), exact for that start.
__device__ __forceinline__ double block_chain(double start, double q, double t0, double t1, double t2, double t3,
                                              int lane) {
    double st = lane == 0 ? start : __dadd_rn(start, q);
    for (;;) {
        const double e = __dadd_rn(__dadd_rn(__dadd_rn(__dadd_rn(st, t0), t1), t2), t3);
        const double next = dpp64<0x130>(st);         // wave_shl:1
        const uint64_t off = __ballot(lane < 63 && !same_bits(e, next));
        if (off == 0) return readlane64(e, 63);
        const int f = __builtin_ctzll(off);
        st = move_starts(st, readlane64(e, f), f, lane);
    }
}

// tensor_add (slm/tensor.c:284-291) of an optional delta, then
// tensor_rms_norm (slm/tensor.c:345-367) of the sum, then optionally
// quantize_row_q8_K (slm/tensor.c:683-720) of the normalized row:
//   r      = h + delta                      (stored to h_out if given)
//   ssq    = sum over i of (double)(r_i * r_i), in index order (see above)
//   rscale = 1 / sqrtf((float)(ssq / k) + eps)
//   x_i    = (r_i * rscale) * w_i           (stored to x_out if given)
// One workgroup per row; wave v owns the 256-element blocks v, v + W, ...
// (W waves, NB blocks each), four consecutive elements per lane, kept in
// registers from the loads (h, delta and w all in flight at once) to the
// stores. What bounds a decode row is latency: one round of loads, two
// barriers (block totals; block ends), one division and square root.
// Against one lane walking the squares in blocks of 64 (a block whose adds
// round went term by term): 1 x 1024 5.80 -> 2.40 us a launch, 512 x 1024
// 12.9 -> 3.8 us.
template <int NB>
__global__ __launch_bounds__(1024) void k_add_rmsnorm(const float *h, const float *delta,
                                                      const float *__restrict__ w, float eps, int k, float *h_out,
                                                      float *x_out, uint8_t *__restrict__ xq) {
    __shared__ double total[QK_NORM_MAX_K / QK_K], ends[QK_NORM_MAX_K / QK_K];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, W = blockDim.x >> 6;
    const int nblk = (k + QK_K - 1) / QK_K;
    const int64_t row = (int64_t)blockIdx.x * k;
    float4 r[NB], g[NB];
    {
        float4 a[NB];
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int i = (wave + W * b) * QK_K + 4 * lane;
            r[b] = a[b] = g[b] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (i < k) {                              // k is a multiple of 4
                r[b] = *reinterpret_cast<const float4 *>(h + row + i);
                if (delta) a[b] = *reinterpret_cast<const float4 *>(delta + row + i);
                g[b] = *reinterpret_cast<const float4 *>(w + i);
            }
        }
        if (delta)
#pragma unroll
            for (int b = 0; b < NB; b++)
                r[b] = make_float4(__fadd_rn(r[b].x, a[b].x), __fadd_rn(r[b].y, a[b].y), __fadd_rn(r[b].z, a[b].z),
                                   __fadd_rn(r[b].w, a[b].w));
    }
    double t[NB][4], q[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int i = (wave + W * b) * QK_K + 4 * lane;
        if (h_out && i < k) *reinterpret_cast<float4 *>(h_out + row + i) = r[b];
        t[b][0] = (double)__fmul_rn(r[b].x, r[b].x);
        t[b][1] = (double)__fmul_rn(r[b].y, r[b].y);
        t[b][2] = (double)__fmul_rn(r[b].z, r[b].z);
        t[b][3] = (double)__fmul_rn(r[b].w, r[b].w);
        const double own = __dadd_rn(__dadd_rn(t[b][0], t[b][1]), __dadd_rn(t[b][2], t[b][3]));
        const double incl = wave_scan64(own, false);
        q[b] = dpp64<0x138>(incl);                    // wave_shr:1
        if (lane == 63 && wave + W * b < nblk) total[wave + W * b] = incl;
    }
    __syncthreads();
    // lane b of every wave: the guessed start of block b
    double starts = dpp64<0x138>(wave_scan64(lane < nblk ? total[lane] : 0.0, nblk <= 16));
    double ssq;
    for (;;) {                                        // uniform: every wave sees the same ends
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int blk = wave + W * b;
            if (blk < nblk) {
                const double e = block_chain(readlane64(starts, blk), q[b], t[b][0], t[b][1], t[b][2], t[b][3], lane);
                if (lane == 0) ends[blk] = e;
            }
        }
        __syncthreads();
        const double e = lane < nblk ? ends[lane] : 0.0;
        const double next = dpp64<0x130>(starts);
        const uint64_t off = __ballot(lane < nblk - 1 && !same_bits(e, next));
        if (off == 0) {
            ssq = readlane64(e, nblk - 1);
            break;
        }
        const int f = __builtin_ctzll(off);
        starts = move_starts(starts, readlane64(e, f), f, lane);
        __syncthreads();                              // the ends are rewritten
    }
    // ssq / k; for a power of two the product with 1 / k is the same value
    const double mean = (k & (k - 1)) == 0 ? __dmul_rn(ssq, 1.0 / (double)k) : __ddiv_rn(ssq, (double)k);
    // __builtin_sqrtf is the correctly rounded square root (the raw
    // v_sqrt_f32 that __fsqrt_rn maps to is not)
    const float rscale = __fdiv_rn(1.0f, __builtin_sqrtf(__fadd_rn(__double2float_rn(mean), eps)));
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int blk = wave + W * b, i = blk * QK_K + 4 * lane;
        if (blk >= nblk) break;                       // whole wave
        const float e[4] = {__fmul_rn(__fmul_rn(r[b].x, rscale), g[b].x),
                            __fmul_rn(__fmul_rn(r[b].y, rscale), g[b].y),
                            __fmul_rn(__fmul_rn(r[b].z, rscale), g[b].z),
                            __fmul_rn(__fmul_rn(r[b].w, rscale), g[b].w)};
        if (x_out && i < k) *reinterpret_cast<float4 *>(x_out + row + i) = make_float4(e[0], e[1], e[2], e[3]);
        if (xq) {                                     // k % 256 == 0: every lane is in range
            uint32_t packed, bs;
            float d;
            q8k_block_wave(e, lane, packed, d, bs);
            uint8_t *out = xq + ((int64_t)blockIdx.x * nblk + blk) * Q8K_BYTES;
            reinterpret_cast<uint32_t *>(out + 4)[lane] = packed;
            if ((lane & 7) == 0) reinterpret_cast<uint32_t *>(out + 260)[lane >> 3] = bs;
            if (lane == 0) *reinterpret_cast<float *>(out) = d;
        }
    }
}

// simd_silu_f32 (simd/simd.c:271-277) over n floats; dst may equal src.
__global__ __launch_bounds__(256) void k_silu(const float *src, float *dst, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        dst[i] = silu(src[i], qk_exp2_32);
}

// The FFN's SwiGLU link: simd_silu_f32 of the gate then tensor_mul
// (slm/tensor.c:293-300) by up (slm/qwen.c:949-954), optionally
// quantized to Q8_K for the down projection. One wave per 256 elements
// of the flattened m x k rows (k a multiple of 256 with xq; of 4
// without), 4 consecutive elements per lane.
__global__ __launch_bounds__(256) void k_swiglu(const float *__restrict__ gate, const float *__restrict__ up,
                                                int64_t n, float *__restrict__ act, uint8_t *__restrict__ xq) {
    // the table in LDS: read while the rows arrive, instead of a trip to
    // memory after them (1 x 3584 2.36 -> 2.26 us, 512 x 3584 4.64 -> 4.54)
    __shared__ uint64_t tab[32];
    const int lane = threadIdx.x & 63;
    const int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int64_t i = b * 64 + lane;                   // float4 index
    float4 g = make_float4(0.0f, 0.0f, 0.0f, 0.0f), u = g;
    if (i * 4 < n) {
        g = reinterpret_cast<const float4 *>(gate)[i];
        u = reinterpret_cast<const float4 *>(up)[i];
    }
    if (threadIdx.x < 32) tab[threadIdx.x] = qk_exp2_32[threadIdx.x];
    __syncthreads();
    if (b * QK_K >= n) return;                         // whole wave
    const float e[4] = {__fmul_rn(silu(g.x, tab), u.x), __fmul_rn(silu(g.y, tab), u.y),
                        __fmul_rn(silu(g.z, tab), u.z), __fmul_rn(silu(g.w, tab), u.w)};
    if (act && i * 4 < n) reinterpret_cast<float4 *>(act)[i] = make_float4(e[0], e[1], e[2], e[3]);
    if (xq) {                                          // n % 256 == 0: every lane is in range
        uint32_t packed, bs;
        float d;
        q8k_block_wave(e, lane, packed, d, bs);
        uint8_t *out = xq + b * Q8K_BYTES;
        reinterpret_cast<uint32_t *>(out + 4)[lane] = packed;
        if ((lane & 7) == 0) reinterpret_cast<uint32_t *>(out + 260)[lane >> 3] = bs;
        if (lane == 0) *reinterpret_cast<float *>(out) = d;
    }
}

// ---- launchers ---------------------------------------------------------
// One wave per 256-element block up to 16 waves, then several blocks each.
// A dispatch counts its work-items in 32 bits, so more than 2^21 rows of
// up to 1024 threads go out in several launches.
hipError_t launch_add_rmsnorm(const float *h, const float *delta, const float *w, float eps, int64_t m, int64_t k,
                              float *h_out, float *x_out, uint8_t *xq, hipStream_t s) {
    const int nblk = (int)((k + QK_K - 1) / QK_K), waves = nblk < 16 ? nblk : 16;
    auto kernel = nblk <= 16 ? k_add_rmsnorm<1> : nblk <= 32 ? k_add_rmsnorm<2> : k_add_rmsnorm<4>;
    const int64_t rows = (int64_t)1 << 21;
    for (int64_t t = 0; t < m; t += rows) {
        const unsigned grid = (unsigned)(m - t < rows ? m - t : rows);
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * waves), 0, s, h + t * k, delta ? delta + t * k : nullptr, w,
                           eps, (int)k, h_out ? h_out + t * k : nullptr, x_out ? x_out + t * k : nullptr,
                           xq ? xq + t * nblk * Q8K_BYTES : nullptr);
    }
    return hipGetLastError();
}

hipError_t launch_silu(const float *src, float *dst, int64_t n, hipStream_t s) {
    const int64_t want = (n + 255) / 256;
    const unsigned grid = (unsigned)(want < 8192 ? want : 8192);
    hipLaunchKernelGGL(k_silu, dim3(grid), dim3(256), 0, s, src, dst, n);
    return hipGetLastError();
}

hipError_t launch_swiglu(const float *gate, const float *up, int64_t n, float *act, uint8_t *xq, hipStream_t s) {
    const int64_t waves = (n + QK_K - 1) / QK_K;
    hipLaunchKernelGGL(k_swiglu, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, gate, up, n, act, xq);
    return hipGetLastError();
}

}  // namespace qk
