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
// cut into segments of four terms, one per lane, and blocks of 64 segments.
// First every segment's start is guessed (a scan of the segment sums, whose
// roundings differ from the chain's now and then), every lane runs its own
// four adds from its guess, and the guesses are checked: the first segment's
// start (0) is right, and a segment whose start is right ends right, so when
// each end equals the next start bit for bit the last end is the chain's.
// At the first end that differs, the next start takes it and the later
// guesses move by the same difference. A few such steps settle a row whose
// sum seldom rounds (most Gaussian ones: none). Every step costs a pass over
// the block (0.09 us), so a row that rounds often (outliers among ordinary
// values) gets NORM_MOVES of them per block, NORM_MOVES_ON where a block moved,
// and NORM_ROUNDS over the blocks; then the rest of the row is added exactly
// (exact_from). One Gaussian block in 400000 needs more than ten. Rows with
// every 400th element 3000, Gaussian else, us a launch: 1 x 1024 6, 4096 12,
// 16384 28; by such steps alone 7 to 10, 62, 1150; by one lane, term by term,
// 13, 47, 182. (Only rows of 256 of widely different terms take longer so than
// on one lane: 5 to 8 us against 5.)
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

__device__ __forceinline__ uint64_t bits64(double v) { return (uint64_t)__double_as_longlong(v); }
__device__ __forceinline__ double double64(uint64_t b) { return __longlong_as_double((long long)b); }

__device__ __forceinline__ double add4(double s, const double (&t)[4]) {
    return __dadd_rn(__dadd_rn(__dadd_rn(__dadd_rn(s, t[0]), t[1]), t[2]), t[3]);
}

__device__ __forceinline__ void squares(float4 r, double (&t)[4]) {
    t[0] = (double)__fmul_rn(r.x, r.x);
    t[1] = (double)__fmul_rn(r.y, r.y);
    t[2] = (double)__fmul_rn(r.z, r.z);
    t[3] = (double)__fmul_rn(r.w, r.w);
}

constexpr int NORM_WAVES = 16;                         // of a workgroup, at most
constexpr int NORM_MOVES = 10, NORM_MOVES_ON = 4, NORM_ROUNDS = 5;

// The guesses after segment f (lanes above f) once f's end is known.
__device__ __forceinline__ double move_starts(double st, double end, int f, int lane) {
    const double was = readlane64(st, f + 1), by = __dsub_rn(end, was);
    const bool finite = fabs(by) <= 1.0e308;
    const double moved = finite ? __dadd_rn(st, by) : end;
    return lane <= f ? st : (lane == f + 1 ? end : moved);
}

// One wave's block of 256 terms, four per lane, the lanes' guessed starts in
// st (moved on as they are found wrong). Lane 63's value is the block's end,
// exact for lane 0's start unless a guess is still wrong: the ends are right
// up to lane `open` then (64: all).
__device__ __forceinline__ double check_block(double &st, const double (&t)[4], int lane, int most, int &open) {
    for (int m = 0;; m++) {
        const double e = add4(st, t), next = dpp64<0x130>(st);   // wave_shl:1, in every lane
        const uint64_t off = __ballot((lane < 63) & !same_bits(e, next));
        open = off ? (int)__builtin_ctzll(off) : 64;
        if (__builtin_expect(off == 0 || m == most, 1)) return e;
        st = move_starts(st, readlane64(e, open), open, lane);
    }
}

// One step of pair_scan (below): the lane's segments after those of the lane
// that the DPP control reads (lanes without one: after none, the bases).
template <int CTRL, int ROWS>
__device__ __forceinline__ void pair_step(double (&c)[2], const double (&base)[2]) {
    const double d0 = __dsub_rn(c[0], base[0]), d1 = __dsub_rn(c[1], base[1]);
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const uint64_t b = bits64(base[p]), own = bits64(c[p]);
        const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)b, (int)(uint32_t)own, CTRL, ROWS, 0xF, false);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)(b >> 32), (int)(uint32_t)(own >> 32), CTRL,
                                                                  ROWS, 0xF, false);
        c[p] = __dadd_rn(double64((uint64_t)hi << 32 | lo), lo & 1 ? d1 : d0);
    }
}

// A block's segments in the binade [2^E, 2^(E+1)) of `at` (finite, above 0).
// A sum in it is a multiple of u = 2^(E-52), and an add of t moves it by t
// rounded to a multiple of u, which depends on the sum only where t ends in
// exactly u/2, and then on the sum's parity alone. So a segment is two
// numbers, its sum from an even start (2^E) and from an odd one (2^E + u),
// and two neighbours combine by the parity in between (every such add is
// exact). c: lane l's sums over the segments of lanes `from` .. l, right
// while they stay in the binade; past it they are no smaller than 2^(E+1).
// (The same on the doubles' bits, as 64-bit integers, took 1.7 times as long.)
struct Pair {
    double base[2], c[2];
    // the sum from s, of the same binade
    __device__ __forceinline__ double after(double s) const {
        return __dadd_rn(s, bits64(s) & 1 ? __dsub_rn(c[1], base[1]) : __dsub_rn(c[0], base[0]));
    }
    __device__ __forceinline__ bool within(double end) const { return end < __dadd_rn(base[0], base[0]); }
};

__device__ __forceinline__ uint64_t binade(double v) { return bits64(v) & (0x7ffull << 52); }

__device__ __forceinline__ Pair pair_scan(double at, const double (&t)[4], int lane, int from) {
    Pair r;
#pragma unroll
    for (int p = 0; p < 2; p++) {
        r.base[p] = double64(binade(at) + p);
        r.c[p] = lane >= from ? add4(r.base[p], t) : r.base[p];
    }
    pair_step<0x111, 0xF>(r.c, r.base);                // row_shr:1
    pair_step<0x112, 0xF>(r.c, r.base);                // row_shr:2
    pair_step<0x114, 0xF>(r.c, r.base);                // row_shr:4
    pair_step<0x118, 0xF>(r.c, r.base);                // row_shr:8
    pair_step<0x142, 0xA>(r.c, r.base);                // row_bcast:15 into rows 1 and 3
    pair_step<0x143, 0xC>(r.c, r.base);                // row_bcast:31 into rows 2 and 3
    return r;
}

// The chain over one wave's block of 256 terms from s, exact for any terms.
// The first segment whose end leaves the binade starts right, so its own
// four adds end right, and the lanes after it go on from there in the new
// binade. A row's squares span 277 binades. A scan (0.45 us) costs about as
// much as NORM_NEAR segments one by one (an add waits 11 ns for the one
// before), so that is how the segments up to a near crossing go, and the whole
// block where more than NORM_MANY are crossed.
constexpr int NORM_NEAR = 9, NORM_MANY = 7;

__device__ __forceinline__ double block_exact(double s, const double (&t)[4], int lane, int from) {
    const double own = add4(0.0, t);                   // 0 only if every term is
    while (from < 64) {                                // lanes below `from` are in s; uniform
        if (s != s) return s;
        uint64_t out, crossed;                         // segments that leave the binade; that seem to, past the first
        double start = s, end = s;
        if (!(s > 0.0 && s < __builtin_inf())) {       // 0: the first term that isn't; inf: the first NaN
            out = __ballot(lane >= from && (s == 0.0 ? !(own == 0.0) : own != own));
            crossed = s == 0.0 ? 0xfeull << __builtin_ctzll(out | 1ull << 63) : 0;   // a sum that begins soon doubles
        } else {
            const Pair p = pair_scan(s, t, lane, from);
            end = p.after(s);
            const double before = dpp64<0x138>(end);   // wave_shr:1
            start = lane == 0 ? s : before;
            out = __ballot(!p.within(end));
            crossed = __ballot(binade(start) != binade(end));
        }
        if (out == 0) return readlane64(end, 63);
        const int f = __builtin_ctzll(out);
        s = readlane64(add4(start, t), f);
        from = f + 1;
        if (from < 64) {
            crossed = crossed >> from << from;
            int to = from;
            if (__builtin_popcountll(crossed) > NORM_MANY) to = 64;
            else
                while (crossed && (int)__builtin_ctzll(crossed) < to + NORM_NEAR) {
                    to = __builtin_ctzll(crossed) + 1;
                    crossed &= crossed - 1;
                }
            double v[4], next[4];
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = readlane64(t[i], from);
            for (; from < to; from++) {
#pragma unroll
                for (int i = 0; i < 4; i++) next[i] = readlane64(t[i], (from + 1) & 63);
                s = add4(s, v);
#pragma unroll
                for (int i = 0; i < 4; i++) v[i] = next[i];
            }
        }
    }
    return s;
}

// The end of a row's chain from `sum` at the start of block `first` on, by
// the whole workgroup: every block's sums in the binade of its guessed start
// (lane b of `starts`: block b's) by the block's wave; then wave 0 goes from
// block to block, and where the sum is in another binade or leaves it runs
// the block. row: the row in LDS (each wave's blocks written by itself).
// pairs: two doubles a block and one more. Of block `first`, the lanes below
// `from` are known to end at `sure`.
__device__ __forceinline__ double exact_from(const float4 *row, double *pairs, double starts, double sum, int first,
                                             int nblk, int W, int from, double sure) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool scan = nblk - first > 1;
    double u[4];
    for (int blk = wave; blk < nblk; blk += W) {
        if (blk < first || !scan) continue;
        squares(row[blk * 64 + lane], u);
        const Pair p = pair_scan(readlane64(starts, blk), u, lane, 0);
        if (lane == 63) {
            pairs[2 * blk] = p.c[0];
            pairs[2 * blk + 1] = p.c[1];
        }
    }
    __syncthreads();
    if (wave == 0) {
        const double none = __builtin_nan("");
        Pair p = {{double64(binade(starts)), double64(binade(starts) + 1)}, {none, none}};   // lane b: block b's
        if (scan && lane >= first && lane < nblk) p.c[0] = pairs[2 * lane], p.c[1] = pairs[2 * lane + 1];
        for (int blk = first; blk < nblk; blk++) {
            const double end = p.after(sum);           // meant in lane blk
            if (__ballot(binade(sum) == binade(starts) && p.within(end)) >> blk & 1) {
                sum = readlane64(end, blk);
            } else {
                squares(row[blk * 64 + lane], u);      // zeros past k
                sum = block_exact(from ? sure : sum, u, lane, from);
            }
            from = 0;
        }
        if (lane == 0) pairs[2 * nblk] = sum;
    }
    __syncthreads();
    return pairs[2 * nblk];
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
// round went term by term), Gaussian rows: 1 x 1024 5.80 -> 2.40 us a launch,
// 512 x 1024 12.9 -> 4.0 us.
template <int NB>
__global__ __launch_bounds__(1024) void k_add_rmsnorm(const float *h, const float *delta,
                                                      const float *__restrict__ w, float eps, int k, float *h_out,
                                                      float *x_out, uint8_t *__restrict__ xq) {
    __shared__ double total[QK_NORM_MAX_K / QK_K], ends[QK_NORM_MAX_K / QK_K];   // an end of -1: a guess is still wrong
    __shared__ double pairs[2 * QK_NORM_MAX_K / QK_K + 1];
    __shared__ double sure[QK_NORM_MAX_K / QK_K];      // of such a block: the last end that is right,
    __shared__ int upto[QK_NORM_MAX_K / QK_K];         // and its lane
    extern __shared__ float4 row4[];                   // the row, where a guess was wrong
    const int nblk = (k + QK_K - 1) / QK_K, W = NB == 1 ? nblk : NORM_WAVES;   // as launched
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
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
        squares(r[b], t[b]);
        const double own = __dadd_rn(__dadd_rn(t[b][0], t[b][1]), __dadd_rn(t[b][2], t[b][3]));
        const double incl = wave_scan64(own, false);
        q[b] = dpp64<0x138>(incl);                    // wave_shr:1
        if (lane == 63 && wave + W * b < nblk) total[wave + W * b] = incl;
    }
    __syncthreads();
    // lane b of every wave: the guessed start of block b
    double starts = dpp64<0x138>(wave_scan64(lane < nblk ? total[lane] : 0.0, nblk <= 16));
#pragma unroll
    for (int b = 0; b < NB; b++) {                     // q: the guessed starts of the lane's segments
        const double from = readlane64(starts, min(wave + W * b, nblk - 1));
        q[b] = lane == 0 ? from : __dadd_rn(from, q[b]);
    }
    double ssq;                                        // the chain up to block `first`
    int first = nblk;
    for (int round = 0;; round++) {                    // uniform: every wave sees the same ends
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int blk = wave + W * b;
            if (blk < nblk) {
                int open;
                const double e = check_block(q[b], t[b], lane, round == 0 ? NORM_MOVES : NORM_MOVES_ON, open);
                if (__builtin_expect(open == 64, 1)) {
                    if (lane == 63) ends[blk] = e;
                } else if (lane == open) {
                    ends[blk] = -1.0;
                    sure[blk] = e;
                    upto[blk] = open;
                }
            }
        }
        __syncthreads();
        const double e = lane < nblk ? ends[lane] : 0.0, next = dpp64<0x130>(starts);   // wave_shl:1
        const uint64_t off = __ballot((e == -1.0) | ((lane < nblk - 1) & !same_bits(e, next)));
        if (__builtin_expect(off == 0, 1)) {
            ssq = readlane64(e, nblk - 1);
            break;
        }
        // block f starts right, and ends right unless a guess in it is still wrong
        const int f = __builtin_ctzll(off);
        const double end = readlane64(e, f);
        if (end == -1.0 || round == NORM_ROUNDS) {
            first = end == -1.0 ? f : f + 1;
            ssq = end == -1.0 ? readlane64(starts, f) : end;
            break;
        }
        // the blocks after f start where f ends or move by as much, and their
        // segments with them (what the checks settled in them stays)
        const double later = move_starts(starts, end, f, lane);
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int blk = min(wave + W * b, nblk - 1);
            const double was = readlane64(starts, blk), now = readlane64(later, blk);
            if (!same_bits(was, now)) q[b] = lane == 0 ? now : __dadd_rn(q[b], __dsub_rn(now, was));
        }
        starts = later;
        __syncthreads();                               // the ends are rewritten
    }
    if (__builtin_expect(first < nblk, 0)) {
#pragma unroll
        for (int b = 0; b < NB; b++)
            if (wave + W * b < nblk) row4[(wave + W * b) * 64 + lane] = r[b];
        const bool open = ends[first] == -1.0;
        ssq = exact_from(row4, pairs, starts, ssq, first, nblk, W, open ? upto[first] + 1 : 0, sure[first]);
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
    const int nblk = (int)((k + QK_K - 1) / QK_K), waves = nblk < NORM_WAVES ? nblk : NORM_WAVES;
    auto kernel = nblk <= NORM_WAVES ? k_add_rmsnorm<1> : nblk <= 2 * NORM_WAVES ? k_add_rmsnorm<2> : k_add_rmsnorm<4>;
    const int64_t rows = (int64_t)1 << 21;
    for (int64_t t = 0; t < m; t += rows) {
        const unsigned grid = (unsigned)(m - t < rows ? m - t : rows);
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * waves), (size_t)nblk * QK_K * sizeof(float), s, h + t * k, delta ? delta + t * k : nullptr, w,
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
