// qk_deltanet.hip -- the chunked Gated DeltaNet prefill (gfx950).
//
// chunked_ssm_step_f32 (slm/chunked.c:287-521) for every head of a layer
// and every chunk of up to 64 tokens, the state of each head carried from
// chunk to chunk as slm_forward_ssm_batch does (slm/qwen.c:772-807).
//
// The reference runs on the host with plain fp32 loops; on x86 each dot
// and each axpy is a sequential chain of separately rounded products and
// sums (no FMA in its build), and its result depends on that order. Here
// every output element is one lane's chain in exactly the reference's
// order; the parallelism is across outputs, heads and chunks (this file is
// built with -ffp-contract=off; the only fused multiply-adds are inside
// qk_expf). Two launches per group of chunks:
//
//   k_dn_chunk  what does not depend on the carried state, every (chunk,
//               head) at once: the gates, KK^T and KQ^T with the decay, the
//               triangular solve, attn @ V*beta and attn @ K*beta*exp(gcs)
//   k_dn_carry  chunk after chunk: the state against Q*exp(gcs) and the
//               decayed keys, v_new, the output rows, the state carried on
//
// Where the reference skips a zero coefficient, the chain adds the zero
// product instead: a sum that starts at +0 is never -0, so adding +-0 leaves
// it as it is. That fails only for an infinite or NaN factor, so the kernels
// watch the factors (V*beta, K*beta*exp(gcs), the state) and take a copy of
// the loop with the skip when one is not finite.
#include "qk_dev.h"
#include "qk_expf.h"
#include "qk_kernels.h"

namespace qk {

constexpr int DN_C = 64;                               // chunk size (CHUNK_SIZE)
constexpr int DN_D = 128;                              // largest head dim handled; row stride of the scratch

// Scratch of one group of chunks (floats), one slot per (chunk, head). Rows
// past the chunk and columns past the head dims hold zeros.
struct DnScratch {
    float *qg;      // [64][128] Q * exp(gcs)
    float *kcd;     // [64][128] attn @ K*beta*exp(gcs)
    float *veff;    // [64][128] attn @ V*beta
    float *kgt;     // [128][64] (K * exp(glast - gcs))^T
    float *akq;     // [64][64] lower (K_j . Q_i) * decay
    float *gl;      // exp(glast)
};

struct DnArgs {
    const float *q, *k, *v, *g, *beta;   // [n_tok][H][...]
    float *state;                        // [H][kd][vd]
    float *out;                          // [n_tok][H][vd]
    int64_t n_tok;                       // tokens of the call
    int64_t g0;                          // first chunk of the group in flight
    int32_t H, kd, vd;
    int32_t vec;                         // kd and vd are multiples of 4
};

// A scratch slot is one (chunk of the group, head): slot = c * H + h.
struct DnChunk {
    int slot, h, n;                      // slot, head, tokens of the chunk (1..64)
    int64_t c0;                          // first token of the chunk
};

__device__ __forceinline__ DnChunk dn_chunk(const DnArgs &a, int slot) {
    DnChunk ck;
    ck.slot = slot;
    ck.h = slot % a.H;
    ck.c0 = (a.g0 + slot / a.H) * DN_C;
    const int64_t rest = a.n_tok - ck.c0;
    ck.n = rest < DN_C ? (int)rest : DN_C;
    return ck;
}

// Elements 4c .. 4c + 3 of row t of a chunk, dim a multiple of 4 (zeros past
// the row or the chunk). Rows start on 4-byte boundaries.
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ float4 dn_load4(const float *base, const DnArgs &a, const DnChunk &ck, int t, int c,
                                           int dim) {
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (t < ck.n && 4 * c < dim) {
        const f4u x = *reinterpret_cast<const f4u *>(base + ((ck.c0 + t) * a.H + ck.h) * (int64_t)dim + 4 * c);
        v = make_float4(x[0], x[1], x[2], x[3]);
    }
    return v;
}

__device__ __forceinline__ float4 scale4(float4 v, float s) {
    return make_float4(__fmul_rn(v.x, s), __fmul_rn(v.y, s), __fmul_rn(v.z, s), __fmul_rn(v.w, s));
}

// The same for columns 4c .. of which `left` lie within the head dim: the
// padding stays 0 where s is infinite or NaN.
__device__ __forceinline__ float4 scale4(float4 v, float s, int left) {
    const float4 p = scale4(v, s);
    return make_float4(left > 0 ? p.x : 0.0f, left > 1 ? p.y : 0.0f, left > 2 ? p.z : 0.0f, left > 3 ? p.w : 0.0f);
}

__device__ __forceinline__ bool finite(float x) { return fabsf(x) < __builtin_inff(); }
__device__ __forceinline__ bool finite4(float4 v) { return finite(v.x) && finite(v.y) && finite(v.z) && finite(v.w); }

__device__ __forceinline__ float dn_term(float acc, float c, float x) { return __fadd_rn(acc, __fmul_rn(c, x)); }

// As the reference writes it where it skips a zero coefficient c.
__device__ __forceinline__ float dn_term_skip(float acc, float c, float x) { return c != 0.0f ? dn_term(acc, c, x) : acc; }

__device__ __forceinline__ float lane_value(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// ---- phase 1: everything of a chunk that the state does not enter ---------------
// Grid (slots, 3 parts) of 512 threads; LDS leaves room for two workgroups
// per CU:
//   part 0  KK^T * decay, the solve, attn @ V*beta
//   part 1  KK^T * decay, the solve, attn @ K*beta*exp(gcs)
//   part 2  KQ^T * decay, Q*exp(gcs), (K*exp(glast - gcs))^T, exp(glast)
// Parts 0 and 1 repeat the dots and the solve: it costs less than a second
// launch with its loads. A workgroup is a chain of phases, each bound by
// issue or latency (16 heads x 512 tokens, microseconds of one workgroup):
// loads and the gates' sum 3.4, the dots 3.6 (4 rows from LDS for 4 chains),
// the solve 4.3 (64 dependent steps), the apply 3.2. Against one launch per
// phase, with the matrices through memory in between: 70 -> 22 us at 512
// tokens, 38 -> 19 us at 100.
constexpr int DN_WG = 512;

// float4 column c of row t in the dots' operands: rows 2b of sixteen
// consecutive b fall on sixteen different 16-byte columns.
__device__ __forceinline__ int dn_swz(int t, int c) { return t * (DN_D / 4) + (c ^ ((t >> 1) & 15)); }

// Element (i, j) of the triangular matrices: rows r, r + 8, ... of one column
// lie 512 floats apart (two to an LDS read), rows 0 .. 7 on different banks.
__device__ __forceinline__ int dn_tri(int i, int j) { return i * DN_C + (j ^ ((i & 7) << 3)); }

// X = (I + L)^-1 - I below the diagonal (slm/chunked.c:196-213): X[i][j] =
// (-L[i][j] - sum_{t<i} L[i][t] X[t][j]) / 1. Lane (j, rg) holds the sums of
// rows rg, rg + 8, ... of column j; eight lanes side by side share a column.
// Right-looking: as soon as X[k][j] is known every later row adds its term
// k, so each row's sum runs t = 0, 1, 2, ... in the reference's order.
// X[k][j] goes from its lane to the column's eight by DPP; column k + 2 of L
// is read while step k runs. Dividing by the unit diagonal returns its
// operand unchanged (a quiet NaN included), so the division is left out.
// xs[m]: row rg + 8m (rows of a finished slot keep adding what the array holds
// from the diagonal on, which nothing reads).
__device__ __forceinline__ void dn_solve(const float *L, int j, int rg, float (&xs)[8]) {
    float acc[8], nl[8], cf[3][8];
    auto column = [&](int k) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < 8; m++)
            if (m >= k / 8) cf[k % 3][m] = L[dn_tri(rg, k) + 8 * DN_C * m];
    };
#pragma unroll
    for (int m = 0; m < 8; m++) {
        const int i = rg + 8 * m;
        // -L of a zero from the diagonal on, where the array holds what was there before
        nl[m] = j < i ? -L[dn_tri(rg, j) + 8 * DN_C * m] : -0.0f;
        acc[m] = xs[m] = 0.0f;
    }
    column(0);
    column(1);
#pragma unroll
    for (int k = 0; k < DN_C; k++) {
        if (k + 2 < DN_C) column(k + 2);
        asm volatile("" ::: "memory");                 // the reads stay two steps ahead
        const int mk = k / 8, ok = k % 8;              // row k is slot mk of lane ok
        const float x0 = __fsub_rn(nl[mk], acc[mk]);   // meant in lane ok
        xs[mk] = rg == ok ? x0 : xs[mk];
        int b = 0;                                     // its quad's copy, then the other quad's
        switch (ok & 3) {
            case 0: b = __builtin_amdgcn_mov_dpp(__float_as_int(x0), 0x00, 0xF, 0xF, true); break;
            case 1: b = __builtin_amdgcn_mov_dpp(__float_as_int(x0), 0x55, 0xF, 0xF, true); break;
            case 2: b = __builtin_amdgcn_mov_dpp(__float_as_int(x0), 0xAA, 0xF, 0xF, true); break;
            default: b = __builtin_amdgcn_mov_dpp(__float_as_int(x0), 0xFF, 0xF, 0xF, true); break;
        }
        const int o = dpp_hmirror(b);
        const float x = __int_as_float((rg >> 2) == (ok >> 2) ? b : o);
        float p[8];
#pragma unroll
        for (int m = mk; m < 8; m++) p[m] = __fmul_rn(cf[k % 3][m], x);
#pragma unroll
        for (int m = mk; m < 8; m++) acc[m] = __fadd_rn(acc[m], p[m]);
    }
}

// Rows wave + 8m of attn @ M (M [64][128] in LDS), two columns per lane. A
// row of attn sits in one register (lane j: column j) and its elements
// become wave-uniform factors by readlane. Row wave + 8m ends at column
// wave + 8m; the columns from there to 8m + 7 are zeros. n8: 8-row slots
// that hold rows of the chunk.
__device__ __forceinline__ void dn_apply(const float (&at)[8], const float *M, int lane, int n8, float (&o)[8][2]) {
    float x[4][2];
#pragma unroll
    for (int q = 0; q < 4; q++) x[q][0] = M[q * DN_D + lane], x[q][1] = M[q * DN_D + 64 + lane];
#pragma unroll
    for (int mj = 0; mj < 8; mj++) {
        if (mj >= n8) break;                           // uniform
#pragma unroll
        for (int h = 0; h < 2; h++) {                  // four columns of attn, the next four's rows in flight
            float nx[4][2];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int j = (8 * mj + 4 * h + 4 + q) & (DN_C - 1);
                nx[q][0] = M[j * DN_D + lane];
                nx[q][1] = M[j * DN_D + 64 + lane];
            }
            asm volatile("" ::: "memory");
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int j = 8 * mj + 4 * h + q;
                float c[8], p0[8], p1[8];
#pragma unroll
                for (int m = mj; m < 8; m++) c[m] = lane_value(at[m], j);
#pragma unroll
                for (int m = mj; m < 8; m++) {
                    p0[m] = __fmul_rn(c[m], x[q][0]);
                    p1[m] = __fmul_rn(c[m], x[q][1]);
                }
#pragma unroll
                for (int m = mj; m < 8; m++) {
                    o[m][0] = __fadd_rn(o[m][0], p0[m]);
                    o[m][1] = __fadd_rn(o[m][1], p1[m]);
                }
            }
#pragma unroll
            for (int q = 0; q < 4; q++) x[q][0] = nx[q][0], x[q][1] = nx[q][1];
        }
    }
}

// The same with the reference's skips, for a factor that is not finite.
__device__ __forceinline__ void dn_apply_skip(const float (&at)[8], const float *M, int lane, float (&o)[8][2]) {
#pragma unroll 1
    for (int j = 0; j < DN_C; j++) {
        const float x0 = M[j * DN_D + lane], x1 = M[j * DN_D + 64 + lane];
#pragma unroll
        for (int m = 0; m < 8; m++) {
            const float c = lane_value(at[m], j);
            o[m][0] = dn_term_skip(o[m][0], c, x0);
            o[m][1] = dn_term_skip(o[m][1], c, x1);
        }
    }
}

__global__ __launch_bounds__(DN_WG) void k_dn_chunk(DnArgs a, DnScratch s) {
    const DnChunk ck = dn_chunk(a, blockIdx.x);
    const int part = blockIdx.y, n = ck.n, kd = a.kd;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    __shared__ float4 A[DN_C * DN_D / 4];              // K rows; then V*beta or K*beta*exp(gcs)
    __shared__ float4 B[DN_C * DN_D / 4];              // K*beta or Q rows; then KK^T or KQ^T; then attn
    __shared__ float gcs[DN_C], glast;                 // the gates' running sum; its last
    __shared__ uint64_t etab[32];
    __shared__ int bad;                                // a factor of the apply is not finite
    // thread: float4 column c of rows t0, t0 + 16, ...
    const int c = tid & 31, t0 = tid >> 5;
    float4 kr[4], r2[4];                               // K; V (part 0) or Q (part 2)
    const float *other = part == 0 ? a.v : a.q;
    const int odim = part == 0 ? a.vd : kd;
    if (a.vec) {                                       // uniform
#pragma unroll
        for (int u = 0; u < 4; u++) {
            kr[u] = dn_load4(a.k, a, ck, t0 + 16 * u, c, kd);
            r2[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (part != 1) r2[u] = dn_load4(other, a, ck, t0 + 16 * u, c, odim);
        }
    } else {                                           // element by element through LDS
        float *Af = reinterpret_cast<float *>(A), *Bf = reinterpret_cast<float *>(B);
#pragma unroll 1
        for (int p = tid; p < DN_C * DN_D; p += DN_WG) {
            const int t = p / DN_D, d = p % DN_D;
            const int64_t row = (ck.c0 + t) * a.H + ck.h;
            Af[p] = t < n && d < kd ? a.k[row * kd + d] : 0.0f;
            Bf[p] = part != 1 && t < n && d < odim ? other[row * odim + d] : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 4; u++) {
            kr[u] = A[(t0 + 16 * u) * (DN_D / 4) + c];
            r2[u] = B[(t0 + 16 * u) * (DN_D / 4) + c];
        }
        __syncthreads();                               // the same rows are written below, in another column order
    }
    float bt[4];                                       // beta of the thread's rows
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int t = t0 + 16 * u;
        bt[u] = t < n ? a.beta[(ck.c0 + t) * a.H + ck.h] : 0.0f;
    }
    if (wave == 0) {                                   // the gates' sums, lane t for token t
        const float g = lane < n ? a.g[(ck.c0 + lane) * a.H + ck.h] : 0.0f;
        if (lane < 32) etab[lane] = qk_exp2_32[lane];
        if (lane == 0) bad = 0;
        float run = 0.0f, mine = 0.0f;
        for (int t = 0; t < n; t += 8)                 // g past the chunk adds +0
#pragma unroll
            for (int q = 0; q < 8; q++) {
                run = __fadd_rn(run, lane_value(g, t + q));
                mine = lane == t + q ? run : mine;
            }
        gcs[lane] = lane < n ? mine : 0.0f;            // exp 1 past the chunk: its rows stay zeros
        if (lane == 0) glast = run;
    }
    const int64_t ro = (int64_t)ck.slot * DN_C * DN_D; // a [64][128] (or [128][64]) array of the slot
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int t = t0 + 16 * u;
        A[dn_swz(t, c)] = kr[u];
        if (part == 2) {
            B[dn_swz(t, c)] = r2[u];
        } else {
            kr[u] = scale4(kr[u], bt[u], kd - 4 * c);  // K * beta
            B[dn_swz(t, c)] = kr[u];
        }
    }
    __syncthreads();
    if (part == 2) {
        // exp(gcs) * Q; (K * exp(glast - gcs))^T, 4 tokens a store
        if (tid == 0) s.gl[ck.slot] = qk_expf_tab(glast, etab);
#pragma unroll
        for (int u = 0; u < 4; u++) {                  // rows past the chunk are zeros
            const int t = t0 + 16 * u;
            const float4 qg = scale4(r2[u], qk_expf_tab(gcs[t], etab), kd - 4 * c);
            *reinterpret_cast<float4 *>(s.qg + ro + t * DN_D + 4 * c) = qg;
        }
        const float *Af = reinterpret_cast<const float *>(A);
        const int tq = (tid & 15) * 4;
        float gf[4];
#pragma unroll
        for (int i = 0; i < 4; i++) gf[i] = qk_expf_tab(__fsub_rn(glast, gcs[tq + i]), etab);
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int d = (tid + DN_WG * u) >> 4;
            float e[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int t = tq + i;
                e[i] = t < n && d < kd ? __fmul_rn(Af[4 * dn_swz(t, d >> 2) + (d & 3)], gf[i]) : 0.0f;
            }
            *reinterpret_cast<float4 *>(s.kgt + ro + d * DN_C + tq) = make_float4(e[0], e[1], e[2], e[3]);
        }
    }
    // the dots, two rows against two per thread: the 496 tiles of row pairs
    // below the diagonal, then 16 that hold the pairs (2b + 1, 2b)
    float *D = reinterpret_cast<float *>(B);           // KK^T or KQ^T, once every thread is done with B
    const int k4 = (kd + 3) / 4;
    int i0, i1, j0, j1;
    if (tid < 496) {                                   // p (p - 1) / 2 + q, q < p
        int p = (int)((1.0f + __builtin_sqrtf(1.0f + 8.0f * (float)tid)) * 0.5f);
        if (p * (p - 1) / 2 > tid) p--;
        if (p * (p + 1) / 2 <= tid) p++;
        i0 = 2 * p;
        j0 = 2 * (tid - p * (p - 1) / 2);
        i1 = i0 + 1;
        j1 = j0 + 1;
    } else {
        j0 = 4 * (tid - 496);
        i0 = j0 + 1;
        j1 = j0 + 2;
        i1 = j0 + 3;
    }
    float r[4] = {0.0f, 0.0f, 0.0f, 0.0f};             // (i0, j0), (i0, j1), (i1, j0), (i1, j1)
    if (min(i0, i1) < n) {
#pragma unroll 2
        for (int d = 0; d < k4; d++) {
            const float4 x0 = B[dn_swz(i0, d)], x1 = B[dn_swz(i1, d)];
            const float4 y0 = A[dn_swz(j0, d)], y1 = A[dn_swz(j1, d)];
            const float xa[4] = {x0.x, x0.y, x0.z, x0.w}, xb[4] = {x1.x, x1.y, x1.z, x1.w};
            const float ya[4] = {y0.x, y0.y, y0.z, y0.w}, yb[4] = {y1.x, y1.y, y1.z, y1.w};
            float p[4][4];
#pragma unroll
            for (int i = 0; i < 4; i++) {              // zeros past kd add +-0
                p[0][i] = __fmul_rn(ya[i], xa[i]);
                p[1][i] = __fmul_rn(yb[i], xa[i]);
                p[2][i] = __fmul_rn(ya[i], xb[i]);
                p[3][i] = __fmul_rn(yb[i], xb[i]);
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) r[e] = __fadd_rn(r[e], p[e][i]);
        }
    }
    float diag = 0.0f;                                 // part 2, wave 0: (lane, lane)
    if (part == 2 && wave == 0) {
#pragma unroll 2
        for (int d = 0; d < k4; d++) {
            const float4 x = B[dn_swz(lane, d)], y = A[dn_swz(lane, d)];
            diag = dn_term(dn_term(dn_term(dn_term(diag, y.x, x.x), y.y, x.y), y.z, x.z), y.w, x.w);
        }
    }
    const float gi[2] = {gcs[i0], gcs[i1]}, gj[2] = {gcs[j0], gcs[j1]};
#pragma unroll
    for (int e = 0; e < 4; e++)                        // the decay exp(gcs_i - gcs_j)
        r[e] = __fmul_rn(r[e], qk_expf_tab(__fsub_rn(gi[e >> 1], gj[e & 1]), etab));
    __syncthreads();                                   // every thread is done with A and B
    if (i0 < n) {
        D[dn_tri(i0, j0)] = r[0];
        if (tid < 496) D[dn_tri(i0, j1)] = r[1];       // above the diagonal in the last tiles
    }
    if (i1 < n) {
        if (tid < 496) D[dn_tri(i1, j0)] = r[2];       // another tile's in the last tiles
        D[dn_tri(i1, j1)] = r[3];
    }
    if (part == 2) {
        if (wave == 0) D[dn_tri(lane, lane)] = diag;   // the decay there is 1
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int e0 = (tid + DN_WG * u) * 4, i = e0 / DN_C, j = e0 % DN_C;
            float e[4];
#pragma unroll
            for (int v = 0; v < 4; v++) e[v] = j + v <= i && i < n ? D[dn_tri(i, j + v)] : 0.0f;
            *reinterpret_cast<float4 *>(s.akq + (int64_t)ck.slot * DN_C * DN_C + e0) =
                make_float4(e[0], e[1], e[2], e[3]);
        }
        return;
    }
    // L's rows past the chunk: zeros, not what the array held before
    for (int p = tid; p < (DN_C - n) * DN_C; p += DN_WG) D[dn_tri(n + p / DN_C, p % DN_C)] = 0.0f;
    bool fin = true;
#pragma unroll
    for (int u = 0; u < 4; u++) {
        if (part == 0) r2[u] = scale4(r2[u], bt[u], odim - 4 * c);   // V * beta
        else r2[u] = scale4(kr[u], qk_expf_tab(gcs[t0 + 16 * u], etab), kd - 4 * c);   // K * beta * exp(gcs)
        A[(t0 + 16 * u) * (DN_D / 4) + c] = r2[u];     // plain rows: the apply reads along a row
        fin = fin && finite4(r2[u]);
    }
    if (!fin) bad = 1;
    __syncthreads();
    float xs[8];
    const int j = tid >> 3, rg = tid & 7;
    dn_solve(D, j, rg, xs);
    __syncthreads();                                   // the solve is done with L
#pragma unroll
    for (int m = 0; m < 8; m++) {
        const int i = rg + 8 * m;
        D[dn_tri(i, j)] = j < i ? xs[m] : (j == i ? 1.0f : 0.0f);
    }
    __syncthreads();
    float at[8], o[8][2];
#pragma unroll
    for (int m = 0; m < 8; m++) {
        at[m] = D[dn_tri(wave + 8 * m, lane)];
        o[m][0] = o[m][1] = 0.0f;
    }
    const float *M = reinterpret_cast<const float *>(A);
    if (bad) dn_apply_skip(at, M, lane, o);
    else dn_apply(at, M, lane, (n + 7) / 8, o);
    float *dst = (part == 0 ? s.veff : s.kcd) + ro;
#pragma unroll
    for (int m = 0; m < 8; m++) {                      // an infinite attn makes the padding's sums NaN
        const int w = wave + 8 * m < n ? odim : 0;     // and the rows' past the chunk
        dst[(wave + 8 * m) * DN_D + lane] = lane < w ? o[m][0] : 0.0f;
        dst[(wave + 8 * m) * DN_D + 64 + lane] = 64 + lane < w ? o[m][1] : 0.0f;
    }
}

// ---- phase 2: the carried state ----------------------------------------------------
// A workgroup owns DN_E columns of one head's state, keeps them in LDS and
// walks the group's chunks in order; v_new[., e], the output column e and
// the new state column e read only the state column e and rows that every
// column shares, so no workgroup waits for another. Lane (t, e) runs the two
// chains over the state (query and decayed key of token t), then, over
// v_new, the output chain of (t, e) and the state chains of (t, e) and
// (t + 64, e). The four lanes of a quad have one t: each loads a quarter of
// that row's coefficients straight from the scratch (16-byte loads, issued
// while the other half of a chunk computes) and gets the rest by a quad
// broadcast inside the multiply, so LDS carries only the state and v_new.
// That multiply takes 4 cycles a wave against 2, but reading every
// coefficient from LDS would bind earlier (3 reads per 2 terms). Measured:
// 2.9 ns a SIMD for a product and its sum in a loop of these alone, 3.9 ns
// here with the barriers and the reads; the products on the matrix cores (an
// fp32 MFMA of one term rounds a product as the multiply does) took 3.2 ns.
// With the coefficients staged in LDS, one output per lane and the skips in
// the loop, 16 heads x 512 tokens took 91 us; 43 us here.
constexpr int DN_E = 8;                                // state columns per workgroup
constexpr int DN_SS = DN_D + 4;                        // LDS row of a state column
constexpr int DN_VS = DN_C + 4;                        // LDS row of a v_new column

// v of lane Q of the quad.
template <int Q>
__device__ __forceinline__ float quad(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), Q * 0x55, 0xF, 0xF, true));
}

// The products of four terms of N chains (coefficients from quad lane Q,
// factors x), each beside the sum that takes the product of four terms
// before (p): a chain's next sum comes 2N instructions after its last, and
// every product has a register of its own, so neither waits. The empty asm
// keeps that order.
template <int Q, int N>
__device__ __forceinline__ void quad_terms(float (&acc)[N], float (&p)[4][N], const float4 (&cf)[N], float4 x,
                                           bool first) {
    const float xe[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
        for (int i = 0; i < N; i++) {
            const float ce = e == 0 ? cf[i].x : e == 1 ? cf[i].y : e == 2 ? cf[i].z : cf[i].w;
            float m = __fmul_rn(quad<Q>(ce), xe[e]);
            if (!first) acc[i] = __fadd_rn(acc[i], p[e][i]);
            asm volatile("" : "+v"(m), "+v"(acc[i]));
            p[e][i] = m;
        }
}

// The chains over blocks of 16 elements of a column at col (LDS), a block's
// elements read while the one before it computes.
template <int N, int NB>
__device__ __forceinline__ void dn_chains(float (&acc)[N], const float4 (&cf)[NB][N], const float *col, int nb) {
    const float4 *x = reinterpret_cast<const float4 *>(col);
    float4 cur[4], nxt[4];
    float p[4][N];
#pragma unroll
    for (int i = 0; i < 4; i++) cur[i] = x[i];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        if (b + 1 < NB)
#pragma unroll
            for (int i = 0; i < 4; i++) nxt[i] = x[4 * (b + 1) + i];
        asm volatile("" ::: "memory");                 // the reads stay above this block's terms
        quad_terms<0>(acc, p, cf[b], cur[0], b == 0);
        quad_terms<1>(acc, p, cf[b], cur[1], false);
        quad_terms<2>(acc, p, cf[b], cur[2], false);
        quad_terms<3>(acc, p, cf[b], cur[3], false);
        if (b + 1 >= nb) break;                        // uniform
#pragma unroll
        for (int i = 0; i < 4; i++) cur[i] = nxt[i];
    }
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
        for (int i = 0; i < N; i++) acc[i] = __fadd_rn(acc[i], p[e][i]);
}

__global__ __launch_bounds__(512) void k_dn_carry(DnArgs a, DnScratch s, int gc, int ncol) {
    __shared__ __align__(16) float S[DN_E * DN_SS], V[DN_E * DN_VS];
    __shared__ int bad;                                // the state holds or held an inf or NaN
    // workgroups of one head on one XCD where the heads allow it: they
    // read the same rows
    int h, cg;
    if ((a.H & 7) == 0) {
        const int x = blockIdx.x >> 3;
        h = (blockIdx.x & 7) + 8 * (x / ncol);
        cg = x % ncol;
    } else {
        h = blockIdx.x / ncol;
        cg = blockIdx.x % ncol;
    }
    const int e0 = cg * DN_E, kd = a.kd, vd = a.vd;
    const int tid = threadIdx.x, el = tid % DN_E, e = e0 + el, t = tid / DN_E, ql = tid & 3;
    const bool col = e < vd;
    float *st = a.state + (int64_t)h * kd * vd;
    if (tid == 0) bad = 0;
    __syncthreads();
    for (int p = tid; p < DN_D * DN_E; p += 512) {
        const int d = p / DN_E, cc = p % DN_E;
        const float x = d < kd && e0 + cc < vd ? st[(int64_t)d * vd + e0 + cc] : 0.0f;
        S[cc * DN_SS + d] = x;
        if (!finite(x)) bad = 1;
    }
    constexpr int B5 = DN_D / 16, B6 = DN_C / 16;
    float4 c5[B5][2], c6[B6][3];
    float ve, gl;
    auto load5 = [&](int c) __attribute__((always_inline)) {
        const int64_t ro = (int64_t)(c * a.H + h) * DN_C * DN_D + t * DN_D;
#pragma unroll
        for (int b = 0; b < B5; b++) {
            c5[b][0] = *reinterpret_cast<const float4 *>(s.qg + ro + 16 * b + 4 * ql);
            c5[b][1] = *reinterpret_cast<const float4 *>(s.kcd + ro + 16 * b + 4 * ql);
        }
        ve = s.veff[ro + (col ? e : 0)];
    };
    auto load6 = [&](int c) __attribute__((always_inline)) {
        const int64_t slot = c * a.H + h;
        const float *aq = s.akq + slot * DN_C * DN_C + t * DN_C, *kg = s.kgt + slot * DN_C * DN_D + t * DN_C;
#pragma unroll
        for (int b = 0; b < B6; b++) {
            c6[b][0] = *reinterpret_cast<const float4 *>(aq + 16 * b + 4 * ql);
            c6[b][1] = *reinterpret_cast<const float4 *>(kg + 16 * b + 4 * ql);
            c6[b][2] = *reinterpret_cast<const float4 *>(kg + 64 * DN_C + 16 * b + 4 * ql);
        }
        gl = s.gl[slot];
    };
    load5(0);
    load6(0);
    __syncthreads();
    const int nd = (kd + 15) / 16;
    for (int c = 0; c < gc; c++) {
        const DnChunk ck = dn_chunk(a, c * a.H + h);
        const int n = ck.n;
        // the chains against the state: query and decayed key of token t
        float a5[2] = {0.0f, 0.0f};
        if (bad) {                                     // uniform; with the reference's skips
            const float *qg = s.qg + (int64_t)ck.slot * DN_C * DN_D + t * DN_D;
            const float *kc = s.kcd + (int64_t)ck.slot * DN_C * DN_D + t * DN_D;
#pragma unroll 1
            for (int d = 0; d < kd; d++) {
                const float x = S[el * DN_SS + d];
                a5[0] = dn_term_skip(a5[0], qg[d], x);
                a5[1] = dn_term_skip(a5[1], kc[d], x);
            }
        } else {
            dn_chains(a5, c5, S + el * DN_SS, nd);
        }
        V[el * DN_VS + t] = t < n && col ? __fsub_rn(ve, a5[1]) : 0.0f;
        __syncthreads();
        if (c + 1 < gc) load5(c + 1);
        // over v_new: the intra-chunk attention row t, the state rows t, t + 64
        float a6[3] = {0.0f, 0.0f, 0.0f};
        dn_chains(a6, c6, V + el * DN_VS, (n + 15) / 16);
        if (t < n && col) a.out[((ck.c0 + t) * a.H + h) * (int64_t)vd + e] = __fadd_rn(a5[0], a6[0]);
        float *s0 = &S[el * DN_SS + t];
        const float n0 = t < kd ? __fadd_rn(__fmul_rn(s0[0], gl), a6[1]) : 0.0f;
        const float n1 = t + 64 < kd ? __fadd_rn(__fmul_rn(s0[64], gl), a6[2]) : 0.0f;
        s0[0] = n0;
        s0[64] = n1;
        if (!finite(n0) || !finite(n1)) bad = 1;
        if (c + 1 < gc) load6(c + 1);
        __syncthreads();
    }
    for (int p = tid; p < DN_D * DN_E; p += 512) {
        const int d = p / DN_E, cc = p % DN_E;
        if (d < kd && e0 + cc < vd) st[(int64_t)d * vd + e0 + cc] = S[cc * DN_SS + d];
    }
}

// ---- launcher -----------------------------------------------------------------
// The chunks go in groups of at most DN_SLOTS (chunk, head) slots (147 KB of
// scratch each) and at least one chunk.
constexpr int DN_SLOTS = 256;

static int dn_group(int32_t H, int64_t n_tok) {
    const int64_t chunks = (n_tok + DN_C - 1) / DN_C;
    const int64_t g = DN_SLOTS / H > 1 ? DN_SLOTS / H : 1;
    return (int)(g < chunks ? g : chunks);
}

size_t deltanet_scratch_bytes(int32_t H, int32_t kd, int32_t vd, int64_t n_tok) {
    (void)kd, (void)vd;                                // rows are padded to DN_D
    const size_t slots = (size_t)dn_group(H, n_tok) * (size_t)H;
    return (slots * (4 * DN_C * DN_D + DN_C * DN_C + 1) + 6 * 64) * sizeof(float) + 256;
}

hipError_t launch_deltanet(const float *q, const float *k, const float *v, const float *g, const float *beta,
                           int64_t n_tok, int32_t H, int32_t kd, int32_t vd, float *state, float *out,
                           void *scratch, hipStream_t st) {
    if (kd > DN_D || vd > DN_D || n_tok < 1 || H < 1) return hipErrorInvalidValue;
    const int G = dn_group(H, n_tok);
    const size_t slots = (size_t)G * (size_t)H;
    float *p = reinterpret_cast<float *>((reinterpret_cast<uintptr_t>(scratch) + 255) & ~(uintptr_t)255);
    auto take = [&](size_t n_floats) {
        float *r = p;
        p += (n_floats + 63) & ~(size_t)63;            // 256-byte aligned arrays
        return r;
    };
    DnScratch s;
    s.qg = take(slots * DN_C * DN_D);
    s.kcd = take(slots * DN_C * DN_D);
    s.veff = take(slots * DN_C * DN_D);
    s.kgt = take(slots * DN_C * DN_D);
    s.akq = take(slots * DN_C * DN_C);
    s.gl = take(slots);
    const int vec = kd % 4 == 0 && vd % 4 == 0;
    const int64_t chunks = (n_tok + DN_C - 1) / DN_C;
    const int ncol = (vd + DN_E - 1) / DN_E;
    for (int64_t g0 = 0; g0 < chunks; g0 += G) {
        const int gc = (int)(chunks - g0 < G ? chunks - g0 : G);   // chunks in this group
        DnArgs a{q, k, v, g, beta, state, out, n_tok, g0, H, kd, vd, vec};
        hipLaunchKernelGGL(k_dn_chunk, dim3((unsigned)(gc * H), 3), dim3(DN_WG), 0, st, a, s);
        hipLaunchKernelGGL(k_dn_carry, dim3((unsigned)(ncol * H)), dim3(512), 0, st, a, s, gc, ncol);
    }
    return hipGetLastError();
}

}  // namespace qk
