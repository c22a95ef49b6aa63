// The chunked gated delta rule, forward and backward (crates/dash-ops/src/gated_delta/chunk.rs,
// chunk/cube.rs): the plan over packed sequences, and the f32 kernel set (any dtype, heads up to
// 256 wide, f32 arithmetic throughout). The 16-bit MFMA kernels are in gdr_chunk_mfma.hip and are
// chosen when they take the call.
//
// Notation per chunk of C = 64 tokens (chunk/reference.rs:11-18), Q already scaled:
//   G = cumsum(g), gamma = exp(G), lam = exp(G_last - G), decay_ij = exp(G_i - G_j) (i >= j)
//   A_ij = beta_i (k_i . k_j) decay_ij (i > j), T = (I + A)^-1
//   W = T (beta gamma K), U = T (beta V), V' = U - W S, O = (gamma Q) S + (Q K^T o decay) V'
//   S_next = exp(G_last) S + (lam K)^T V'.
//
// Launches (forward): plan -> prep (per chunk and head) -> state pass (per sequence and head,
// serial over its chunks) -> output (per chunk and head). Backward: plan -> prep -> state pass
// -> local terms (per chunk) -> reverse state pass (per sequence) -> gradients (per chunk, four
// launches).
#include <string>

#include "attention_kernels.h"
#include "gdr_common.h"
#include "mfma.h"

namespace dm {

// ------------------------------------------------------------------------------------------
// Plan (chunk/cube.rs:80-175) of packed sequences: per sequence its first chunk, per chunk its first
// token and token count. Sequences are chunked from their own first token; every chunk index up to
// the host's bound n_max that no sequence uses gets a count of 0. A batch without offsets needs no
// plan: GdrPlan has it in closed form.
// ------------------------------------------------------------------------------------------

__global__ __launch_bounds__(1024) void gdr_plan(int64_t nseq, int64_t T, int64_t n_max,
                                                 const int32_t *__restrict__ cu, GdrPlan p) {
    int32_t *seq_chunk0 = p.seq_chunk0, *chunk_tok0 = p.chunk_tok0, *chunk_len = p.chunk_len,
            *seq_order = p.seq_order;
    __shared__ int32_t part[1024];
    const int tid = threadIdx.x;
    const int64_t per = (nseq + 1023) / 1024;
    const int64_t s0 = tid * per, s1 = s0 + per < nseq ? s0 + per : nseq;
    auto span = [&](int64_t s, int64_t *a, int64_t *b) {
        *a = cu[s];
        *b = cu[s + 1];
        if (*a < 0) *a = 0;
        if (*b > T) *b = T;  // malformed offsets stay inside the tokens (cube.rs:80-91)
        if (*b < *a) *b = *a;
    };
    // chunks per thread's sequences, then an inclusive scan over the threads
    int32_t local = 0;
    for (int64_t s = s0; s < s1; s++) {
        int64_t a, b;
        span(s, &a, &b);
        local += (int32_t)((b - a + kChunk - 1) / kChunk);
    }
    part[tid] = local;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        const int32_t y = tid >= o ? part[tid - o] : 0;
        __syncthreads();
        part[tid] += y;
        __syncthreads();
    }
    int32_t c = part[tid] - local;
    for (int64_t s = s0; s < s1; s++) {
        int64_t a, b;
        span(s, &a, &b);
        seq_chunk0[s] = c < n_max ? c : (int32_t)n_max;
        c += (int32_t)((b - a + kChunk - 1) / kChunk);
    }
    const int32_t used = part[1023] < n_max ? part[1023] : (int32_t)n_max;
    if (tid == 0) seq_chunk0[nseq] = used;
    __syncthreads();  // (orders the global writes above for the whole workgroup)
    // the sequences by chunk count, the most first (ties by index): the state passes start the
    // longest chains first. Past kOrderMax sequences, the identity.
    for (int64_t s = tid; s < nseq; s += 1024) {
        if (nseq > kOrderMax) {
            seq_order[s] = (int32_t)s;
            continue;
        }
        const int32_t n = seq_chunk0[s + 1] - seq_chunk0[s];
        int32_t rank = 0;
        for (int64_t u = 0; u < nseq; u++) {
            const int32_t m = seq_chunk0[u + 1] - seq_chunk0[u];
            rank += (m > n) | ((m == n) & (u < s));
        }
        seq_order[rank] = (int32_t)s;
    }
    // every chunk in parallel: its sequence is the last whose first chunk is at or before it
    for (int64_t x = tid; x < n_max; x += 1024) {
        if (x >= used) {
            chunk_tok0[x] = 0;
            chunk_len[x] = 0;
            continue;
        }
        int64_t lo = 0, hi = nseq - 1;  // seq_chunk0[lo] <= x
        while (lo < hi) {
            const int64_t mid = (lo + hi + 1) >> 1;
            if (seq_chunk0[mid] <= x)
                lo = mid;
            else
                hi = mid - 1;
        }
        int64_t a, b;
        span(lo, &a, &b);
        const int64_t t = a + (x - seq_chunk0[lo]) * kChunk;
        chunk_tok0[x] = (int32_t)t;
        chunk_len[x] = (int32_t)(b - t < kChunk ? b - t : kChunk);
    }
}

// ------------------------------------------------------------------------------------------
// 64 x 64 products in f32 on the matrix cores (v_mfma_f32_16x16x4_f32), by a workgroup of four
// wavefronts, each a 32 x 32 quadrant of 2 x 2 tiles of 16 x 16.
//
// Both operands lie in LDS with k contiguous (A as [row][k], B as [column][k]), rows padded by 4
// floats, so a lane reads its 4 consecutive k of a row with one 16-byte access free of bank
// conflicts; which k of the 16 a step covers falls to which lane does not matter as long as A and
// B agree: lane l takes k = 4 (l / 16) + r in product r. One such read per operand tile feeds four
// products of 32 cycles each, so the matrix cores are not waiting on LDS. Operands in memory come
// through panels of 64 x 32, the next panel's loads in flight while this one's products run.
// The f32 rate of the matrix cores is twice the vector unit's (packed f32 is not used here). The
// one-lane-per-element dot products that these replace ran at 0.2 TFLOP/s, every multiply waiting
// on two loads, with each (sequence, head) on one compute unit in the state passes: forward and
// backward of 2048 tokens in sequences of 700, 1001 and 347, 8 heads of 128, took 48.4 ms (state
// passes 11.4 and 16.3 ms, gradients 6.2 ms) and take 0.44 ms (state passes 40 and 46 us, prep 59
// us, the gradients' four launches 129 us). What bounds a call of that size is latency: 33 chunks of 8 heads are
// one workgroup per compute unit, each a chain of panels (load, barrier, products).
// ------------------------------------------------------------------------------------------

constexpr int kPan = 32;           // k columns of a panel
constexpr int kPanS = kPan + 4;    // a panel's row stride
constexpr int kMatS = kChunk + 4;  // row stride of a 64 x 64 matrix in LDS
constexpr int kPanels = 64 * kPanS;

typedef f32x4_t Quad[2][2];

__device__ __forceinline__ void zero_quad(Quad &acc) {
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i >> 1][i & 1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
}

__device__ __forceinline__ float at4(const float4 &v, int r) {
    return r == 0 ? v.x : r == 1 ? v.y : r == 2 ? v.z : v.w;
}

// acc += A[64 x K] B[K x 64], this wavefront's quadrant.
template <int K>
__device__ __forceinline__ void mma64(Quad &acc, const float *A, int lda, const float *B, int ldb) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const float *pa = A + ((wave >> 1) * 32 + (lane & 15)) * lda + 4 * (lane >> 4);
    const float *pb = B + ((wave & 1) * 32 + (lane & 15)) * ldb + 4 * (lane >> 4);
#pragma unroll
    for (int s = 0; s < K / 16; s++) {
        const float4 a0 = *(const float4 *)(pa + 16 * s), a1 = *(const float4 *)(pa + 16 * lda + 16 * s);
        const float4 b0 = *(const float4 *)(pb + 16 * s), b1 = *(const float4 *)(pb + 16 * ldb + 16 * s);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            acc[0][0] = mfma4(at4(a0, r), at4(b0, r), acc[0][0]);
            acc[0][1] = mfma4(at4(a0, r), at4(b1, r), acc[0][1]);
            acc[1][0] = mfma4(at4(a1, r), at4(b0, r), acc[1][0]);
            acc[1][1] = mfma4(at4(a1, r), at4(b1, r), acc[1][1]);
        }
    }
}

// A panel's load: f(row, c) gives four consecutive floats of the operand in memory. Without TR
// the memory has k contiguous (f(i, k)); with TR its rows are k (f(k, i)) and the panel is
// transposed on its way into LDS (8 rows x 128 bytes a wavefront's load, the four 4-byte writes
// of a lane at worst 2-way bank conflicts).
template <bool TR, class F>
__device__ __forceinline__ void panel_load(float4 (&r)[2], F f, int k0) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        if constexpr (TR) {
            r[u] = f(k0 + ((tid >> 3) & 7) + 8 * (tid >> 6), 4 * ((tid & 7) + 8 * u));
        } else {
            const int x = tid + 256 * u;
            r[u] = f(x >> 3, k0 + 4 * (x & 7));
        }
    }
}
template <bool TR>
__device__ __forceinline__ void panel_store(const float4 (&r)[2], float *p) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        if constexpr (TR) {
            float *d = p + 4 * ((tid & 7) + 8 * u) * kPanS + ((tid >> 3) & 7) + 8 * (tid >> 6);
#pragma unroll
            for (int e = 0; e < 4; e++) d[e * kPanS] = at4(r[u], e);
        } else {
            const int x = tid + 256 * u;
            *(float4 *)(p + (x >> 3) * kPanS + 4 * (x & 7)) = r[u];
        }
    }
}

// acc += A B over K (a multiple of 32) with both operands in memory; sm: two panels. A workgroup
// barrier comes before the first write to sm.
template <bool TA, bool TB, class FA, class FB>
__device__ __forceinline__ void gemm64(Quad &acc, FA fa, FB fb, int K, float *sm) {
    float4 ra[2], rb[2];
    panel_load<TA>(ra, fa, 0);
    panel_load<TB>(rb, fb, 0);
    for (int k0 = 0; k0 < K; k0 += kPan) {
        __syncthreads();
        panel_store<TA>(ra, sm);
        panel_store<TB>(rb, sm + kPanels);
        __syncthreads();
        if (k0 + kPan < K) {
            panel_load<TA>(ra, fa, k0 + kPan);
            panel_load<TB>(rb, fb, k0 + kPan);
        }
        mma64<kPan>(acc, sm, kPanS, sm + kPanels, kPanS);
    }
}
// The same with A a 64 x 64 matrix resident in LDS.
template <bool TB, class FB>
__device__ __forceinline__ void gemm64_lds(Quad &acc, const float *A, FB fb, float *sm) {
    float4 rb[2];
    panel_load<TB>(rb, fb, 0);
    for (int k0 = 0; k0 < kChunk; k0 += kPan) {
        __syncthreads();
        panel_store<TB>(rb, sm);
        __syncthreads();
        if (k0 + kPan < kChunk) panel_load<TB>(rb, fb, k0 + kPan);
        mma64<kPan>(acc, A + k0, kMatS, sm, kPanS);
    }
}

// Products with a triangular matrix (A[i][k], used where k <= i, or with UPPER where k >= i): the zeros of
// its other half are multiplied like the rest, and 0 * inf is NaN, so a token's value that is not
// finite would reach tokens that do not depend on it (the earlier ones forward). Such a product is NaN
// somewhere; a workgroup that finds one takes the sum again term by term over the triangle alone
// (finite inputs pay the test: 16 compares a lane and a barrier).
__device__ __forceinline__ bool not_finite(const Quad &acc) {
    bool bad = false;
#pragma unroll
    for (int ti = 0; ti < 2; ti++)
#pragma unroll
        for (int tj = 0; tj < 2; tj++)
#pragma unroll
            for (int r = 0; r < 4; r++) bad |= !(fabsf(acc[ti][tj][r]) < INFINITY);
    return bad;
}
// Whether any thread of the workgroup says so; a barrier must lie between two uses of sm (4 ints).
__device__ __forceinline__ bool block_any(bool x, int *sm) {
    const bool w = __any(x);
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = w;
    __syncthreads();
    return (sm[0] | sm[1] | sm[2] | sm[3]) != 0;
}
// acc += A B over the triangle; fa, fb, TA and TB as gemm64's.
template <bool TA, bool TB, bool UPPER, class FA, class FB>
__device__ __forceinline__ void tri_sum(Quad &acc, FA fa, FB fb) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i0 = (wave >> 1) * 32 + 4 * (lane >> 4), j0 = (wave & 1) * 32 + (lane & 15);
#pragma unroll 1
    for (int k = 0; k < kChunk; k++) {
        float b[2];
#pragma unroll
        for (int tj = 0; tj < 2; tj++) {
            const int j = j0 + 16 * tj;
            b[tj] = TB ? at4(fb(k, j & ~3), j & 3) : at4(fb(j, k & ~3), k & 3);
        }
#pragma unroll
        for (int ti = 0; ti < 2; ti++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = i0 + 16 * ti + r;
                const float a = TA ? at4(fa(k, i & ~3), i & 3) : at4(fa(i, k & ~3), k & 3);
                if (UPPER ? k >= i : k <= i) {
                    acc[ti][0][r] = fmaf(a, b[0], acc[ti][0][r]);
                    acc[ti][1][r] = fmaf(a, b[1], acc[ti][1][r]);
                }
            }
    }
}

// f(row, column, values): rows row .. row + 3 of one column, for each tile of the quadrant.
template <class F>
__device__ __forceinline__ void each4(const Quad &acc, F f) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int ti = 0; ti < 2; ti++)
#pragma unroll
        for (int tj = 0; tj < 2; tj++)
            f((wave >> 1) * 32 + ti * 16 + 4 * (lane >> 4), (wave & 1) * 32 + tj * 16 + (lane & 15),
              acc[ti][tj]);
}

// Sums of a 64 x 64 matrix held as quadrants, in a fixed order: of its rows into red[2][64] (the
// two column halves), of its columns into red[2][64] (the two row halves).
__device__ __forceinline__ void row_sums(const Quad &v, float *red) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int ti = 0; ti < 2; ti++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float s = group_sum<16>(v[ti][0][r] + v[ti][1][r]);
            if ((lane & 15) == 0)
                red[(wave & 1) * 64 + (wave >> 1) * 32 + ti * 16 + 4 * (lane >> 4) + r] = s;
        }
}
__device__ __forceinline__ void col_sums(const Quad &v, float *red) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int tj = 0; tj < 2; tj++) {
        float s = 0.f;
#pragma unroll
        for (int ti = 0; ti < 2; ti++)
#pragma unroll
            for (int r = 0; r < 4; r++) s += v[ti][tj][r];
        s += __shfl_xor(s, 16, 64);
        s += __shfl_xor(s, 32, 64);
        if (lane < 16) red[(wave >> 1) * 64 + (wave & 1) * 32 + tj * 16 + lane] = s;
    }
}

__device__ __forceinline__ float4 scaled(const float4 &v, float s) {
    return make_float4(v.x * s, v.y * s, v.z * s, v.w * s);
}
__device__ __forceinline__ float4 as_f4(const f32x4_t &v) { return make_float4(v[0], v[1], v[2], v[3]); }

// Rows of `ld` floats, four at a time.
struct Rows {
    const float *p;
    int64_t ld;
    __device__ __forceinline__ float4 operator()(int r, int c) const {
        return *(const float4 *)(p + r * ld + c);
    }
};

// ------------------------------------------------------------------------------------------
// Prep (intra, chunk/reference.rs:429-479): per (chunk, head) the input rows as f32 padded to
// multiples of 64 columns (zeros past a width and past the chunk's tokens), queries and keys
// normalised, queries scaled; G; A and P = Q K^T o decay; T = (I + A)^-1; W and U.
// T in f32 by 16 x 16 blocks: each diagonal block by column forward substitution (a wavefront a
// block), the blocks below by doubling, T21 = -T22 (A21 T11).
// ------------------------------------------------------------------------------------------

// One wavefront's 16 x 16 block product over k = 16: A[i][k] at A, B[k][j] at B.
__device__ __forceinline__ f32x4_t block16(const float *A, int lda, const float *B, int ldb, f32x4_t acc) {
    const int c = threadIdx.x & 15, g = (threadIdx.x >> 4) & 3;
#pragma unroll
    for (int s = 0; s < 4; s++) acc = mfma4(A[c * lda + 4 * s + g], B[(4 * s + g) * ldb + c], acc);
    return acc;
}

template <int DT, bool BWD>
__global__ __launch_bounds__(256) void gdr_prep(GdrArgs a, GdrWs w, const void *d_out) {
    const int64_t ch = blockIdx.x, n = ch / a.H, h = ch % a.H;
    const int len = w.plan.len(n);
    if (len == 0) return;
    const int64_t tok0 = w.plan.tok0(n);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t Dk = a.Dk, Dv = a.Dv, KP = w.KP, VP = w.VP;
    __shared__ float4 smem[(2 * kPanels + 2 * kChunk * kMatS) / 4];
    __shared__ double G[kChunk];
    __shared__ float gam[kChunk], bet[kChunk], lam[kChunk];
    __shared__ int flag[4];
    float *pan = (float *)smem, *Ts = pan + 2 * kPanels, *As = Ts + kChunk * kMatS;
    float *mm = pan;  // four 16 x 16 blocks, while no panel is in use

    float *qn = w.qn + ch * kChunk * KP, *kn = w.kn + ch * kChunk * KP;
    float *vp = w.vp + ch * kChunk * VP;
    // 16 lanes a row, a row's loads all issued before any is used
    float *dop = BWD ? w.dop + ch * kChunk * VP : nullptr;
#pragma unroll 2
    for (int it = 0; it < 4; it++) {
        const int i = it * 16 + wave * 4 + (lane >> 4), c0 = 4 * (lane & 15);
        const int64_t tok = tok0 + (i < len ? i : len - 1);
        float x[BWD ? 4 : 3][4][4];  // q, k, v, d_out
        auto row = [&](float (&d)[4][4], const void *p, int64_t at, int64_t D) {
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int e = 0; e < 4; e++) d[c][e] = 64 * c + c0 + e < D ? ld<DT>(p, at + 64 * c + c0 + e) : 0.f;
        };
        row(x[0], a.q, q_at(a, tok, h), Dk);
        row(x[1], a.k, k_at(a, tok, h), Dk);
        row(x[2], a.v, v_at(a, tok, h), Dv);
        if constexpr (BWD) row(x[3], d_out, o_at(a, tok, h), Dv);
        float sq = 0.f, sk = 0.f, qi = 1.f, ki = 1.f;
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
#pragma unroll
                for (int m = 0; m < (BWD ? 4 : 3); m++) x[m][c][e] = i < len ? x[m][c][e] : 0.f;
                sq += x[0][c][e] * x[0][c][e];
                sk += x[1][c][e] * x[1][c][e];
            }
        if (a.l2norm) {
            qi = 1.f / sqrtf(group_sum<16>(sq) + 1e-6f);
            ki = 1.f / sqrtf(group_sum<16>(sk) + 1e-6f);
            if (BWD && (lane & 15) == 0) {
                w.inv[ch * 2 * kChunk + i] = qi;
                w.inv[ch * 2 * kChunk + kChunk + i] = ki;
            }
        }
        auto put = [&](float *d, int64_t ld, const float (&v)[4][4], float f1, float f2) {
#pragma unroll
            for (int c = 0; c < 4; c++)
                if (64 * c < ld)
                    *(float4 *)(d + i * ld + 64 * c + c0) =
                        make_float4(v[c][0] * f1 * f2, v[c][1] * f1 * f2, v[c][2] * f1 * f2, v[c][3] * f1 * f2);
        };
        put(qn, KP, x[0], qi, a.scale);
        put(kn, KP, x[1], ki, 1.f);
        put(vp, VP, x[2], 1.f, 1.f);
        if constexpr (BWD) put(dop, VP, x[3], 1.f, 1.f);
    }
    if (tid < 4) flag[tid] = 0;
    if (wave == 0) {
        const bool ok = lane < len;
        double x = ok ? ld_any(a.g_dt, a.g, g_at(a, tok0 + lane, h)) : 0.f;
        bet[lane] = ok ? ld_any(a.beta_dt, a.beta, b_at(a, tok0 + lane, h)) : 0.f;
        // G = cumsum(g) by an inclusive scan across the wavefront, in f64: the decays are
        // exponentials of differences of sums of the size of 50, whose f32 rounding would be the
        // largest error of the final state
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const double y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        G[lane] = x;
        gam[lane] = expf((float)x);
        lam[lane] = expf((float)(__shfl(x, kChunk - 1, 64) - x));
        w.G[ch * kChunk + lane] = x;
    }
    __syncthreads();  // the rows just written are read back below, by this workgroup alone

    // K K^T and Q K^T (they share the key panels); nothing above the diagonal is kept
    Quad kk, qk;
    zero_quad(kk);
    zero_quad(qk);
    {
        const Rows fq{qn, KP}, fk{kn, KP};
        float4 rq[2], rk[2];
        panel_load<false>(rq, fq, 0);
        panel_load<false>(rk, fk, 0);
        for (int k0 = 0; k0 < KP; k0 += kPan) {
            __syncthreads();
            panel_store<false>(rq, pan);
            panel_store<false>(rk, pan + kPanels);
            __syncthreads();
            if (k0 + kPan < KP) {
                panel_load<false>(rq, fq, k0 + kPan);
                panel_load<false>(rk, fk, k0 + kPan);
            }
            if (wave != 1) {  // wavefront 1's quadrant is all above the diagonal
                mma64<kPan>(kk, pan + kPanels, kPanS, pan + kPanels, kPanS);
                mma64<kPan>(qk, pan, kPanS, pan + kPanels, kPanS);
            }
        }
    }
    float *Pg = w.P + ch * kChunk * kChunk, *Ag = BWD ? w.Am + ch * kChunk * kChunk : nullptr;
#pragma unroll
    for (int ti = 0; ti < 2; ti++)
#pragma unroll
        for (int tj = 0; tj < 2; tj++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = (wave >> 1) * 32 + ti * 16 + 4 * (lane >> 4) + r;
                const int j = (wave & 1) * 32 + tj * 16 + (lane & 15);
                // masked before the exponential
                const float dec = expf(i >= j ? (float)(G[i] - G[j]) : 0.f);
                const float av = i > j ? bet[i] * kk[ti][tj][r] * dec : 0.f;
                As[i * kMatS + j] = av;
                Pg[i * kChunk + j] = i >= j ? qk[ti][tj][r] * dec : 0.f;
                if constexpr (BWD) Ag[i * kChunk + j] = av;
            }
    __syncthreads();
    bool bad = false;  // T is not finite somewhere
    auto note = [&](const f32x4_t &v) {
#pragma unroll
        for (int r = 0; r < 4; r++) bad |= !(fabsf(v[r]) < INFINITY);
        return v;
    };
    {
        // diagonal block b = wave, lane c holding column c of its inverse:
        // T[i][c] = [i == c] - sum_{x < i} A[i][x] T[x][c]
        const int b = wave, c = lane & 15;
        float tc[16];
#pragma unroll
        for (int i = 0; i < 16; i++) {
            float sp[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int x4 = 0; x4 < i; x4 += 4) {
                const float4 a4 = *(const float4 *)(As + (16 * b + i) * kMatS + 16 * b + x4);
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (x4 + e < i) sp[e] += at4(a4, e) * tc[x4 + e];
            }
            tc[i] = (i == c ? 1.f : 0.f) - ((sp[0] + sp[1]) + (sp[2] + sp[3]));
            bad |= !(fabsf(tc[i]) < INFINITY);
        }
        if (lane < 16) {
#pragma unroll
            for (int i = 0; i < 16; i++) Ts[(16 * b + i) * kMatS + 16 * b + c] = tc[i];
        }
        for (int x = lane; x < 256; x += 64)
            for (int bj = b + 1; bj < 4; bj++) Ts[(16 * b + x / 16) * kMatS + 16 * bj + x % 16] = 0.f;
    }
    __syncthreads();
    {
        const int c = lane & 15, r0 = 4 * (lane >> 4);
        const f32x4_t z = {0.f, 0.f, 0.f, 0.f};
        auto put = [&](float *d, int ldd, const f32x4_t &v, float s) {
#pragma unroll
            for (int r = 0; r < 4; r++) d[(r0 + r) * ldd + c] = s * v[r];
        };
        auto blk = [&](float *m, int bi, int bj) { return m + 16 * bi * kMatS + 16 * bj; };
        // the diagonal 32 x 32 halves (wavefronts 0 and 1)
        const int bj1 = 2 * (wave & 1), bi1 = bj1 + 1;
        if (wave < 2) put(mm + wave * 320, 20, block16(blk(As, bi1, bj1), kMatS, blk(Ts, bj1, bj1), kMatS, z), 1.f);
        __syncthreads();
        if (wave < 2)
            put(blk(Ts, bi1, bj1), kMatS, note(block16(blk(Ts, bi1, bi1), kMatS, mm + wave * 320, 20, z)), -1.f);
        __syncthreads();
        // the lower-left quarter, wavefront w its block (2 + w / 2, w % 2)
        const int bi = 2 + (wave >> 1), bj = wave & 1;
        f32x4_t x = z;
        for (int kb = bj; kb < 2; kb++) x = block16(blk(As, bi, kb), kMatS, blk(Ts, kb, bj), kMatS, x);
        put(mm + wave * 320, 20, x, 1.f);
        __syncthreads();
        x = z;
        for (int kb = 2; kb <= bi; kb++)
            x = block16(blk(Ts, bi, kb), kMatS, mm + (2 * (kb - 2) + bj) * 320, 20, x);
        put(blk(Ts, bi, bj), kMatS, note(x), -1.f);
        if (__any(bad) && lane == 0) flag[wave] = 1;
    }
    __syncthreads();
    if (flag[0] | flag[1] | flag[2] | flag[3]) {
        // a column a thread, row after row, so that a row comes from the ones before it alone
        if (tid < kChunk) {
            for (int i = 0; i < kChunk; i++) {
                float s = i == tid ? 1.f : 0.f;
                for (int x = tid; x < i; x++) s -= As[i * kMatS + x] * Ts[x * kMatS + tid];
                Ts[i * kMatS + tid] = s;
            }
        }
        __syncthreads();
    }
    if constexpr (BWD) {
        float *Tg = w.Tm + ch * kChunk * kChunk;
        for (int x = tid; x < kChunk * kChunk / 4; x += 256)
            *(float4 *)(Tg + 4 * x) = *(const float4 *)(Ts + (x >> 4) * kMatS + 4 * (x & 15));
    }
    // W = T (beta gamma K), U = T (beta V); W as the state pass's rows and, for the backward's,
    // transposed; U transposed
    auto wu = [&](auto product) {
        bool bad = false;
        for (int x0 = 0; x0 < KP; x0 += 64) {
            Quad acc;
            zero_quad(acc);
            product(acc, [&](int j, int c) {
                return scaled(*(const float4 *)(kn + j * KP + x0 + c), bet[j] * gam[j]);
            });
            bad |= not_finite(acc);
            each4(acc, [&](int i, int x, const f32x4_t &v) {
                float *W = w.W + ch * kChunk * KP;
#pragma unroll
                for (int r = 0; r < 4; r++) W[(i + r) * KP + x0 + x] = v[r];
                if constexpr (BWD) *(float4 *)(w.WT + ch * kChunk * KP + (x0 + x) * kChunk + i) = as_f4(v);
            });
        }
        for (int y0 = 0; y0 < VP; y0 += 64) {
            Quad acc;
            zero_quad(acc);
            product(acc, [&](int j, int c) { return scaled(*(const float4 *)(vp + j * VP + y0 + c), bet[j]); });
            bad |= not_finite(acc);
            each4(acc, [&](int i, int y, const f32x4_t &v) {
                *(float4 *)(w.UT + ch * kChunk * VP + (y0 + y) * kChunk + i) = as_f4(v);
            });
        }
        return bad;
    };
    if (block_any(wu([&](Quad &acc, auto f) { gemm64_lds<true>(acc, Ts, f, pan); }), flag))
        wu([&](Quad &acc, auto f) { tri_sum<false, true, false>(acc, Rows{Ts, kMatS}, f); });
    // (lam K)^T
    float *KT = w.KT + ch * kChunk * KP;
    const int ld = (int)KP;
#pragma unroll 4
    for (int x = tid; x < ld * (kChunk / 4); x += 256) {
        const int i4 = 4 * (x % (kChunk / 4)), c = x / (kChunk / 4);
        const float *k = kn + i4 * ld + c;
        *(float4 *)(KT + c * kChunk + i4) = make_float4(k[0] * lam[i4], k[ld] * lam[i4 + 1],
                                                        k[2 * ld] * lam[i4 + 2], k[3 * ld] * lam[i4 + 3]);
    }
}

// ------------------------------------------------------------------------------------------
// State passes, per (sequence, head, 16 NT columns of the state), serial over the chunks, the
// state (64 KTn x 16 NT) in the products' accumulators, its rows split over four wavefronts:
//   forward   (chunk/reference.rs:348-372):  V' = U - W S;  S <- exp(G_last) S + (lam K)^T V'
//   backward  (:382-427), from the last chunk: dV' = lam o (K dS) + dv_local;
//             dS <- exp(G_last) dS + (gamma Q)^T dO - W^T dV'.
// Each stores the state its chunk is entered with, and V' or dV', transposed (a lane holds 4
// consecutive rows of a column). The state and V' change hands through LDS, two barriers a chunk;
// the operands W and (lam K)^T (K and W^T) come from memory straight into registers, 16 bytes a
// lane, as soon as the products have taken the previous chunk's. A chunk is two chains of
// 16 KTn and 16 KTn dependent products per wavefront and column tile, so the columns are split
// as finely as the chip has room for: 16 a workgroup until that makes about a workgroup per
// compute unit, else 32 (half the operand reads per column).
// ------------------------------------------------------------------------------------------

template <int KTn, int NT, bool BWD>
__global__ __launch_bounds__(256) void gdr_chain(GdrArgs a, GdrWs w, int64_t nsh, int64_t nshp,
                                                 const float *init, float *final_state) {
    // the column blocks of a (sequence, head) nshp (a multiple of 8) workgroups apart: on one XCD
    const int64_t slot = blockIdx.x % nshp;
    if (slot >= nsh) return;
    const int64_t s = w.plan.order(slot / a.H), h = slot % a.H, sh = s * a.H + h;
    const int y0 = (int)(blockIdx.x / nshp) * 16 * NT;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane & 15, g4 = 4 * (lane >> 4);
    constexpr int KP = 64 * KTn, SS = KP + 4;
    const int64_t Dk = a.Dk, Dv = a.Dv, VP = w.VP;
    const int c0 = w.plan.first(s), c1 = w.plan.first(s + 1);
    __shared__ float4 st4[16 * NT * SS / 4], vt4[16 * NT * kMatS / 4];
    float *St = (float *)st4, *Vt = (float *)vt4;

    // the wavefront's state tile t: rows xr(t) + [0, 4), column y0 + 16 nt + c
    auto xr = [&](int t) { return wave * 16 * KTn + 16 * t + g4; };
    f32x4_t S[KTn][NT];
#pragma unroll
    for (int t = 0; t < KTn; t++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int64_t x = xr(t) + r, y = y0 + 16 * nt + c;
                S[t][nt][r] = init && x < Dk && y < Dv ? init[(sh * Dk + x) * Dv + y] : 0.f;
            }

    const float *A1 = BWD ? w.kn : w.W, *A2 = BWD ? w.WT : w.KT, *add = BWD ? w.dvlT : w.UT;
    float *Sout = BWD ? w.dSnT : w.ScT, *Vout = BWD ? w.dVnT : w.VnT;
    float4 a1[4 * KTn], a2[KTn][4], au[NT], af[KTn][NT];
    double gr[4], gl;
    auto load1 = [&](int cc) {
        const float *p = A1 + ((int64_t)cc * a.H + h) * kChunk * KP + (16 * wave + c) * KP + g4;
#pragma unroll
        for (int i = 0; i < 4 * KTn; i++) a1[i] = *(const float4 *)(p + 16 * i);
    };
    auto load2 = [&](int cc) {
        const int64_t ch = (int64_t)cc * a.H + h;
        const float *p = A2 + ch * kChunk * KP + (wave * 16 * KTn + c) * kChunk + g4;
#pragma unroll
        for (int t = 0; t < KTn; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) a2[t][i] = *(const float4 *)(p + t * 16 * kChunk + 16 * i);
        if constexpr (BWD) {
#pragma unroll
            for (int t = 0; t < KTn; t++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    af[t][nt] = *(const float4 *)(w.F + (ch * VP + y0 + 16 * nt + c) * KP + xr(t));
        }
    };
    auto load0 = [&](int cc) {
        const int64_t ch = (int64_t)cc * a.H + h;
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
            au[nt] = *(const float4 *)(add + (ch * VP + y0 + 16 * nt + c) * kChunk + 16 * wave + g4);
        if constexpr (BWD) {
#pragma unroll
            for (int r = 0; r < 4; r++) gr[r] = w.G[ch * kChunk + 16 * wave + g4 + r];
        }
        gl = w.G[ch * kChunk + kChunk - 1];
    };
    const int n = c1 - c0;
    auto chunk_of = [&](int i) { return BWD ? c1 - 1 - i : c0 + i; };
    if (n > 0) {
        load0(chunk_of(0));
        load1(chunk_of(0));
        load2(chunk_of(0));
    }
    for (int i = 0; i < n; i++) {
        const int64_t ch = (int64_t)chunk_of(i) * a.H + h;
        const int nx = chunk_of(i + 1 < n ? i + 1 : i);
#pragma unroll
        for (int t = 0; t < KTn; t++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const float4 v = as_f4(S[t][nt]);
                *(float4 *)(St + (16 * nt + c) * SS + xr(t)) = v;
                *(float4 *)(Sout + (ch * VP + y0 + 16 * nt + c) * KP + xr(t)) = v;
            }
        __syncthreads();
        f32x4_t m[NT];
#pragma unroll
        for (int nt = 0; nt < NT; nt++) m[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 4 * KTn; k++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const float4 b = *(const float4 *)(St + (16 * nt + c) * SS + 16 * k + g4);
#pragma unroll
                for (int r = 0; r < 4; r++) m[nt] = mfma4(at4(a1[k], r), at4(b, r), m[nt]);
            }
        load1(nx);
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            f32x4_t v;
#pragma unroll
            for (int r = 0; r < 4; r++)
                v[r] = BWD ? m[nt][r] * expf((float)(gl - gr[r])) + at4(au[nt], r) : at4(au[nt], r) - m[nt][r];
            *(float4 *)(Vout + (ch * VP + y0 + 16 * nt + c) * kChunk + 16 * wave + g4) = as_f4(v);
            *(float4 *)(Vt + (16 * nt + c) * kMatS + 16 * wave + g4) = BWD ? as_f4(-v) : as_f4(v);
        }
        const float e = expf((float)gl);
        load0(nx);
        __syncthreads();
#pragma unroll
        for (int t = 0; t < KTn; t++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    S[t][nt][r] = BWD ? S[t][nt][r] * e + at4(af[t][nt], r) : S[t][nt][r] * e;
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const float4 b = *(const float4 *)(Vt + (16 * nt + c) * kMatS + 16 * k + g4);
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int t = 0; t < KTn; t++)
                        S[t][nt] = mfma4(at4(a2[t][k], r), at4(b, r), S[t][nt]);
            }
        load2(nx);
    }
    if (final_state) {
#pragma unroll
        for (int t = 0; t < KTn; t++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int64_t x = xr(t) + r, y = y0 + 16 * nt + c;
                    if (x < Dk && y < Dv) final_state[(sh * Dk + x) * Dv + y] = S[t][nt][r];
                }
    }
}

// ------------------------------------------------------------------------------------------
// Output (forward, chunk/reference.rs:502-508), per (chunk, head) and 64 columns:
// O = (gamma Q) S + P V'.
// ------------------------------------------------------------------------------------------

template <int DT>
__global__ __launch_bounds__(256) void gdr_output(GdrArgs a, GdrWs w, void *out) {
    const int64_t ch = blockIdx.x, n = ch / a.H, h = ch % a.H;
    const int len = w.plan.len(n);
    if (len == 0) return;
    const int64_t tok0 = w.plan.tok0(n), KP = w.KP, VP = w.VP;
    const int y0 = blockIdx.y * 64;
    __shared__ float4 smem[2 * kPanels / 4];
    __shared__ float gam[kChunk];
    __shared__ int flag[4];
    if (threadIdx.x < kChunk) gam[threadIdx.x] = expf((float)w.G[ch * kChunk + threadIdx.x]);
    Quad acc;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const Rows fp{w.P + ch * kChunk * kChunk, kChunk}, fv{w.VnT + (ch * VP + y0) * kChunk, kChunk};
    auto from_state = [&] {
        zero_quad(acc);
        gemm64<false, false>(acc, Rows{w.qn + ch * kChunk * KP, KP}, Rows{w.ScT + (ch * VP + y0) * KP, KP},
                             (int)KP, (float *)smem);
#pragma unroll
        for (int ti = 0; ti < 2; ti++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float gm = gam[(wave >> 1) * 32 + ti * 16 + 4 * (lane >> 4) + r];
                acc[ti][0][r] *= gm;
                acc[ti][1][r] *= gm;
            }
    };
    from_state();
    gemm64<false, false>(acc, fp, fv, kChunk, (float *)smem);
    if (block_any(not_finite(acc), flag)) {
        from_state();
        tri_sum<false, false, false>(acc, fp, fv);
    }
    each4(acc, [&](int i, int y, const f32x4_t &v) {
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (i + r < len && y0 + y < a.Dv)
                st<DT>(out, ((tok0 + i + r) * a.H + h) * a.Dv + y0 + y, v[r]);
    });
}

// ------------------------------------------------------------------------------------------
// Backward (chunk/reference.rs:519-695)
// ------------------------------------------------------------------------------------------

// What the reverse state pass adds at each chunk, per (chunk, head): in blocks y < VP / 64 the
// columns of dv_local = P^T dO, in the others a 64 x 64 tile of F = (gamma Q)^T dO; transposed.
__global__ __launch_bounds__(256) void gdr_bwd_local(GdrArgs a, GdrWs w) {
    const int64_t ch = blockIdx.x, KP = w.KP, VP = w.VP;
    if (w.plan.len(ch / a.H) == 0) return;
    const int vt = (int)(VP / 64), job = blockIdx.y;
    __shared__ float4 smem[2 * kPanels / 4];
    __shared__ float gam[kChunk];
    __shared__ int flag[4];
    if (threadIdx.x < kChunk) gam[threadIdx.x] = expf((float)w.G[ch * kChunk + threadIdx.x]);
    __syncthreads();
    const int y0 = (job % vt) * 64;
    const Rows dO{w.dop + ch * kChunk * VP + y0, VP};
    Quad acc;
    zero_quad(acc);
    if (job < vt) {
        const Rows fp{w.P + ch * kChunk * kChunk, kChunk};
        gemm64<true, true>(acc, fp, dO, kChunk, (float *)smem);
        if (block_any(not_finite(acc), flag)) {
            zero_quad(acc);
            tri_sum<true, true, true>(acc, fp, dO);
        }
        each4(acc, [&](int j, int y, const f32x4_t &v) {
            *(float4 *)(w.dvlT + (ch * VP + y0 + y) * kChunk + j) = as_f4(v);
        });
    } else {
        const int x0 = (job / vt - 1) * 64;
        const float *qn = w.qn + ch * kChunk * KP + x0;
        gemm64<true, true>(acc, [&](int i, int c) {
            return scaled(*(const float4 *)(qn + i * KP + c), gam[i]);
        }, dO, kChunk, (float *)smem);
        each4(acc, [&](int x, int y, const f32x4_t &v) {
            *(float4 *)(w.F + (ch * VP + y0 + y) * KP + x0 + x) = as_f4(v);
        });
    }
}

// Per (chunk, head) and 64 key columns, from the states: d_qg = dO S^T (dq = gamma d_qg),
// d_kt = V' dS_next^T (dk = lam d_kt) and dw = -dV' S^T, with the row sums of d_qg o Q and
// d_kt o K and the tile's part of sum(S o dS_next).
__global__ __launch_bounds__(256) void gdr_bwd_states(GdrArgs a, GdrWs w) {
    const int64_t ch = blockIdx.x, KP = w.KP, VP = w.VP;
    if (w.plan.len(ch / a.H) == 0) return;
    const int x0 = blockIdx.y * 64, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    __shared__ float4 smem[5 * kPanels / 4];
    __shared__ float gam[kChunk], lam[kChunk], red[2][2 * kChunk], sds[4];
    float *pan = (float *)smem;
    if (tid < kChunk) {
        const double G = w.G[ch * kChunk + tid];
        gam[tid] = expf((float)G);
        lam[tid] = expf((float)(w.G[ch * kChunk + kChunk - 1] - G));
    }
    Quad xq, xk, xw;
    zero_quad(xq);
    zero_quad(xk);
    zero_quad(xw);
    float part = 0.f;
    {
        const Rows fo{w.dop + ch * kChunk * VP, VP}, fv{w.VnT + ch * kChunk * VP, kChunk},
            fd{w.dVnT + ch * kChunk * VP, kChunk}, fs{w.ScT + ch * VP * KP + x0, KP},
            fn{w.dSnT + ch * VP * KP + x0, KP};
        float4 ro[2], rv[2], rd[2], rs[2], rn[2];
        auto load = [&](int k0) {
            panel_load<false>(ro, fo, k0);
            panel_load<true>(rv, fv, k0);
            panel_load<true>(rd, fd, k0);
            panel_load<true>(rs, fs, k0);
            panel_load<true>(rn, fn, k0);
        };
        load(0);
        for (int k0 = 0; k0 < VP; k0 += kPan) {
            __syncthreads();
            panel_store<false>(ro, pan);
            panel_store<true>(rv, pan + kPanels);
            panel_store<true>(rd, pan + 2 * kPanels);
            panel_store<true>(rs, pan + 3 * kPanels);
            panel_store<true>(rn, pan + 4 * kPanels);
#pragma unroll
            for (int u = 0; u < 2; u++)
#pragma unroll
                for (int e = 0; e < 4; e++) part += at4(rs[u], e) * at4(rn[u], e);
            __syncthreads();
            if (k0 + kPan < VP) load(k0 + kPan);
            mma64<kPan>(xq, pan, kPanS, pan + 3 * kPanels, kPanS);
            mma64<kPan>(xk, pan + kPanels, kPanS, pan + 4 * kPanels, kPanS);
            mma64<kPan>(xw, pan + 2 * kPanels, kPanS, pan + 3 * kPanels, kPanS);
        }
    }
    const float *qn = w.qn + ch * kChunk * KP + x0, *kn = w.kn + ch * kChunk * KP + x0;
    float *gq = w.gq + ch * kChunk * KP + x0, *gk = w.gk + ch * kChunk * KP + x0,
          *dw = w.dw + ch * kChunk * KP + x0;
#pragma unroll
    for (int ti = 0; ti < 2; ti++)
#pragma unroll
        for (int tj = 0; tj < 2; tj++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = (wave >> 1) * 32 + ti * 16 + 4 * (lane >> 4) + r;
                const int64_t at = i * KP + (wave & 1) * 32 + tj * 16 + (lane & 15);
                gq[at] = xq[ti][tj][r] * gam[i];
                gk[at] = xk[ti][tj][r] * lam[i];
                dw[at] = -xw[ti][tj][r];
                xq[ti][tj][r] *= qn[at];
                xk[ti][tj][r] *= kn[at];
            }
    row_sums(xq, red[0]);
    row_sums(xk, red[1]);
    part = wave_sum(part);
    if (lane == 0) sds[wave] = part;
    __syncthreads();
    float *pt = w.part + ch * w.npart + blockIdx.y * 6 * kChunk;
    if (tid < 2 * kChunk) pt[tid] = red[tid >> 6][tid & 63] + red[tid >> 6][kChunk + (tid & 63)];
    if (tid == 0)
        w.part[ch * w.npart + w.npart - kChunk + blockIdx.y] = (sds[0] + sds[1]) + (sds[2] + sds[3]);
}

// The 64 x 64 matrices, per (chunk, head): d_attn = dO V'^T, dT = dw (beta gamma K)^T +
// dV' (beta V)^T, dA = -(T^T dT T^T) strictly lower; kept with the decay applied; and the gates'
// gradient from d_attn o P and dA o A (rows less columns).
__global__ __launch_bounds__(256) void gdr_bwd_mats(GdrArgs a, GdrWs w) {
    const int64_t ch = blockIdx.x, n = ch / a.H, h = ch % a.H, KP = w.KP, VP = w.VP;
    const int len = w.plan.len(n);
    if (len == 0) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    __shared__ float4 smem[(2 * kPanels + 3 * kChunk * kMatS) / 4];
    __shared__ double G[kChunk];
    __shared__ float bet[kChunk], bg[kChunk], red[4][2 * kChunk];
    float *pan = (float *)smem, *Tt = pan + 2 * kPanels, *Ts = Tt + kChunk * kMatS,
          *Dt = Ts + kChunk * kMatS;
    if (tid < kChunk) {
        G[tid] = w.G[ch * kChunk + tid];
        bet[tid] = tid < len ? ld_any(a.beta_dt, a.beta, b_at(a, w.plan.tok0(n) + tid, h)) : 0.f;
        bg[tid] = bet[tid] * expf((float)G[tid]);
    }
    const float *Tg = w.Tm + ch * kChunk * kChunk, *Pg = w.P + ch * kChunk * kChunk,
                *Ag = w.Am + ch * kChunk * kChunk;
    for (int x = tid; x < kChunk * kChunk / 4; x += 256) {
        const int i = x >> 4, c = 4 * (x & 15);
        const float4 v = *(const float4 *)(Tg + 4 * x);
        *(float4 *)(Ts + i * kMatS + c) = v;
#pragma unroll
        for (int e = 0; e < 4; e++) Tt[(c + e) * kMatS + i] = at4(v, e);
    }
    __syncthreads();
    const Rows fd{w.dVnT + ch * kChunk * VP, kChunk};
    Quad acc;
    zero_quad(acc);
    gemm64<false, true>(acc, Rows{w.dop + ch * kChunk * VP, VP}, Rows{w.VnT + ch * kChunk * VP, kChunk},
                        (int)VP, pan);
    float *DP = w.DPd + ch * kChunk * kChunk, *DA = w.dae + ch * kChunk * kChunk;
#pragma unroll
    for (int ti = 0; ti < 2; ti++)
#pragma unroll
        for (int tj = 0; tj < 2; tj++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = (wave >> 1) * 32 + ti * 16 + 4 * (lane >> 4) + r;
                const int j = (wave & 1) * 32 + tj * 16 + (lane & 15);
                const float d = i >= j ? acc[ti][tj][r] : 0.f;
                acc[ti][tj][r] = d * Pg[i * kChunk + j];
                DP[i * kChunk + j] = d * expf(i >= j ? (float)(G[i] - G[j]) : 0.f);  // (where Pg was)
            }
    row_sums(acc, red[0]);
    col_sums(acc, red[1]);
    zero_quad(acc);
    const float *kn = w.kn + ch * kChunk * KP, *vp = w.vp + ch * kChunk * VP;
    gemm64<false, false>(acc, Rows{w.dw + ch * kChunk * KP, KP}, [&](int j, int c) {
        return scaled(*(const float4 *)(kn + j * KP + c), bg[j]);
    }, (int)KP, pan);
    gemm64<true, false>(acc, fd, [&](int j, int c) {
        return scaled(*(const float4 *)(vp + j * VP + c), bet[j]);
    }, (int)VP, pan);
    each4(acc, [&](int x, int j, const f32x4_t &v) { *(float4 *)(Dt + j * kMatS + x) = as_f4(v); });
    __syncthreads();
    zero_quad(acc);
    mma64<kChunk>(acc, Tt, kMatS, Dt, kMatS);  // M = T^T dT
    __syncthreads();
    each4(acc, [&](int i, int x, const f32x4_t &v) {
#pragma unroll
        for (int r = 0; r < 4; r++) Dt[(i + r) * kMatS + x] = v[r];
    });
    __syncthreads();
    zero_quad(acc);
    mma64<kChunk>(acc, Dt, kMatS, Ts, kMatS);  // M T^T
#pragma unroll
    for (int ti = 0; ti < 2; ti++)
#pragma unroll
        for (int tj = 0; tj < 2; tj++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = (wave >> 1) * 32 + ti * 16 + 4 * (lane >> 4) + r;
                const int j = (wave & 1) * 32 + tj * 16 + (lane & 15);
                const float d = i > j ? -acc[ti][tj][r] : 0.f;
                acc[ti][tj][r] = d * Ag[i * kChunk + j];
                DA[i * kChunk + j] = d * expf(i > j ? (float)(G[i] - G[j]) : 0.f);  // (where Ag was)
            }
    row_sums(acc, red[2]);
    col_sums(acc, red[3]);
    __syncthreads();
    if (tid < kChunk)
        w.dgv[ch * kChunk + tid] = ((red[0][tid] + red[0][kChunk + tid]) - (red[1][tid] + red[1][kChunk + tid])) +
                                   ((red[2][tid] + red[2][kChunk + tid]) - (red[3][tid] + red[3][kChunk + tid]));
}

// The rows' gradients within the chunk, per (chunk, head) and 64 columns. Key columns:
//   dq += (d_attn o decay) K;  dk += (d_attn o decay)^T Q + beta gamma T^T dw
//         + beta (dA o decay) K + (dA o decay)^T (beta K)
// with the row sums of T^T dw o K, (dA o decay) K o K, dq o Q and dk o K; value columns:
// dv = beta T^T dV' and the row sums of T^T dV' o V.
template <int DT>
__global__ __launch_bounds__(256) void gdr_bwd_rows(GdrArgs a, GdrWs w, void *dv) {
    const int64_t ch = blockIdx.x, n = ch / a.H, h = ch % a.H, KP = w.KP, VP = w.VP;
    const int len = w.plan.len(n);
    if (len == 0) return;
    const int64_t tok0 = w.plan.tok0(n);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, kt = (int)(KP / 64);
    __shared__ float4 smem[2 * kPanels / 4];
    __shared__ float bet[kChunk], bg[kChunk], red[4][2 * kChunk];
    __shared__ int flag[4];
    float *pan = (float *)smem;
    if (tid < kChunk) {
        bet[tid] = tid < len ? ld_any(a.beta_dt, a.beta, b_at(a, tok0 + tid, h)) : 0.f;
        bg[tid] = bet[tid] * expf((float)w.G[ch * kChunk + tid]);
    }
    __syncthreads();
    const Rows ft{w.Tm + ch * kChunk * kChunk, kChunk};
    float *pt = w.part + ch * w.npart;
    if ((int)blockIdx.y >= kt) {
        const int y0 = ((int)blockIdx.y - kt) * 64;
        const float *vp = w.vp + ch * kChunk * VP + y0;
        Quad acc;
        zero_quad(acc);
        const Rows fd{w.dVnT + (ch * VP + y0) * kChunk, kChunk};
        gemm64<true, false>(acc, ft, fd, kChunk, pan);
        if (block_any(not_finite(acc), flag)) {
            zero_quad(acc);
            tri_sum<true, false, true>(acc, ft, fd);
        }
#pragma unroll
        for (int ti = 0; ti < 2; ti++)
#pragma unroll
            for (int tj = 0; tj < 2; tj++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int i = (wave >> 1) * 32 + ti * 16 + 4 * (lane >> 4) + r;
                    const int y = (wave & 1) * 32 + tj * 16 + (lane & 15);
                    if (i < len && y0 + y < a.Dv)
                        st<DT>(dv, ((tok0 + i) * a.H + h) * a.Dv + y0 + y, acc[ti][tj][r] * bet[i]);
                    acc[ti][tj][r] *= vp[i * VP + y];
                }
        row_sums(acc, red[0]);
        __syncthreads();
        if (tid < kChunk)
            pt[(kt * 6 + (int)blockIdx.y - kt) * kChunk + tid] = red[0][tid] + red[0][kChunk + tid];
        return;
    }
    const int x0 = blockIdx.y * 64;
    const float *qn = w.qn + ch * kChunk * KP + x0, *kn = w.kn + ch * kChunk * KP + x0;
    const Rows fq{qn, KP}, fk{kn, KP}, fp{w.DPd + ch * kChunk * kChunk, kChunk},
        fa{w.dae + ch * kChunk * kChunk, kChunk};
    Quad xq, xk, xw, xe;
    zero_quad(xq);
    zero_quad(xk);
    zero_quad(xw);
    zero_quad(xe);
    gemm64<false, true>(xq, fp, fk, kChunk, pan);
    gemm64<true, true>(xk, fp, fq, kChunk, pan);
    if (block_any(not_finite(xq) || not_finite(xk), flag)) {
        zero_quad(xq);
        zero_quad(xk);
        tri_sum<false, true, false>(xq, fp, fk);
        tri_sum<true, true, true>(xk, fp, fq);
    }
    gemm64<false, true>(xe, fa, fk, kChunk, pan);
    gemm64<true, true>(xk, fa, [&](int j, int c) {
        return scaled(*(const float4 *)(kn + j * KP + c), bet[j]);
    }, kChunk, pan);
    gemm64<true, true>(xw, ft, Rows{w.dw + ch * kChunk * KP + x0, KP}, kChunk, pan);
    float *gq = w.gq + ch * kChunk * KP + x0, *gk = w.gk + ch * kChunk * KP + x0;
#pragma unroll
    for (int ti = 0; ti < 2; ti++)
#pragma unroll
        for (int tj = 0; tj < 2; tj++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = (wave >> 1) * 32 + ti * 16 + 4 * (lane >> 4) + r;
                const int64_t at = i * KP + (wave & 1) * 32 + tj * 16 + (lane & 15);
                const float q = qn[at], k = kn[at];
                const float dqv = gq[at] + xq[ti][tj][r];
                const float dkv = gk[at] + xk[ti][tj][r] + xw[ti][tj][r] * bg[i] + xe[ti][tj][r] * bet[i];
                gq[at] = dqv;
                gk[at] = dkv;
                xw[ti][tj][r] *= k;
                xe[ti][tj][r] *= k;
                xq[ti][tj][r] = dqv * q;
                xk[ti][tj][r] = dkv * k;
            }
    row_sums(xw, red[0]);
    row_sums(xe, red[1]);
    row_sums(xq, red[2]);
    row_sums(xk, red[3]);
    __syncthreads();
    {
        const int m = tid >> 6, i = tid & 63;
        pt[(blockIdx.y * 6 + 2 + m) * kChunk + i] = red[m][i] + red[m][kChunk + i];
    }
}

// The gates' gradients from the tiles' row sums, and dq (scaled) and dk through the l2
// normalisation (l2norm_backward :246-252), per (chunk, head).
template <int DT>
__global__ __launch_bounds__(256) void gdr_bwd_finish(GdrArgs a, GdrWs w, void *dq, void *dk, void *dg,
                                                      void *dbeta) {
    const int64_t ch = blockIdx.x, n = ch / a.H, h = ch % a.H, KP = w.KP, VP = w.VP;
    const int len = w.plan.len(n);
    if (len == 0) return;
    const int64_t tok0 = w.plan.tok0(n), Dk = a.Dk;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, kt = (int)(KP / 64), vt = (int)(VP / 64);
    __shared__ float dots[2][kChunk], inv[2][kChunk];
    const float *pt = w.part + ch * w.npart;
    if (wave == 0) {
        const double G = w.G[ch * kChunk + lane], Gl = w.G[ch * kChunk + kChunk - 1];
        const float gam = expf((float)G), lam = expf((float)(Gl - G));
        const float bet = lane < len ? ld_any(a.beta_dt, a.beta, b_at(a, tok0 + lane, h)) : 0.f;
        float sum[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, sv = 0.f, sds = 0.f;
        for (int t = 0; t < kt; t++) {
#pragma unroll
            for (int m = 0; m < 6; m++) sum[m] += pt[(t * 6 + m) * kChunk + lane];
            sds += pt[w.npart - kChunk + t];
        }
        for (int t = 0; t < vt; t++) sv += pt[(kt * 6 + t) * kChunk + lane];
        dots[0][lane] = sum[4];
        dots[1][lane] = sum[5];
        // d_beta = rowsum(d_vb V) + gamma rowsum(d_kbg K) + rowsum(d_kbeta K)
        const float db = sv + sum[2] * gam + sum[3];
        // d_gamma = rowsum(d_qg Q) + beta rowsum(d_kbg K); lam dlam = lam rowsum(d_kt K)
        const float dgam = sum[0] + sum[2] * bet, ldl = sum[1] * lam;
        float d = w.dgv[ch * kChunk + lane] - ldl + dgam * gam;
        const float tail = wave_sum(ldl) + sds * expf((float)Gl);
        if (lane == kChunk - 1) d += tail;
        // g's gradient: the reverse cumulative sum
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const float y = __shfl_down(d, o, 64);
            if (lane + o < 64) d += y;
        }
        if (lane < len) {
            st_any(a.g_dt, dg, (tok0 + lane) * a.H + h, d);
            st_any(a.beta_dt, dbeta, (tok0 + lane) * a.H + h, db);
        }
    } else if (wave < 3) {
        inv[wave - 1][lane] = a.l2norm ? w.inv[ch * 2 * kChunk + (wave - 1) * kChunk + lane] : 1.f;
    }
    __syncthreads();
    // 16 lanes a row
#pragma unroll 2
    for (int it = 0; it < 4; it++) {
        const int i = it * 16 + wave * 4 + (lane >> 4), c0 = 4 * (lane & 15);
        if (i >= len) continue;
        const int64_t tok = tok0 + i, qa = q_at(a, tok, h), ka = k_at(a, tok, h);
        const int64_t at = (ch * kChunk + i) * KP, to = (tok * a.H + h) * Dk;
        const float qi = inv[0][i], ki = inv[1][i], dq_q = dots[0][i], dk_k = dots[1][i];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int x0 = 64 * c + c0;
            if (x0 >= Dk) break;
            const float4 gq = *(const float4 *)(w.gq + at + x0), gk = *(const float4 *)(w.gk + at + x0);
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (x0 + e < Dk) {
                    float yq = at4(gq, e) * a.scale, yk = at4(gk, e);
                    if (a.l2norm) {
                        yq = qi * (yq - ld<DT>(a.q, qa + x0 + e) * qi * dq_q);
                        yk = ki * (yk - ld<DT>(a.k, ka + x0 + e) * ki * dk_k);
                    }
                    st<DT>(dq, to + x0 + e, yq);
                    st<DT>(dk, to + x0 + e, yk);
                }
        }
    }
}

// ------------------------------------------------------------------------------------------
// Host side
// ------------------------------------------------------------------------------------------

int64_t gdr_nseq(const dm_gdr_desc *d) { return d->cu_seqlens ? d->nseq : d->b; }

int64_t gdr_chunk_bound(const dm_gdr_desc *d) {
    if (d->cu_seqlens) return (d->t + (kChunk - 1) * d->nseq) / kChunk;
    return d->b * ((d->t + kChunk - 1) / kChunk);
}

// Carves the workspace; returns the bytes needed (layout identical when `base` is null).
size_t gdr_ws_layout(const dm_gdr_desc *d, bool backward, char *base, GdrWs *w) {
    const int64_t nc = gdr_chunk_bound(d), S = gdr_nseq(d), H = d->h, C = kChunk, ch = nc * H;
    GdrWs x{};
    const int64_t KP = x.KP = (d->dk + 63) / 64 * 64, VP = x.VP = (d->dv + 63) / 64 * 64;
    x.npart = (KP / 64 * 6 + VP / 64 + 1) * C;
    size_t off = 0;
    auto take = [&](size_t bytes) -> char * {
        char *p = base ? base + off : nullptr;
        off += align_up(bytes);
        return p;
    };
    auto rows = [&](int64_t a, int64_t b) { return (float *)take((size_t)(ch * a * b) * 4); };
    x.plan = gdr_plan_layout(d, take);
    x.G = (double *)rows(C, 2);
    x.qn = rows(C, KP);
    x.kn = rows(C, KP);
    x.vp = rows(C, VP);
    x.P = rows(C, C);
    x.W = rows(C, KP);
    x.KT = rows(KP, C);
    x.UT = rows(VP, C);
    // What a launch writes goes where an earlier one's is done with. The forward alone: the states over
    // the rows that prep read (kn and vp follow each other). The state pass: V' over U, each lane reading
    // its values of a chunk before it writes them.
    x.ScT = !backward && VP * KP <= C * (KP + VP) ? x.kn : rows(VP, KP);
    x.VnT = x.UT;
    if (backward) {
        x.inv = rows(2, C);
        x.dop = rows(C, VP);
        x.Tm = rows(C, C);
        x.Am = rows(C, C);
        x.WT = rows(KP, C);
        x.dvlT = rows(VP, C);
        x.F = rows(VP, KP);
        x.dgv = rows(C, 1);
        x.part = rows(x.npart, 1);
        // the reverse state pass as the forward's, and lane by lane too the matrices' gradients; W and
        // (lam K)^T serve the state pass alone, W^T the reverse one (2048 tokens of 8 heads of 128: 190 ->
        // 123 MB)
        x.dVnT = x.dvlT;
        x.dSnT = x.F;
        x.DPd = x.P;
        x.dae = x.Am;
        x.gq = x.W;
        x.gk = x.KT;
        x.dw = x.WT;
    }
    if (w) *w = x;
    return off;
}

bool gdr_strides_ok(const dm_gdr_desc *d, bool step) {
    if (!d->strided) return true;
    const int64_t T = step ? 1 : d->t;
    for (const dm_strides *x : {&d->sq, &d->sk, &d->sv, &d->sg, &d->sbeta, &d->sdo}) {
        if (x->b < 0 || x->t < 0 || x->h < 0) return false;
        if (!step && d->b > 1 && x->b != T * x->t) return false;
    }
    return true;
}

bool gdr_strides_16b(const dm_gdr_desc *d) {
    if (!d->strided) return true;
    for (const dm_strides *x : {&d->sq, &d->sk, &d->sv, &d->sdo})
        if (x->b % 8 || x->t % 8 || x->h % 8) return false;
    return true;
}

GdrArgs gdr_args(const dm_gdr_desc *d, const void *q, const void *k, const void *v,
                 const void *g, const void *beta, bool step) {
    GdrArgs a;
    // contiguous rows unless given: [rows, H, D] and [rows, H]; the step's rows are its batch
    // (t stride = b stride)
    const int64_t H = d->h;
    a.q_t = a.k_t = H * d->dk, a.q_h = a.k_h = d->dk;
    a.v_t = a.o_t = H * d->dv, a.v_h = a.o_h = d->dv;
    a.g_t = a.b_t = H, a.g_h = a.b_h = 1;
    if (d->strided) {
        auto rowst = [&](const dm_strides &x) { return step ? x.b : x.t; };
        a.q_t = rowst(d->sq), a.q_h = d->sq.h;
        a.k_t = rowst(d->sk), a.k_h = d->sk.h;
        a.v_t = rowst(d->sv), a.v_h = d->sv.h;
        a.g_t = rowst(d->sg), a.g_h = d->sg.h;
        a.b_t = rowst(d->sbeta), a.b_h = d->sbeta.h;
        a.o_t = rowst(d->sdo), a.o_h = d->sdo.h;
    }
    a.H = d->h;
    a.rows = d->b * d->t;
    a.Dk = d->dk;
    a.Dv = d->dv;
    a.g_dt = d->g_dtype;
    a.beta_dt = d->beta_dtype;
    a.l2norm = d->qk_l2norm;
    a.scale = d->has_scale ? d->scale : (float)(1.0 / std::sqrt((double)d->dk));
    a.q = q;
    a.k = k;
    a.v = v;
    a.g = g;
    a.beta = beta;
    return a;
}

int launch_plan(const dm_gdr_desc *d, const GdrPlan &p, hipStream_t st) {
    if (p.closed) return DM_OK;
    gdr_plan<<<1, 1024, 0, st>>>(gdr_nseq(d), d->t, gdr_chunk_bound(d), d->cu_seqlens, p);
    DM_LAUNCH_CHECK("chunk_gated_delta_rule: plan");
    return DM_OK;
}

template <bool BWD>
static void launch_chain(const dm_gdr_desc *d, const GdrArgs &a, const GdrWs &w, const float *init,
                         float *final_state, hipStream_t st) {
    const int64_t nsh = gdr_nseq(d) * d->h, nshp = (nsh + 7) / 8 * 8;
    const int nt = nsh * (w.VP / 32) >= 256 ? 2 : 1;
    const unsigned grid = (unsigned)(nshp * (w.VP / (16 * nt)));
#define CHAIN(KTn)                                                                             \
    case KTn:                                                                                  \
        if (nt == 1)                                                                           \
            gdr_chain<KTn, 1, BWD><<<grid, 256, 0, st>>>(a, w, nsh, nshp, init, final_state);  \
        else                                                                                   \
            gdr_chain<KTn, 2, BWD><<<grid, 256, 0, st>>>(a, w, nsh, nshp, init, final_state);  \
        break;
    switch (w.KP / 64) {
        CHAIN(1)
        CHAIN(2)
        CHAIN(3)
        CHAIN(4)
    }
#undef CHAIN
}

}  // namespace dm

using namespace dm;

extern "C" {

size_t dm_gdr_chunk_fwd_workspace(const dm_gdr_desc *d) {
    if (!d) return 0;
    if (gdr_mfma_takes(d)) return gdr_mfma_fwd_workspace(d);
    return gdr_ws_layout(d, false, nullptr, nullptr);
}

int dm_gdr_chunk_fwd(const dm_gdr_desc *d, const void *q, const void *k, const void *v,
                     const void *g, const void *beta, const float *h0, void *out,
                     float *final_state, void *workspace, size_t workspace_bytes, void *stream) {
    int rc = check_gdr(d, "chunk_gated_delta_rule", false);
    if (rc) return rc;
    if (workspace_bytes < dm_gdr_chunk_fwd_workspace(d))
        return refuse("chunk_gated_delta_rule: the workspace is smaller than "
                      "dm_gdr_chunk_fwd_workspace");
    hipStream_t st = (hipStream_t)stream;
    const int64_t S = gdr_nseq(d), nc = gdr_chunk_bound(d);
    if (S * d->h == 0) return DM_OK;
    if (gdr_mfma_takes(d)) {
        for (const void *p : {q, k, v, (const void *)out})
            if (!aligned_16b(p))
                return refuse("chunk_gated_delta_rule: q, k, v and out must be 16-byte aligned "
                              "(16-bit heads that are multiples of 8 wide read and write whole "
                              "rows; the host copies other views)");
        return launch_gdr_mfma_fwd(d, q, k, v, g, beta, h0, out, final_state, workspace, st);
    }
    GdrWs w;
    gdr_ws_layout(d, false, (char *)workspace, &w);
    GdrArgs a = gdr_args(d, q, k, v, g, beta);
    if ((rc = launch_plan(d, w.plan, st))) return rc;
    const unsigned chunks = (unsigned)(nc * d->h);
    const unsigned vt = (unsigned)(w.VP / 64);
#define FWD(DT)                                                                        \
    if (chunks) gdr_prep<DT, false><<<chunks, 256, 0, st>>>(a, w, nullptr);            \
    launch_chain<false>(d, a, w, h0, final_state, st);                                 \
    if (chunks) gdr_output<DT><<<dim3(chunks, vt), 256, 0, st>>>(a, w, out);
    if (d->dtype == DM_F32) {
        FWD(DM_F32)
    } else if (d->dtype == DM_BF16) {
        FWD(DM_BF16)
    } else {
        FWD(DM_F16)
    }
#undef FWD
    probe_add(DM_PROBE_GDR_CHUNK_FWD, !w.plan.closed + (chunks ? 3 : 1));
    DM_LAUNCH_CHECK("chunk_gated_delta_rule: launch");
    return DM_OK;
}

size_t dm_gdr_chunk_bwd_workspace(const dm_gdr_desc *d) {
    if (!d) return 0;
    if (gdr_mfma_takes(d)) return gdr_mfma_bwd_workspace(d);
    return gdr_ws_layout(d, true, nullptr, nullptr);
}

int dm_gdr_chunk_bwd(const dm_gdr_desc *d, const void *q, const void *k, const void *v,
                     const void *g, const void *beta, const float *h0, const void *d_out,
                     const float *d_final, void *dq, void *dk, void *dv, void *dg, void *dbeta,
                     float *dh0, void *workspace, size_t workspace_bytes, void *stream) {
    int rc = check_gdr(d, "chunk_gated_delta_rule_backward", false);
    if (rc) return rc;
    if (workspace_bytes < dm_gdr_chunk_bwd_workspace(d))
        return refuse("chunk_gated_delta_rule_backward: the workspace is smaller than "
                      "dm_gdr_chunk_bwd_workspace");
    hipStream_t st = (hipStream_t)stream;
    const int64_t S = gdr_nseq(d), nc = gdr_chunk_bound(d);
    if (S * d->h == 0) return DM_OK;
    if (gdr_mfma_takes(d)) {
        for (const void *p : {q, k, v, d_out, (const void *)dq, (const void *)dk, (const void *)dv})
            if (!aligned_16b(p))
                return refuse("chunk_gated_delta_rule_backward: q, k, v, d_out, dq, dk and dv "
                              "must be 16-byte aligned (16-bit heads that are multiples of 8 "
                              "wide read and write whole rows; the host copies other views)");
        return launch_gdr_mfma_bwd(d, q, k, v, g, beta, h0, d_out, d_final, dq, dk, dv, dg,
                                   dbeta, dh0, workspace, st);
    }
    GdrWs w;
    gdr_ws_layout(d, true, (char *)workspace, &w);
    GdrArgs a = gdr_args(d, q, k, v, g, beta);
    if ((rc = launch_plan(d, w.plan, st))) return rc;
    const unsigned chunks = (unsigned)(nc * d->h);
    const unsigned kt = (unsigned)(w.KP / 64), vt = (unsigned)(w.VP / 64);
#define BWD(DT)                                                                              \
    if (chunks) gdr_prep<DT, true><<<chunks, 256, 0, st>>>(a, w, d_out);                     \
    launch_chain<false>(d, a, w, h0, nullptr, st);                                           \
    if (chunks) gdr_bwd_local<<<dim3(chunks, vt * (1 + kt)), 256, 0, st>>>(a, w);            \
    launch_chain<true>(d, a, w, d_final, dh0, st);                                           \
    if (chunks) {                                                                            \
        gdr_bwd_states<<<dim3(chunks, kt), 256, 0, st>>>(a, w);                              \
        gdr_bwd_mats<<<chunks, 256, 0, st>>>(a, w);                                          \
        gdr_bwd_rows<DT><<<dim3(chunks, kt + vt), 256, 0, st>>>(a, w, dv);                   \
        gdr_bwd_finish<DT><<<chunks, 256, 0, st>>>(a, w, dq, dk, dg, dbeta);                 \
    }
    if (d->dtype == DM_F32) {
        BWD(DM_F32)
    } else if (d->dtype == DM_BF16) {
        BWD(DM_BF16)
    } else {
        BWD(DM_F16)
    }
#undef BWD
    probe_add(DM_PROBE_GDR_CHUNK_BWD, !w.plan.closed + (chunks ? 8 : 2));
    DM_LAUNCH_CHECK("chunk_gated_delta_rule_backward: launch");
    return DM_OK;
}

}  // extern "C"
