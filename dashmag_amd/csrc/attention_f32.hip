// Attention forward and backward in f32 on the matrix cores (v_mfma_f32_16x16x4_f32): f32 inputs
// of any head width up to 256, and 16-bit inputs of widths the 16-bit MFMA kernels do not take.
// (crates/dash-ops/src/attention/kernels.rs:683-997 computes the same with tiles; the reference,
// reference.rs:305-431, with the scores materialised.)
//
// A workgroup of four wavefronts takes 16 queries of one head (dK and dV: 16 keys of one key-value
// head); its wavefronts take in turn the 16-key (16-query) tiles that any of
// them sees, each on its own, and add up through LDS at the end in a fixed order. Operands go from memory straight into
// registers, a row's 4 consecutive elements a lane where the product's k runs along the head
// (lane l: d = 16 s + 4 (l / 16) + r in product r), one element of 4 rows where it runs along the
// keys; a product's output (lane: 4 rows of one column) is the next one's operand as it stands, so
// nothing passes through LDS inside the loop and there is no barrier in it. Small calls are why
// the keys and not the queries are split over the wavefronts: 256 tokens of 4 heads are 64
// workgroups of 4 tiles a wavefront at most. (With eight wavefronts
// at width 64 that call's kernels took 10.2, 13.1 and 16.0 us against 11.4, 13.3 and 16.8: what is
// left is the chain of a workgroup's first loads, its bounds and the sum at its end.)
//
// At 256 tokens of 4 heads of 64, causal, forward and backward took 410 us as one wavefront a row
// (a dot product, a wavefront reduction and an exponential a key, one after another), and take 48.
#include <string>

#include "attention_kernels.h"
#include "mfma.h"

namespace dm {

// What the dK/dV kernel reads per query row and head: log-sum-exp, delta = rowsum(dO o O), and the
// row's interval of keys (empty where the row sees none).
struct RowRec {
    float lse, delta;
    int32_t lo, hi;
};

struct AttnF32 {
    MaskInfo m;
    int64_t B, Hq, Hkv, D;
    float scale;
    AttnStrides sd;
    const void *q, *k, *v, *o, *d_o;
    const float *lse;
    RowRec *rec;    // [B, Tq, Hq]
    int2 *tile;     // [B, query tiles]: the keys any query of a tile sees
};

constexpr int kQT = 16;  // rows of a tile
constexpr int kNW = 4;   // wavefronts of a workgroup

// Elements 16 s + 4 g + [0, 4) of the row at `off`, zeros past D.
template <int DT, bool VEC, int NS>
__device__ __forceinline__ void row_load(float4 (&f)[NS], const void *p, int64_t off, int D, int g) {
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int d = 16 * s + 4 * g;
        if constexpr (VEC) {
            f[s] = d < D ? *(const float4 *)((const float *)p + off + d) : make_float4(0.f, 0.f, 0.f, 0.f);
        } else {
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; e++) x[e] = d + e < D ? ld<DT>(p, off + d + e) : 0.f;
            f[s] = make_float4(x[0], x[1], x[2], x[3]);
        }
    }
}
// Element 16 s + c of the four rows at `off`, zeros past D.
template <int DT>
__device__ __forceinline__ f32x4_t col_load(const void *p, const int64_t (&off)[4], int d, int D) {
    f32x4_t v;
#pragma unroll
    for (int r = 0; r < 4; r++) v[r] = d < D ? ld<DT>(p, off[r] + d) : 0.f;
    return v;
}

__device__ __forceinline__ float elem(const float4 &v, int r) {
    return r == 0 ? v.x : r == 1 ? v.y : r == 2 ? v.z : v.w;
}

// acc += A[16 x D] B[D x 16], both as row_load leaves them.
template <int NS>
__device__ __forceinline__ f32x4_t rows_dot(const float4 (&a)[NS], const float4 (&b)[NS]) {
    // four sums, one a slot: shorter sums round less, and no product waits on the one before it
    f32x4_t x[4];
#pragma unroll
    for (int r = 0; r < 4; r++) x[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NS; s++)
#pragma unroll
        for (int r = 0; r < 4; r++) x[r] = mfma4(elem(a[s], r), elem(b[s], r), x[r]);
    return (x[0] + x[1]) + (x[2] + x[3]);
}

// What a row does not see must not reach it, whatever it holds (the positions past the last packed
// sequence, a later token), and a product's zero weight does not see to that: 0 * inf is NaN. So of a
// tile of 16 x 16 pairs the terms that no row sees are cleared, as padded ones; and where some rows see a
// term and others don't, values that are not finite are cleared too, and a wavefront that met one goes
// over its tiles again after the loop and adds them to the rows that see them (in the loop that code
// would take the registers of the next tile's loads: 724 bytes a lane spilled at width 256). Tiles of
// seen pairs alone branch past all of it. 1024 causal tokens of 8 heads, forward and backward, without
// any of this and with it: width 64 168 and 167 us, 128 270 and 288, 256 581 and 587.
struct Hidden {
    bool seen[4];  // lane (c, g): whether any row sees term 4 g + r
    bool cut;      // some row (of those that are kept) does not see a term that another sees
    __device__ __forceinline__ Hidden(const bool (&on)[4], bool kept) {
        const int g = (threadIdx.x >> 4) & 3;
        bool part = false;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            seen[r] = ((__ballot(on[r]) >> (16 * g)) & 0xffff) != 0;
            part |= kept && seen[r] && !on[r];
        }
        cut = __any(part);
    }
    // Whether values were cleared that some row sees.
    template <int N>
    __device__ __forceinline__ bool clear(f32x4_t (&x)[N]) const {
#pragma unroll
        for (int s = 0; s < N; s++)
#pragma unroll
            for (int r = 0; r < 4; r++) x[s][r] = seen[r] ? x[s][r] : 0.f;
        if (!cut) return false;
        bool bad = false;
#pragma unroll
        for (int s = 0; s < N; s++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const bool fin = fabsf(x[s][r]) < INFINITY;
                bad |= !fin;
                x[s][r] = fin ? x[s][r] : 0.f;
            }
        return __any(bad);
    }
};
// No pair of the tile is hidden: the terms are taken as they are.
__device__ __forceinline__ bool all_seen(const bool (&on)[4]) { return __all(on[0] && on[1] && on[2] && on[3]); }
// x . y over D elements, in the four lanes (c, 0 .. 3) of a row.
template <int DT>
__device__ __forceinline__ float dot4(const void *x, int64_t xo, const void *y, int64_t yo, int D) {
    float t = 0.f;
    for (int d = (threadIdx.x >> 4) & 3; d < D; d += 4) t += ld<DT>(x, xo + d) * ld<DT>(y, yo + d);
    t += __shfl_xor(t, 16, 64);
    return t + __shfl_xor(t, 32, 64);
}
// acc[s][e] += w * (element 16 s + 4 g + e at `off`) over the elements that are not finite, where the
// lane's row sees them.
template <int DT, int NS>
__device__ __forceinline__ void add_not_finite(f32x4_t (&acc)[NS], const void *p, int64_t off, bool see, float w,
                                               int D) {
    const int g = (threadIdx.x >> 4) & 3;
#pragma unroll
    for (int s = 0; s < NS; s++) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int d = 16 * s + 4 * g + e;
            const float v = see && d < D ? ld<DT>(p, off + d) : 0.f;
            acc[s][e] = fabsf(v) < INFINITY ? acc[s][e] : fmaf(w, v, acc[s][e]);
        }
        __builtin_amdgcn_sched_barrier(0);  // (all the loads at once would take the registers)
    }
}

// The smallest lo and largest hi of a tile's rows (lane c's row in lanes c, c + 16, ...); [0, 0)
// where none sees a key.
__device__ __forceinline__ int2 tile_union(int lo, int hi) {
    int a = hi > lo ? lo : 0x7fffffff, z = hi > lo ? hi : 0;
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) {
        a = min(a, __shfl_xor(a, o, 64));
        z = max(z, __shfl_xor(z, o, 64));
    }
    return make_int2(z ? a : 0, z);
}

__device__ __forceinline__ float across4(float x) {  // the four 16-lane groups' sum
    x += __shfl_xor(x, 16, 64);
    return x + __shfl_xor(x, 32, 64);
}

// (at width 64 held to 128 registers, of 136 taken freely: four workgroups a compute unit)
template <int DT, int DP, bool VEC>
__global__ __launch_bounds__(64 * kNW, DP == 64 ? 4 : 1) void attn_fwd_f32(AttnF32 a, void *o, float *lse) {
    constexpr int NS = DP / 16, OS = DP + 4;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
    const int D = (int)a.D;
    const int64_t Tq = a.m.tq, Tk = a.m.tk, nt = (Tq + kQT - 1) / kQT;
    const unsigned Hq = (unsigned)a.Hq, B = (unsigned)a.B, x = blockIdx.x / Hq;
    const int64_t h = blockIdx.x % Hq, b = x % B, qt = nt - 1 - x / B;  // a causal mask's longest tiles first
    const int64_t i = qt * kQT + c, kh = (unsigned)h / (Hq / (unsigned)a.Hkv);
    __shared__ float4 os4[kNW * kQT * OS / 4];
    __shared__ float ms[kNW][kQT], ls[kNW][kQT];
    float *os = (float *)os4;

    int64_t lo = 0, hi = 0;
    if (i < Tq) row_bounds(a.m, i, &lo, &hi);
    const int2 u = tile_union((int)lo, (int)hi);
    float4 qf[NS], kf[NS];
    const int64_t qo = b * a.sd.q.b + (i < Tq ? i : Tq - 1) * a.sd.q.t + h * a.sd.q.h;
    row_load<DT, VEC>(qf, a.q, qo, D, g);
    const int64_t kb = b * a.sd.k.b + kh * a.sd.k.h, vb = b * a.sd.v.b + kh * a.sd.v.h;
    const uint8_t *pad = a.m.pad ? a.m.pad + b * Tk : nullptr;
    // rows past the union are not read: the last row it holds stands in, and is masked
    auto key = [&](int j) { return j < u.y ? j : u.y - 1; };
    auto sees = [&](int j) { return !(pad && pad[key(j)]) && j >= lo && j < hi; };
    f32x4_t acc[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) acc[s] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float mx = -INFINITY, l = 0.f;
    bool bad = false;
    int j0 = u.x + wave * kQT;
    if (j0 < u.y) row_load<DT, VEC>(kf, a.k, kb + (int64_t)key(j0 + c) * a.sd.k.t, D, g);
    for (; j0 < u.y; j0 += kNW * kQT) {
        int64_t vo[4];
        bool on[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            vo[r] = vb + (int64_t)key(j0 + 4 * g + r) * a.sd.v.t;
            on[r] = sees(j0 + 4 * g + r);
        }
        f32x4_t vf[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) vf[s] = col_load<DT>(a.v, vo, 16 * s + c, D);
        if (!all_seen(on)) bad |= Hidden(on, i < Tq).clear(vf);
        const f32x4_t sv = rows_dot(kf, qf);
        if (j0 + kNW * kQT < u.y)
            row_load<DT, VEC>(kf, a.k, kb + (int64_t)key(j0 + kNW * kQT + c) * a.sd.k.t, D, g);
        float p[4], tm = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            p[r] = on[r] ? sv[r] * a.scale : -INFINITY;
            tm = fmaxf(tm, p[r]);
        }
        tm = fmaxf(tm, __shfl_xor(tm, 16, 64));
        tm = fmaxf(tm, __shfl_xor(tm, 32, 64));
        const float mn = fmaxf(mx, tm), ref = mn == -INFINITY ? 0.f : mn;
        const float alpha = expf(mx - ref);
        mx = mn;
        l *= alpha;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            p[r] = expf(p[r] - ref);
            l += p[r];
        }
        if (__any(alpha != 1.f)) {
#pragma unroll
            for (int s = 0; s < NS; s++) acc[s] *= alpha;
        }
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[s] = mfma4(vf[s][r], p[r], acc[s]);
    }
    if (bad) {
        const float ref = mx == -INFINITY ? 0.f : mx;
        for (j0 = u.x + wave * kQT; j0 < u.y; j0 += kNW * kQT) {
            const int j = j0 + 4 * g;
            const bool on[4] = {sees(j), sees(j + 1), sees(j + 2), sees(j + 3)};
            if (!Hidden(on, i < Tq).cut) continue;
#pragma unroll 1
            for (int x = j0; x < j0 + kQT; x++) {
                const int64_t jx = key(x);
                const float sc = dot4<DT>(a.q, qo, a.k, kb + jx * a.sd.k.t, D);
                add_not_finite<DT>(acc, a.v, vb + jx * a.sd.v.t, sees(x), expf(sc * a.scale - ref), D);
            }
        }
    }
    l = across4(l);
    if (g == 0) {
        ms[wave][c] = mx;
        ls[wave][c] = l;
    }
    __syncthreads();
    auto top = [&](int r) {
        float t = ms[0][r];
#pragma unroll
        for (int w = 1; w < kNW; w++) t = fmaxf(t, ms[w][r]);
        return t == -INFINITY ? 0.f : t;
    };
    const float f = expf(mx - top(c));
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const f32x4_t x = acc[s] * f;
        *(float4 *)(os + (wave * kQT + c) * OS + 16 * s + 4 * g) = make_float4(x[0], x[1], x[2], x[3]);
    }
    __syncthreads();
    // kL lanes a row
    constexpr int kL = 4 * kNW;
    const int r = threadIdx.x / kL, x0 = threadIdx.x % kL;
    if (qt * kQT + r >= Tq) return;
    const int64_t row = (b * Tq + qt * kQT + r) * a.Hq + h;
    float L = 0.f;
#pragma unroll
    for (int w = 0; w < kNW; w++) L += ls[w][r] * expf(ms[w][r] - top(r));
    const float inv = L > 0.f ? 1.f / L : 0.f;
    for (int d = x0; d < D; d += kL) {
        float x = 0.f;
#pragma unroll
        for (int w = 0; w < kNW; w++) x += os[(w * kQT + r) * OS + d];
        st<DT>(o, row * D + d, x * inv);
    }
    if (x0 == 0) lse[row] = L > 0.f ? top(r) + logf(L) : -INFINITY;
}

// dQ = scale sum_j P (dP - delta) K_j, with delta and the rows' records for the dK/dV kernel.
template <int DT, int DP, bool VEC>
__global__ __launch_bounds__(64 * kNW) void attn_dq_f32(AttnF32 a, void *dq) {
    constexpr int NS = DP / 16, OS = DP + 4;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
    const int D = (int)a.D;
    const int64_t Tq = a.m.tq, Tk = a.m.tk, nt = (Tq + kQT - 1) / kQT;
    const unsigned Hq = (unsigned)a.Hq, B = (unsigned)a.B, x = blockIdx.x / Hq;
    const int64_t h = blockIdx.x % Hq, b = x % B, qt = nt - 1 - x / B;
    const int64_t i = qt * kQT + c, ic = i < Tq ? i : Tq - 1, kh = (unsigned)h / (Hq / (unsigned)a.Hkv);
    __shared__ float4 os4[kNW * kQT * OS / 4];
    float *os = (float *)os4;

    int64_t lo = 0, hi = 0;
    if (i < Tq) row_bounds(a.m, i, &lo, &hi);
    int2 u = tile_union((int)lo, (int)hi);
    if (h == 0 && threadIdx.x == 0) a.tile[b * nt + qt] = u;
    float4 qf[NS], gf[NS], kf[NS], vf[NS];
    const int64_t qo = b * a.sd.q.b + ic * a.sd.q.t + h * a.sd.q.h, go = b * a.sd.g.b + ic * a.sd.g.t + h * a.sd.g.h;
    row_load<DT, VEC>(qf, a.q, qo, D, g);
    row_load<DT, VEC>(gf, a.d_o, go, D, g);
    row_load<DT, VEC>(kf, a.o, b * a.sd.o.b + ic * a.sd.o.t + h * a.sd.o.h, D, g);
    const int64_t row = (b * Tq + ic) * a.Hq + h;
    const float ls = a.lse[row];
    float delta = 0.f;
#pragma unroll
    for (int s = 0; s < NS; s++)
#pragma unroll
        for (int r = 0; r < 4; r++) delta += elem(kf[s], r) * elem(gf[s], r);
    delta = across4(delta);
    if (ls == -INFINITY) hi = lo = 0;  // a query that sees no key
    if (wave == 0 && g == 0 && i < Tq) a.rec[row] = RowRec{ls, delta, (int32_t)lo, (int32_t)hi};
    u = tile_union((int)lo, (int)hi);

    const int64_t kb = b * a.sd.k.b + kh * a.sd.k.h, vb = b * a.sd.v.b + kh * a.sd.v.h;
    const uint8_t *pad = a.m.pad ? a.m.pad + b * Tk : nullptr;
    auto key = [&](int j) { return (int64_t)(j < u.y ? j : u.y - 1); };
    auto sees = [&](int j) { return !(pad && pad[key(j)]) && j >= lo && j < hi; };
    auto grad = [&](float s, float dp) { return expf(s * a.scale - ls) * (dp - delta); };
    bool bad = false;
    f32x4_t acc[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) acc[s] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    int j0 = u.x + wave * kQT;
    auto load = [&](int j) {
        row_load<DT, VEC>(kf, a.k, kb + key(j + c) * a.sd.k.t, D, g);
        row_load<DT, VEC>(vf, a.v, vb + key(j + c) * a.sd.v.t, D, g);
    };
    if (j0 < u.y) load(j0);
    for (; j0 < u.y; j0 += kNW * kQT) {
        int64_t ko[4];
        bool on[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            ko[r] = kb + key(j0 + 4 * g + r) * a.sd.k.t;
            on[r] = sees(j0 + 4 * g + r);
        }
        f32x4_t kc[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) kc[s] = col_load<DT>(a.k, ko, 16 * s + c, D);
        if (!all_seen(on)) bad |= Hidden(on, i < Tq).clear(kc);
        const f32x4_t sv = rows_dot(kf, qf), dp = rows_dot(vf, gf);
        if (j0 + kNW * kQT < u.y) load(j0 + kNW * kQT);
        float ds[4];
#pragma unroll
        for (int r = 0; r < 4; r++) ds[r] = on[r] ? grad(sv[r], dp[r]) : 0.f;
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[s] = mfma4(kc[s][r], ds[r], acc[s]);
    }
    if (bad) {
        for (j0 = u.x + wave * kQT; j0 < u.y; j0 += kNW * kQT) {
            const int j = j0 + 4 * g;
            const bool on[4] = {sees(j), sees(j + 1), sees(j + 2), sees(j + 3)};
            if (!Hidden(on, i < Tq).cut) continue;
#pragma unroll 1
            for (int x = j0; x < j0 + kQT; x++) {
                const int64_t k0 = kb + key(x) * a.sd.k.t, v0 = vb + key(x) * a.sd.v.t;
                const float w = grad(dot4<DT>(a.q, qo, a.k, k0, D), dot4<DT>(a.d_o, go, a.v, v0, D));
                add_not_finite<DT>(acc, a.k, k0, sees(x), w, D);
            }
        }
    }
#pragma unroll
    for (int s = 0; s < NS; s++)
        *(float4 *)(os + (wave * kQT + c) * OS + 16 * s + 4 * g) =
            make_float4(acc[s][0], acc[s][1], acc[s][2], acc[s][3]);
    __syncthreads();
    constexpr int kL = 4 * kNW;
    const int r = threadIdx.x / kL;
    if (qt * kQT + r >= Tq) return;
    const int64_t to = ((b * Tq + qt * kQT + r) * a.Hq + h) * D;
    for (int d = threadIdx.x % kL; d < D; d += kL) {
        float x = 0.f;
#pragma unroll
        for (int w = 0; w < kNW; w++) x += os[(w * kQT + r) * OS + d];
        st<DT>(dq, to + d, x * a.scale);
    }
}

// dK = scale sum dS Q and dV = sum P dO over the group's query heads and the queries that see the
// keys: the wavefronts take the (query tile, head) pairs in turn.
template <int DT, int DP, bool VEC>
__global__ __launch_bounds__(64 * kNW) void attn_dkdv_f32(AttnF32 a, void *dk, void *dv) {
    constexpr int NS = DP / 16, OS = DP + 4;
    // at width 256 the operands along the queries are loaded where they are used: held from the
    // step's start they would not fit the registers
    constexpr bool kEarly = DP <= 128;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
    const int D = (int)a.D, group = (int)((unsigned)a.Hq / (unsigned)a.Hkv);
    const int64_t Tq = a.m.tq, Tk = a.m.tk;
    const int nt = (int)((Tq + kQT - 1) / kQT);
    const unsigned Hkv = (unsigned)a.Hkv, B = (unsigned)a.B;
    const int64_t kh = blockIdx.x % Hkv, b = blockIdx.x / Hkv % B, kt = blockIdx.x / Hkv / B;
    const int64_t j = kt * kQT + c, jc = j < Tk ? j : Tk - 1;
    __shared__ float4 os4[kNW * kQT * OS / 4];
    __shared__ int range[2];
    float *os = (float *)os4;

    const bool pad = j >= Tk || (a.m.pad && a.m.pad[b * Tk + jc]);
    // the query tiles that see any of the 16 keys lie in [range[0], range[1]) (none where all are padded)
    if (threadIdx.x == 0) {
        range[0] = nt;
        range[1] = 0;
    }
    __syncthreads();
    for (int t = __all(pad) ? nt : threadIdx.x; t < nt; t += 64 * kNW) {
        const int2 u = a.tile[b * nt + t];
        if (u.x < kt * kQT + kQT && u.y > kt * kQT) {
            atomicMin(&range[0], t);
            atomicMax(&range[1], t + 1);
        }
    }
    float4 kf[NS], vf[NS], qf[NS], gf[NS];
    const int64_t ko = b * a.sd.k.b + jc * a.sd.k.t + kh * a.sd.k.h, vo = b * a.sd.v.b + jc * a.sd.v.t + kh * a.sd.v.h;
    row_load<DT, VEC>(kf, a.k, ko, D, g);
    row_load<DT, VEC>(vf, a.v, vo, D, g);
    f32x4_t ak[NS], av[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) ak[s] = av[s] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    __syncthreads();
    const int t0 = range[0], n = range[1] > t0 ? (range[1] - t0) * group : 0;
    auto q_off = [&](int64_t h, int64_t i) { return b * a.sd.q.b + i * a.sd.q.t + h * a.sd.q.h; };
    auto g_off = [&](int64_t h, int64_t i) { return b * a.sd.g.b + i * a.sd.g.t + h * a.sd.g.h; };
    auto clampq = [&](int64_t i) { return i < Tq ? i : Tq - 1; };
    auto load = [&](int e) {
        const int64_t h = kh * group + e % group, i = clampq((int64_t)(t0 + e / group) * kQT + c);
        row_load<DT, VEC>(qf, a.q, q_off(h, i), D, g);
        row_load<DT, VEC>(gf, a.d_o, g_off(h, i), D, g);
    };
    auto record = [&](int64_t h, int64_t i) {
        RowRec x = a.rec[(b * Tq + clampq(i)) * a.Hq + h];
        if (i >= Tq) x.lo = x.hi = 0;
        return x;
    };
    auto sees = [&](const RowRec &x) { return !pad && j >= x.lo && j < x.hi; };
    bool badq = false, badg = false;
    if (wave < n) load(wave);
    for (int e = wave; e < n; e += kNW) {
        const int64_t h = kh * group + e % group, i0 = (int64_t)(t0 + e / group) * kQT + 4 * g;
        RowRec rec[4];
        int64_t qo[4], go[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int64_t i = clampq(i0 + r);
            rec[r] = record(h, i0 + r);
            qo[r] = q_off(h, i);
            go[r] = g_off(h, i);
        }
        f32x4_t qc[kEarly ? NS : 1], gc[kEarly ? NS : 1];
        if constexpr (kEarly) {
#pragma unroll
            for (int s = 0; s < NS; s++) {
                qc[s] = col_load<DT>(a.q, qo, 16 * s + c, D);
                gc[s] = col_load<DT>(a.d_o, go, 16 * s + c, D);
            }
        }
        bool on[4];
#pragma unroll
        for (int r = 0; r < 4; r++) on[r] = sees(rec[r]);
        const bool all = all_seen(on);
        if constexpr (kEarly) {
            if (!all) {
                const Hidden hid(on, !pad);
                badq |= hid.clear(qc);
                badg |= hid.clear(gc);
            }
        }
        const f32x4_t sv = rows_dot(qf, kf), dp = rows_dot(gf, vf);
        if (e + kNW < n) load(e + kNW);
        float p[4], ds[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            p[r] = on[r] ? expf(sv[r] * a.scale - rec[r].lse) : 0.f;
            ds[r] = on[r] ? p[r] * (dp[r] - rec[r].delta) : 0.f;
        }
#pragma unroll
        for (int s = 0; s < NS; s++) {
            f32x4_t x[1], y[1];
            if constexpr (kEarly) {
                x[0] = qc[s];
                y[0] = gc[s];
            } else {
                x[0] = col_load<DT>(a.q, qo, 16 * s + c, D);
                y[0] = col_load<DT>(a.d_o, go, 16 * s + c, D);
                if (!all) {
                    const Hidden hid(on, !pad);
                    badq |= hid.clear(x);
                    badg |= hid.clear(y);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                ak[s] = mfma4(x[0][r], ds[r], ak[s]);
                av[s] = mfma4(y[0][r], p[r], av[s]);
            }
        }
    }
    auto again = [&](f32x4_t (&acc)[NS], const void *which, auto own, auto weight) {
        for (int e = wave; e < n; e += kNW) {
            const int64_t h = kh * group + e % group, i0 = (int64_t)(t0 + e / group) * kQT;
            bool on[4];
#pragma unroll
            for (int r = 0; r < 4; r++) on[r] = sees(record(h, i0 + 4 * g + r));
            if (!Hidden(on, !pad).cut) continue;
#pragma unroll 1
            for (int64_t i = i0; i < i0 + kQT; i++) {
                const RowRec x = record(h, i);
                const int64_t q0 = q_off(h, clampq(i)), g0 = g_off(h, clampq(i));
                const float p = expf(dot4<DT>(a.q, q0, a.k, ko, D) * a.scale - x.lse);
                add_not_finite<DT>(acc, which, own(q0, g0), sees(x), weight(p, x.delta, g0), D);
            }
        }
    };
    if (badq)
        again(ak, a.q, [](int64_t q0, int64_t) { return q0; },
              [&](float p, float delta, int64_t g0) { return p * (dot4<DT>(a.d_o, g0, a.v, vo, D) - delta); });
    if (badg) again(av, a.d_o, [](int64_t, int64_t g0) { return g0; }, [](float p, float, int64_t) { return p; });
    constexpr int kL = 4 * kNW;
    const int r = threadIdx.x / kL;
    const int64_t to = ((b * Tk + kt * kQT + r) * a.Hkv + kh) * D;
    auto give = [&](const f32x4_t (&x)[NS], void *out, float f) {
        __syncthreads();
        // (a padded key sees nothing, and its column may hold 0 * NaN: its terms were not looked at)
#pragma unroll
        for (int s = 0; s < NS; s++)
            *(float4 *)(os + (wave * kQT + c) * OS + 16 * s + 4 * g) =
                pad ? make_float4(0.f, 0.f, 0.f, 0.f) : make_float4(x[s][0], x[s][1], x[s][2], x[s][3]);
        __syncthreads();
        if (kt * kQT + r >= Tk) return;
        for (int d = threadIdx.x % kL; d < D; d += kL) {
            float y = 0.f;
#pragma unroll
            for (int w = 0; w < kNW; w++) y += os[(w * kQT + r) * OS + d];
            st<DT>(out, to + d, y * f);
        }
    };
    give(ak, dk, a.scale);
    give(av, dv, 1.f);
}

// ------------------------------------------------------------------------------------------
// Host side
// ------------------------------------------------------------------------------------------

// Rows as 16-byte loads: f32, every stride and the width a multiple of 4 elements, bases aligned.
static bool f32_rows_16b(const dm_attention_desc *d, const AttnStrides &s, const void *q, const void *k,
                         const void *v, const void *o, const void *d_o) {
    auto ok = [](const Strd &x) { return x.b % 4 == 0 && x.t % 4 == 0 && x.h % 4 == 0; };
    return d->dtype == DM_F32 && d->d % 4 == 0 && ok(s.q) && ok(s.k) && ok(s.v) && aligned_16b(q) &&
           aligned_16b(k) && aligned_16b(v) && (!d_o || (ok(s.o) && ok(s.g) && aligned_16b(o) && aligned_16b(d_o)));
}

template <class F>
static void by_dtype_width(const dm_attention_desc *d, bool vec, F f) {
    auto width = [&](auto dt, auto v) {
        if (d->d <= 64)
            f(dt, std::integral_constant<int, 64>{}, v);
        else if (d->d <= 128)
            f(dt, std::integral_constant<int, 128>{}, v);
        else
            f(dt, std::integral_constant<int, 256>{}, v);
    };
    if (d->dtype == DM_F32 && vec)
        width(std::integral_constant<int, DM_F32>{}, std::true_type{});
    else if (d->dtype == DM_F32)
        width(std::integral_constant<int, DM_F32>{}, std::false_type{});
    else if (d->dtype == DM_BF16)
        width(std::integral_constant<int, DM_BF16>{}, std::false_type{});
    else
        width(std::integral_constant<int, DM_F16>{}, std::false_type{});
}

int launch_attn_fwd_f32(const MaskInfo &m, const dm_attention_desc *d, float scale, const void *q,
                        const void *k, const void *v, void *o, float *lse, hipStream_t st) {
    const int64_t items = (d->tq + kQT - 1) / kQT * d->b * d->hq;
    if (items == 0) return DM_OK;
    const AttnF32 a{m, d->b, d->hq, d->hkv, d->d, scale, attn_strides(d), q, k, v, nullptr, nullptr, nullptr,
                    nullptr, nullptr};
    by_dtype_width(d, f32_rows_16b(d, a.sd, q, k, v, nullptr, nullptr), [&](auto dt, auto w, auto vec) {
        attn_fwd_f32<dt(), w(), vec()><<<(unsigned)items, 64 * kNW, 0, st>>>(a, o, lse);
    });
    probe_add(DM_PROBE_ATTN_FWD_GENERIC);
    DM_LAUNCH_CHECK("attention: forward launch");
    return DM_OK;
}

size_t attn_bwd_f32_workspace(const dm_attention_desc *d) {
    return align_up((size_t)(d->b * d->tq * d->hq) * sizeof(RowRec)) +
           align_up((size_t)(d->b * ((d->tq + kQT - 1) / kQT)) * sizeof(int2));
}

int launch_attn_bwd_f32(const MaskInfo &m, const dm_attention_desc *d, float scale, const void *q,
                        const void *k, const void *v, const void *o, const float *lse, const void *d_o,
                        void *dq, void *dk, void *dv, void *workspace, hipStream_t st) {
    const int64_t qi = (d->tq + kQT - 1) / kQT * d->b * d->hq, ki = (d->tk + kQT - 1) / kQT * d->b * d->hkv;
    char *ws = (char *)workspace;
    const AttnF32 a{m, d->b, d->hq, d->hkv, d->d, scale, attn_strides(d), q, k, v, o, d_o, lse, (RowRec *)ws,
                    (int2 *)(ws + align_up((size_t)(d->b * d->tq * d->hq) * sizeof(RowRec)))};
    by_dtype_width(d, f32_rows_16b(d, a.sd, q, k, v, o, d_o), [&](auto dt, auto w, auto vec) {
        attn_dq_f32<dt(), w(), vec()><<<(unsigned)qi, 64 * kNW, 0, st>>>(a, dq);
        attn_dkdv_f32<dt(), w(), vec()><<<(unsigned)ki, 64 * kNW, 0, st>>>(a, dk, dv);
    });
    probe_add(DM_PROBE_ATTN_BWD_GENERIC, 2);
    DM_LAUNCH_CHECK("attention_backward: launch");
    return DM_OK;
}

}  // namespace dm
