// ssa_grad.hip -- gradients of the gather attention (gfx950).
//
// Backward of sparse_gather_attention (autograd through
// sparse_attention.py:1096-1199).  A query row touches K key rows, so dK and
// dV are sums over the transposed graph.  Adding them slot by slot takes
// 2 K d read-modify-writes of memory per query row (at 131,072 rows of 128
// slots, d = 128, 8 kv heads of 4,096 keys: 4.3e9 fp32 atomics, 100 ms).  Here
// the graph is transposed instead, and every key row is summed by one wavefront
// in registers (times of that shape in bf16 behind each kernel; 1.33 ms in all):
//
//   1. grad_count_kernel   counts the slots of each key row per block of query
//                          rows in LDS; the count before a slot is its rank
//                          (47 us)
//   2. grad_chunk_kernel,  prefixes over the blocks and over the key rows: the
//      grad_list_kernel,   place of every slot in its key row's list, and the
//      grad_segs_kernel    lists cut into segments of at most `seg` entries
//                          (15 + 10 + 5 us)
//   3. grad_rows_kernel    per query row: scores and dO.V, the softmax, dQ;
//                          each slot's two weights go to its place in the list
//                          (756 us)
//   4. grad_keys_kernel    per segment: dK = sum draw q, dV = sum p' dO (473 us)
//   5. grad_join_kernel    key rows of several segments: sum of their partials
//                          (21 us)
//
// Numerics: scores, dO.V, softmax, weights and sums in fp32 (16-bit products are
// exact in fp32).  Scores, and dO.V where dout has q's type, are 16-bit rows' pairs
// by v_dot2, as in the forward; dO.V with an fp32 dout, fp32 rows and rows beyond
// LDS are chains of fp32 FMAs.  Deterministic mode: the order of a list's
// entries varies between runs, so its sums are made independent of the order:
// each term (exact in fp64) is rounded to a grid of its key row coarse enough
// that every partial sum is exact in fp64, and what the rounding left to a
// second, finer grid in a second sum, which keeps the bits of terms far below
// the key row's largest (one huge element of a row that names the key).
#include <algorithm>

#include "ssa_apply_dev.h"

namespace {

// One segment of a key row's list.  part < 0: the row's only one.
struct GradSeg {
    int64_t begin;         // first entry (of the chunk's entries)
    int32_t len;
    int32_t key;           // key row within its group
    int32_t part;
    int32_t pad;
};

struct GradP {
    ApplyP a;              // the forward's operands
    const void *dout;
    int64_t dosb, dosh, dosn;
    void *dq, *dk, *dv;
    int64_t dqsb, dqsh, dqsn, dksb, dksh, dksn, dvsb, dvsh, dvsn;
    int32_t out32;         // gradients are fp32 (else q's type)
    int32_t accumulate;    // dk, dv are added to (fp32 only)
    int32_t shift;         // entries hold row offsets in units of 1 << shift elements; -1: rows
    // groups (b, kv head) of this launch: [g0, g0 + ng), with all their query rows,
    // or one group's rows from r0 on (a part: the first, the last, or between)
    int32_t g0, ng;
    int32_t first, last;
    int64_t r0, row0;      // first row within its group, and of all
    int64_t grows, gslots; // rows and slots of each group in this launch
    // blocks of `crows` query rows, nc of them per group
    int32_t crows, nc;
    int32_t seg;           // entries per segment
    int64_t segcap, partcap;
    // workspace
    uint4 *ent;            // (ng * gslots) {q offset, dO offset, draw, p'} ({row, -, ..})
    uint32_t *rank;        // (ng * gslots)
    uint32_t *tab;         // (ng, nc, M) slots before this block
    int64_t *kbegin;       // (ng, M)
    uint32_t *klen;        // (ng, M)
    int32_t *kfirst;       // (ng, M) first segment
    int2 *kpart;           // (ng, M) first partial, partials (0: none)
    uint32_t *bnd;         // (ng * gslots) each entry's term bounds, as row_bound packs them (deterministic)
    uint32_t *wmax;        // (ng, M, 2) the largest of a key row's dK and dV bounds (deterministic)
    uint8_t *poison;       // (ng, M) 1: dK is NaN, 2: dV is NaN
    void *acc;             // (M, 2, d) sums of a group's parts so far, float or double
    GradSeg *segs;         // (ng, segcap)
    int32_t *nseg;         // (ng)
    void *part;            // (ng * partcap, 2, d) float, or (.., 4, d) double when deterministic
};

// Workgroup of a launch: grids of more than GRID_X workgroups continue in y (the
// runtime takes fewer than 2^32 threads in x).
constexpr int64_t GRID_X = (int64_t)1 << 20;
__device__ __forceinline__ int64_t launch_block() { return (int64_t)blockIdx.y * gridDim.x + blockIdx.x; }
dim3 launch_grid(int64_t blocks) {
    return blocks <= GRID_X ? dim3((unsigned)blocks) : dim3((unsigned)GRID_X, (unsigned)ceil_div(blocks, GRID_X));
}

constexpr int CNT_THREADS = 1024;
constexpr int CNT_KEYS = 16384;        // key rows counted at a time: 64 KB of LDS
constexpr int GRAD_KLDS = 3072;        // slots a row's 12 B per slot of LDS hold (4 rows a block)

// id of slot s: >= 0 a key the row attends to; else masked or out of range
__device__ __forceinline__ int slot_key(const ApplyP &p, int64_t s) {
    const int64_t x = p.nb32 ? (int64_t)p.nb32[s] : p.nb[s];
    const bool ok = p.nb32 || !p.valid || p.valid[s] != 0;
    return (ok && x >= 0 && x < p.M) ? (int)x : -1;
}

// ---------------------------------------------------------------- 1. counts
// One workgroup per block of query rows.  Bound: the graph's bytes and one LDS
// atomic per slot (a row's keys differ, so a wave's 64 atomics rarely meet).
__global__ void __launch_bounds__(CNT_THREADS) grad_count_kernel(GradP p) {
    extern __shared__ uint32_t cnt[];
    const int64_t blk = launch_block();
    const int c = (int)(blk % p.nc), gl = (int)(blk / p.nc);
    if (gl >= p.ng) return;
    const int64_t r0 = (int64_t)c * p.crows;
    const int64_t r1 = r0 + p.crows < p.grows ? r0 + p.crows : p.grows;
    const int64_t s0 = ((int64_t)gl * p.grows + r0) * p.a.K, s1 = ((int64_t)gl * p.grows + r1) * p.a.K;
    const int64_t base = p.row0 * p.a.K;                // the graph's first slot of this launch
    for (int k0 = 0; k0 < p.a.M; k0 += CNT_KEYS) {
        const int nk = p.a.M - k0 < CNT_KEYS ? p.a.M - k0 : CNT_KEYS;
        for (int i = threadIdx.x; i < nk; i += CNT_THREADS) cnt[i] = 0u;
        __syncthreads();
        for (int64_t s = s0 + threadIdx.x; s < s1; s += CNT_THREADS) {
            const int x = slot_key(p.a, base + s) - k0;
            if (x >= 0 && x < nk) p.rank[s] = atomicAdd(&cnt[x], 1u);
        }
        __syncthreads();
        uint32_t *t = p.tab + ((int64_t)gl * p.nc + c) * p.a.M + k0;
        for (int i = threadIdx.x; i < nk; i += CNT_THREADS) t[i] = cnt[i];
        __syncthreads();
    }
}

// ---------------------------------------------------------------- 2. places
// thread per (group, key row): prefix over the group's blocks
__global__ void __launch_bounds__(256) grad_chunk_kernel(GradP p) {
    const int64_t i = launch_block() * 256 + threadIdx.x;
    if (i >= (int64_t)p.ng * p.a.M) return;
    const int64_t gl = i / p.a.M, x = i % p.a.M;
    uint32_t *t = p.tab + gl * p.nc * p.a.M + x;
    uint32_t sum = 0;
    constexpr int U = 8;
    for (int c0 = 0; c0 < p.nc; c0 += U) {
        uint32_t v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = t[(int64_t)(c0 + u < p.nc ? c0 + u : p.nc - 1) * p.a.M];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (c0 + u < p.nc) {
                t[(int64_t)(c0 + u) * p.a.M] = sum;
                sum += v[u];
            }
        }
    }
    p.klen[i] = sum;
    p.poison[i] = 0;
    if (p.wmax) p.wmax[2 * i] = p.wmax[2 * i + 1] = 0u;
}

template <typename V>
__device__ __forceinline__ V wave_scan_incl(V v, int lane) {
#pragma unroll
    for (int o = 1; o < SSA_WAVE; o <<= 1) {
        const V u = __shfl_up(v, o, SSA_WAVE);
        if (lane >= o) v += u;
    }
    return v;
}

// One workgroup per group: where each key row's list, segments and partials
// start.  A thread sums LIST_KEYS consecutive key rows, so a group of up to
// 8,192 takes one round of scans.
constexpr int LIST_KEYS = 8;
__global__ void __launch_bounds__(1024) grad_list_kernel(GradP p) {
    __shared__ int64_t wl[16];
    __shared__ int32_t ws[16], wp[16];
    const int gl = (int)launch_block(), tid = threadIdx.x, lane = lane_id(), wid = tid / SSA_WAVE;
    if (gl >= p.ng) return;
    int64_t cl = (int64_t)gl * p.gslots;        // entries before this tile
    int32_t cs = 0, cp = 0;                     // segments, partials before it
    for (int k0 = 0; k0 < p.a.M; k0 += 1024 * LIST_KEYS) {
        const int x0 = k0 + tid * LIST_KEYS;
        const int64_t i0 = (int64_t)gl * p.a.M + x0;
        uint32_t len[LIST_KEYS];
        int64_t tl = 0;
        int ts = 0, tp = 0;
#pragma unroll
        for (int u = 0; u < LIST_KEYS; ++u) len[u] = x0 + u < p.a.M ? p.klen[i0 + u] : 0u;
#pragma unroll
        for (int u = 0; u < LIST_KEYS; ++u) {
            const int ns = x0 + u < p.a.M ? (len[u] ? (int)((len[u] + p.seg - 1) / p.seg) : 1) : 0;
            tl += len[u];
            ts += ns;
            tp += ns > 1 ? ns : 0;
        }
        const int64_t il = wave_scan_incl<int64_t>(tl, lane);
        const int is = wave_scan_incl<int>(ts, lane), ip = wave_scan_incl<int>(tp, lane);
        if (lane == SSA_WAVE - 1) { wl[wid] = il; ws[wid] = is; wp[wid] = ip; }
        __syncthreads();
        int64_t bl = cl + il - tl, al = 0;
        int bs = cs + is - ts, as = 0, bp = cp + ip - tp, ap = 0;
        for (int w = 0; w < 16; ++w) {
            if (w < wid) { bl += wl[w]; bs += ws[w]; bp += wp[w]; }
            al += wl[w]; as += ws[w]; ap += wp[w];
        }
#pragma unroll
        for (int u = 0; u < LIST_KEYS; ++u) {
            if (x0 + u < p.a.M) {
                const int ns = len[u] ? (int)((len[u] + p.seg - 1) / p.seg) : 1;
                const int np = ns > 1 ? ns : 0;
                p.kbegin[i0 + u] = bl;
                p.kfirst[i0 + u] = bs;
                p.kpart[i0 + u] = make_int2(np ? (int)((int64_t)gl * p.partcap) + bp : -1, np);
                bl += len[u]; bs += ns; bp += np;
            }
        }
        cl += al; cs += as; cp += ap;
        __syncthreads();
    }
    if (tid == 0) p.nseg[gl] = cs;
}

// thread per (group, key row): its segments
__global__ void __launch_bounds__(256) grad_segs_kernel(GradP p) {
    const int64_t i = launch_block() * 256 + threadIdx.x;
    if (i >= (int64_t)p.ng * p.a.M) return;
    const int64_t gl = i / p.a.M;
    const uint32_t len = p.klen[i];
    const int2 kp = p.kpart[i];
    const int ns = kp.y ? kp.y : 1;
    const int64_t begin = p.kbegin[i];
    GradSeg *out = p.segs + gl * p.segcap + p.kfirst[i];
    for (int s = 0; s < ns; ++s) {
        GradSeg d;
        d.begin = begin + (int64_t)s * p.seg;
        const int64_t left = (int64_t)len - (int64_t)s * p.seg;
        d.len = (int)(left < p.seg ? left : p.seg);
        d.key = (int)(i - gl * p.a.M);
        d.part = kp.y ? kp.x + s : -1;
        d.pad = 0;
        out[s] = d;
    }
}

// ---------------------------------------------------------------- 3. query rows
// A lane's VEC elements of a row as loaded
template <typename T, int VEC> struct Raw { T e[VEC]; };

template <typename T, int VEC>
__device__ __forceinline__ Raw<T, VEC> load_raw(const T *p) {
    Raw<T, VEC> r;
    constexpr int BYTES = (int)sizeof(T) * VEC;
    if constexpr (BYTES % 16 == 0) {
#pragma unroll
        for (int i = 0; i < BYTES / 16; ++i) {
            const uint4 u = reinterpret_cast<const uint4 *>(p)[i];
            __builtin_memcpy(reinterpret_cast<char *>(&r) + 16 * i, &u, 16);
        }
    } else {
        const uint2 u = *reinterpret_cast<const uint2 *>(p);
        __builtin_memcpy(&r, &u, 8);
    }
    return r;
}

// dot product of a lane's elements: 16-bit pairs by v_dot2 (exact products,
// fp32 accumulate), else fp32 FMAs
template <typename T, typename TD, int VEC>
__device__ __forceinline__ float dot_raw(const Raw<TD, VEC> &a, const Raw<T, VEC> &b) {
    float s = 0.f;
    if constexpr (sizeof(T) == 2 && std::is_same<T, TD>::value) {
        uint32_t x[VEC / 2], y[VEC / 2];
        __builtin_memcpy(x, &a, sizeof(x));
        __builtin_memcpy(y, &b, sizeof(y));
#pragma unroll
        for (int i = 0; i < VEC / 2; ++i) s = Dot2<T>::dot(x[i], y[i], s);
    } else {
#pragma unroll
        for (int e = 0; e < VEC; ++e) s = fmaf(to_f32(a.e[e]), to_f32(b.e[e]), s);
    }
    return s;
}

// rows of a lane group in flight: as many as the butterfly of the group takes
// (8 rows over 16 lanes, 4 over 8), fewer for wide vectors
template <typename T, int D> constexpr int grad_u() {
    constexpr int LPR = Geo<T, D>::LPR, VEC = Geo<T, D>::VEC;
    return VEC > 8 || (VEC == 8 && sizeof(T) == 4) ? 2 : (LPR == 16 ? 8 : 4);
}

template <typename T> struct Bits16 {
    static __device__ __forceinline__ uint32_t of(float v) { return Dot2<T>::bits(v); }
};
template <> struct Bits16<float> {
    static __device__ __forceinline__ uint32_t of(float) { return 0u; }      // not reached
};

// VEC consecutive gradients: 16-byte stores (fp32, or packed 16-bit)
template <typename T, int VEC>
__device__ __forceinline__ void store_vec(void *base, int64_t at, const float (&v)[VEC], bool f32) {
    if (f32 || sizeof(T) == 4) {
        float *o = (float *)base + at;
#pragma unroll
        for (int e = 0; e < VEC; e += 4)
            *reinterpret_cast<float4 *>(o + e) = make_float4(v[e], v[e + 1], v[e + 2], v[e + 3]);
    } else {
        T *o = (T *)base + at;
        uint32_t w[VEC / 2];
#pragma unroll
        for (int e = 0; e < VEC; e += 2) w[e / 2] = Bits16<T>::of(v[e]) | (Bits16<T>::of(v[e + 1]) << 16);
        if constexpr (VEC == 4) {
            *reinterpret_cast<uint2 *>(o) = make_uint2(w[0], w[1]);
        } else {
#pragma unroll
            for (int e = 0; e < VEC / 2; e += 4)
                *reinterpret_cast<uint4 *>(o + 2 * e) = make_uint4(w[e], w[e + 1], w[e + 2], w[e + 3]);
        }
    }
}

template <typename T>
__device__ __forceinline__ void store_grad(void *base, int64_t at, float v, bool f32) {
    if (f32) ((float *)base)[at] = v;
    else Cvt<T>::store((T *)base + at, v);
}

// Deterministic mode: at least |w| x xm, xm the largest finite or infinite |x| of
// the row that w weighs, as a bf16 pattern (0: the term is 0; NaN above infinity).
// A NaN element of x is in no bound: its term carries it.
__device__ __forceinline__ uint32_t row_bound(float w, float xm) {
    const float b = fabsf(w) * xm;
    if (b != b) return w == 0.f ? 0u : 0x7fffu;
    if (w == 0.f || xm == 0.f) return 0u;
    const uint32_t up = (__float_as_uint(fmaxf(b, 1.17549435e-38f)) + 0xffffu) >> 16;
    return b == INFINITY ? up : min(up, 0x7f7fu);     // rounded down at the top: grid_magic doubles it
}

// largest |x| over a row's lanes, NaN left out
template <typename T, int VEC>
__device__ __forceinline__ float row_absmax(const T (&x)[VEC]) {
    float m = 0.f;
#pragma unroll
    for (int e = 0; e < VEC; ++e) m = fmaxf(m, fabsf(to_f32(x[e])));
    return wave_max(m);
}

// What a row's slots leave for their key rows: per slot the weights of q (draw)
// and of dO (p') at the slot's place in the key's list.  A masked slot has no
// place; its weights are 0, or NaN in a row without a finite softmax, which
// then reach the id the graph holds there.
struct RowOut {
    const int64_t *kbegin;     // the group's
    const uint32_t *tab;       // the group's and block's
    const uint32_t *rank;      // the row's
    int64_t ki;                // the group's first key row
    int64_t slot;              // the row's first slot in the graph
    uint32_t qoff, dooff;
    float qm = 0.f, dm = 0.f;  // deterministic: the row's largest |q| and |dO|
    __device__ __forceinline__ RowOut(const GradP &p, int64_t row, int gl, int hl, int n) {
        const int64_t lrow = row - p.row0;
        const int c = (int)((lrow - (int64_t)gl * p.grows) / p.crows);
        ki = (int64_t)gl * p.a.M;
        kbegin = p.kbegin + ki;
        tab = p.tab + ((int64_t)gl * p.nc + c) * p.a.M;
        rank = p.rank + lrow * p.a.K;
        slot = row * p.a.K;
        if (p.shift >= 0) {
            qoff = (uint32_t)(((int64_t)hl * p.a.qsh + (int64_t)n * p.a.qsn) >> p.shift);
            dooff = (uint32_t)(((int64_t)hl * p.dosh + (int64_t)n * p.dosn) >> p.shift);
        } else {
            qoff = (uint32_t)(lrow - (int64_t)gl * p.grows);
            dooff = 0u;
        }
    }
    __device__ __forceinline__ void put(const GradP &p, int x, int j, float draw, float pw) const {
        if (x >= 0) {
            const int64_t at = kbegin[x] + tab[x] + rank[j];
            p.ent[at] = make_uint4(qoff, dooff, __float_as_uint(draw), __float_as_uint(pw));
            if (p.bnd) p.bnd[at] = (row_bound(draw, qm) << 16) | row_bound(pw, dm);
        } else if (draw != draw || pw != pw) {
            const int64_t y = p.a.nb32 ? (int64_t)p.a.nb32[slot + j] : p.a.nb[slot + j];
            if (y >= 0 && y < p.a.M) {
                const uint32_t f = (draw != draw ? 1u : 0u) | (pw != pw ? 2u : 0u);
                const int64_t at = ki + y;
                atomicOr((uint32_t *)(p.poison + (at & ~(int64_t)3)), f << (8 * (int)(at & 3)));
            }
        }
    }
};

// A slot in LDS: the key id it attends to, or negative: masked (its id, whose row
// is read and weighed 0 as autograd does), or no key at all (padding up to a
// whole step, an id out of range), which takes nothing, whatever key row 0, read
// in its place, holds.  OFF32 (ids below 2^24): the row is the low 24 bits, so
// the address takes no step of its own.
template <bool OFF32> struct SlotId {
    static constexpr int32_t NONE = OFF32 ? (int32_t)0xc0000000 : INT32_MIN;
    static __device__ __forceinline__ int32_t masked(int32_t y) { return OFF32 ? (y | INT32_MIN) : ~y; }
    // the row read for a slot (not OFF32)
    static __device__ __forceinline__ int32_t row(int32_t x) { return x >= 0 ? x : x == NONE ? 0 : ~x; }
};

// One wavefront per query row, as in the forward: ids in LDS, K and V rows
// gathered together for the scores and dO.V, the softmax per slot, then the K
// rows again for dQ.  Bound: the gathers' L2 delivery (3 rows of d per slot
// against the forward's 2: 12.9 GB in 756 us, 17.0 TB/s) and the VALU work of
// the products.
template <typename T, typename TD, int D, int U, bool OFF32>
__global__ void __launch_bounds__(WAVES * SSA_WAVE)
grad_rows_kernel(GradP gp) {
    using G = Geo<T, D>;
    constexpr int VEC = G::VEC, LPR = G::LPR, RPI = G::RPI, STEP = RPI * U;
    const ApplyP &p = gp.a;
    extern __shared__ float smem[];
    const int64_t nblocks = ceil_div((int64_t)gp.ng * gp.grows, WAVES);
    const int64_t blk = xcd_logical_block(launch_block(), nblocks);
    if (blk >= nblocks) return;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / SSA_WAVE);
    const int64_t lrow = blk * WAVES + wid;
    if (lrow >= (int64_t)gp.ng * gp.grows) return;
    const int64_t row = gp.row0 + lrow;
    const int gl = (int)(lrow / gp.grows);
    const int lane = lane_id();
    const int sub = lane / LPR, li = lane % LPR;
    const int Kp = (p.K + STEP - 1) / STEP * STEP;
    using S = SlotId<OFF32>;
    int32_t *ix = reinterpret_cast<int32_t *>(smem) + (int64_t)wid * 3 * Kp;
    float *sc = reinterpret_cast<float *>(ix + Kp);      // scores, p, then draw
    float *dpv = sc + Kp;                                // dO.V per slot

    const int n = (int)(row % p.N);
    const int64_t bh = row / p.N;
    const int h = (int)(bh % p.Hq);
    const int b = (int)(bh / p.Hq);
    const int g = h / p.rep;
    const T *qrow = (const T *)p.q + b * p.qsb + h * p.qsh + (int64_t)n * p.qsn;
    const TD *dorow = (const TD *)gp.dout + b * gp.dosb + h * gp.dosh + (int64_t)n * gp.dosn;
    const T *kb = (const T *)p.k + b * p.ksb + g * p.ksh;
    const T *vb = (const T *)p.v + b * p.vsb + g * p.vsh;
    const int64_t *nb = p.nb ? p.nb + row * p.K : nullptr;
    const uint8_t *va = p.valid ? p.valid + row * p.K : nullptr;
    // lanes whose elements lie past the head dim hold zeros and store nothing
    const bool live = li * VEC < p.d;
    const int lofs = live ? li * VEC : 0;
    Raw<T, VEC> qr = load_raw<T, VEC>(qrow + lofs);
    Raw<TD, VEC> dr = load_raw<TD, VEC>(dorow + lofs);
    const uint32_t krb = (uint32_t)(p.ksn * (int64_t)sizeof(T)), vrb = (uint32_t)(p.vsn * (int64_t)sizeof(T));
    auto krow = [&](int x) __attribute__((always_inline)) {
        if constexpr (OFF32)
            return reinterpret_cast<const T *>((const char *)kb + (__umul24((uint32_t)x, krb) +
                                                                  (uint32_t)lofs * (uint32_t)sizeof(T)));
        else return kb + (int64_t)S::row(x) * p.ksn + lofs;
    };
    auto vrow = [&](int x) __attribute__((always_inline)) {
        if constexpr (OFF32)
            return reinterpret_cast<const T *>((const char *)vb + (__umul24((uint32_t)x, vrb) +
                                                                  (uint32_t)lofs * (uint32_t)sizeof(T)));
        else return vb + (int64_t)S::row(x) * p.vsn + lofs;
    };

    auto slots = [&](auto i32) __attribute__((always_inline)) {
        for (int j0 = 0; j0 < Kp; j0 += APPLY_SLOT_BATCH * SSA_WAVE) {
            RowSlots<APPLY_SLOT_BATCH, decltype(i32)::value> rs;
            rs.load(p, row, nb, va, j0, lane);
#pragma unroll
            for (int u = 0; u < APPLY_SLOT_BATCH; ++u) {
                const int j = j0 + u * SSA_WAVE + lane;
                const int64_t y = rs.y[u];
                const bool in = j < p.K && y >= 0 && y < p.M;
                if (j < Kp) ix[j] = !in ? S::NONE : rs.marked(u) ? S::masked((int32_t)y) : (int32_t)y;
            }
        }
    };
    if (p.nb32) slots(std::true_type{});
    else slots(std::false_type{});
    if (!live) {
        __builtin_memset(&qr, 0, sizeof(qr));
        __builtin_memset(&dr, 0, sizeof(dr));
    }
    wave_lds_sync();

    // ---- scores and dO.V
    for (int j0 = 0; j0 < Kp; j0 += STEP) {
        int xi[U];
#pragma unroll
        for (int u = 0; u < U; ++u) xi[u] = ix[j0 + u * RPI + sub];
        Raw<T, VEC> kv[U], vv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) kv[u] = load_raw<T, VEC>(krow(xi[u]));
#pragma unroll
        for (int u = 0; u < U; ++u) vv[u] = load_raw<T, VEC>(vrow(xi[u]));
        float s[U], t[U];
#pragma unroll
        for (int u = 0; u < U; ++u) s[u] = dot_raw<T, T, VEC>(qr, kv[u]);
#pragma unroll
        for (int u = 0; u < U; ++u) t[u] = dot_raw<T, TD, VEC>(dr, vv[u]);
        rows_to_lds<LPR, RPI, U>(s, li, sub, sc + j0, p.scale);
        rows_to_lds<LPR, RPI, U>(t, li, sub, dpv + j0, 1.f);
    }
    wave_lds_sync();

    // ---- softmax and the slots' weights
    float m = -INFINITY;
    for (int j = lane; j < p.K; j += SSA_WAVE) {
        const float s = ix[j] >= 0 ? sc[j] : -INFINITY;
        sc[j] = s;
        m = fmaxf(m, s);
    }
    m = wave_max(m);
    float l = 0.f;
    for (int j = lane; j < p.K; j += SSA_WAVE) l += expf(sc[j] - m);
    l = wave_sum(l);
    auto mask_of = [&](int j) __attribute__((always_inline)) {
        return p.drop_p > 0.f ? ((drop_uniform(p.seed, row, j) < p.drop_p) ? 0.f : drop_scale_of<T>(p))
                              : 1.f;
    };
    // dp w.r.t. the softmax output includes the dropout mask and scale
    float pdp = 0.f;
    for (int j = lane; j < p.K; j += SSA_WAVE) {
        const float pj = expf(sc[j] - m) / l;
        const float dpj = dpv[j] * mask_of(j);
        pdp += pj * dpj;
        sc[j] = pj;
        dpv[j] = dpj;
    }
    pdp = wave_sum(pdp);
    RowOut ro(gp, row, gl, h - g * p.rep, n);
    if (gp.bnd) {
        ro.qm = row_absmax(qr.e);
        ro.dm = row_absmax(dr.e);
    }
    for (int j = lane; j < Kp; j += SSA_WAVE) {
        float draw = 0.f;
        if (j < p.K) {
            const float pj = sc[j];
            draw = pj * (dpv[j] - pdp) * p.scale;
            ro.put(gp, ix[j], j, draw, pj * mask_of(j));
        }
        sc[j] = draw;
    }
    wave_lds_sync();

    // ---- dQ = sum draw k
    float acc[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc[e] = 0.f;
    for (int j0 = 0; j0 < Kp; j0 += STEP) {
        int xi[U];
        float w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            xi[u] = ix[j0 + u * RPI + sub];
            w[u] = sc[j0 + u * RPI + sub];
        }
        Raw<T, VEC> kv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) kv[u] = load_raw<T, VEC>(krow(xi[u]));
        bool none = false;
#pragma unroll
        for (int u = 0; u < U; ++u) none |= xi[u] == S::NONE;
        if (wave_ballot(none)) {
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (xi[u] == S::NONE) {
                    w[u] = 0.f;
                    __builtin_memset(&kv[u], 0, sizeof(kv[u]));
                }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < VEC; ++e) acc[e] = fmaf(w[u], to_f32(kv[u].e[e]), acc[e]);
    }
#pragma unroll
    for (int o = LPR; o < SSA_WAVE; o <<= 1)
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] += __shfl_xor(acc[e], o, SSA_WAVE);
    if (sub == 0 && live) {
        const int64_t at = b * gp.dqsb + h * gp.dqsh + (int64_t)n * gp.dqsn + li * VEC;
        store_vec<T, VEC>(gp.dq, at, acc, gp.out32);
    }
}

// Rows of more than GRAD_KLDS slots: nothing is kept per slot; the scores and
// dO.V are computed again in each pass (the softmax statistics online, then
// sum p dp, then the weights with the same per-slot arithmetic).
template <typename T, typename TD, int D>
__global__ void __launch_bounds__(WAVES * SSA_WAVE)
grad_rows_long_kernel(GradP gp) {
    using G = Geo<T, D>;
    constexpr int VEC = G::VEC, LPR = G::LPR, RPI = G::RPI;
    const ApplyP &p = gp.a;
    const int64_t nblocks = ceil_div((int64_t)gp.ng * gp.grows, WAVES);
    const int64_t blk = xcd_logical_block(launch_block(), nblocks);
    if (blk >= nblocks) return;
    const int wid = threadIdx.x / SSA_WAVE;
    const int64_t lrow = blk * WAVES + wid;
    if (lrow >= (int64_t)gp.ng * gp.grows) return;
    const int64_t row = gp.row0 + lrow;
    const int gl = (int)(lrow / gp.grows);
    const int lane = lane_id();
    const int sub = lane / LPR, li = lane % LPR;
    const int n = (int)(row % p.N);
    const int64_t bh = row / p.N;
    const int h = (int)(bh % p.Hq);
    const int b = (int)(bh / p.Hq);
    const int g = h / p.rep;
    const T *qrow = (const T *)p.q + b * p.qsb + h * p.qsh + (int64_t)n * p.qsn;
    const TD *dorow = (const TD *)gp.dout + b * gp.dosb + h * gp.dosh + (int64_t)n * gp.dosn;
    const bool live = li * VEC < p.d;
    const LongRow<T, VEC, LPR> R{p, row, (const T *)p.k + b * p.ksb + g * p.ksh,
                                 (const T *)p.v + b * p.vsb + g * p.vsh,
                                 p.nb ? p.nb + row * p.K : nullptr,
                                 p.valid ? p.valid + row * p.K : nullptr, live ? li * VEC : 0};
    float qf[VEC], dof[VEC];
    {
        const Raw<T, VEC> qr = load_raw<T, VEC>(qrow + R.lofs);
        const Raw<TD, VEC> dr = load_raw<TD, VEC>(dorow + R.lofs);
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            qf[e] = live ? to_f32(qr.e[e]) : 0.f;
            dof[e] = live ? to_f32(dr.e[e]) : 0.f;
        }
    }
    float m = -INFINITY, l = 0.f;
    for (int j0 = 0; j0 < p.K; j0 += RPI) {
        const int j = j0 + sub;
        const float sj = R.score(qf, j < p.K ? R.id(j) : -1);
        if (j < p.K) online_add(sj, m, l);
    }
    float mm, ll;
    online_merge(li == 0, m, l, mm, ll);
    auto mask_of = [&](int j) {
        return p.drop_p > 0.f ? ((drop_uniform(p.seed, row, j) < p.drop_p) ? 0.f : drop_scale_of<T>(p))
                              : 1.f;
    };
    float pdp = 0.f;
    for (int j0 = 0; j0 < p.K; j0 += RPI) {
        const int j = j0 + sub;
        const int x = j < p.K ? R.id(j) : -1;
        const float pj = expf(R.score(qf, x) - mm) / ll;
        const float dpj = R.dotv(dof, x) * mask_of(j);
        if (j < p.K && li == 0) pdp += pj * dpj;
    }
    pdp = wave_sum(pdp);
    RowOut ro(gp, row, gl, h - g * p.rep, n);
    if (gp.bnd) {
        ro.qm = row_absmax(qf);
        ro.dm = row_absmax(dof);
    }
    float dqa[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) dqa[e] = 0.f;
    for (int j0 = 0; j0 < p.K; j0 += RPI) {
        const int j = j0 + sub;
        const int x = j < p.K ? R.id(j) : -1;
        const float pj = expf(R.score(qf, x) - mm) / ll;
        const float mask = mask_of(j);
        const float draw = pj * (R.dotv(dof, x) * mask - pdp) * p.scale;
        if (j < p.K && li == 0) ro.put(gp, x, j, draw, pj * mask);
        // a masked slot's own row, weighed 0; none for padding and ids out of range
        const int64_t y = j >= p.K ? -1 : p.nb32 ? (int64_t)p.nb32[row * p.K + j] : R.nb[j];
        if (y < 0 || y >= p.M) continue;
        float kf[VEC];
        load_vec<T, VEC>(R.kb + y * p.ksn + R.lofs, kf);
#pragma unroll
        for (int e = 0; e < VEC; ++e) dqa[e] = fmaf(draw, kf[e], dqa[e]);
    }
#pragma unroll
    for (int o = LPR; o < SSA_WAVE; o <<= 1)
#pragma unroll
        for (int e = 0; e < VEC; ++e) dqa[e] += __shfl_xor(dqa[e], o, SSA_WAVE);
    if (sub == 0 && live) {
        const int64_t at = b * gp.dqsb + h * gp.dqsh + (int64_t)n * gp.dqsn + li * VEC;
        store_vec<T, VEC>(gp.dq, at, dqa, gp.out32);
    }
}

// ---------------------------------------------------------------- 4. key rows
// The grids a key row's terms are rounded to in deterministic mode: 2^(e - 51)
// for 2^e above 2 x count x the largest bound of its terms (row_bound), and for
// what that rounding leaves, at most half a unit a term, 2^(f - 51) for 2^f above
// count x 2^(e - 51).  A partial sum then stays below 2^52 units of its grid, so
// adding in fp64 is exact and the order does not matter.  Held as the constants
// 1.5 x 2^52 units (0: no term but zeros and NaNs; NaN: the bound is not finite).
// The first sum starts there, so adding a product rounds it to the grid; which way
// half a unit goes depends on the sum, but then what is left is half a unit too and
// on the second grid, whose rounding knows nothing of the sums: the two sums
// together are the same in any order.
struct GridSum {
    double m1, m2, u2;     // u2: the second grid's unit
    __device__ __forceinline__ GridSum(uint32_t cnt, uint32_t code) {
        const double bound = 2.0 * (double)cnt * (double)__uint_as_float(code << 16);
        m1 = m2 = u2 = 0.0;
        if (!(bound < 1e300)) {
            m1 = __builtin_nan("");
        } else if (bound > 0.0) {
            int e = 0, f = 0;
            (void)frexp(bound, &e);                              // bound < 2^e
            (void)frexp(ldexp((double)cnt, e - 51), &f);
            m1 = ldexp(1.5, e + 1);
            m2 = ldexp(1.5, f + 1);
            u2 = ldexp(1.0, f - 51);
        }
    }
    // hi from m1 on, lo from 0: its units, and m2's bits once a term
    __device__ __forceinline__ void add(double w, double x, double &hi, uint64_t &lo) const {
        const double s = fma(w, x, hi);
        lo += (uint64_t)__double_as_longlong(fma(w, x, hi - s) + m2);
        hi = s;
    }
    __device__ __forceinline__ double second(uint64_t lo, int terms) const {
        return (double)(int64_t)(lo - (uint64_t)terms * (uint64_t)__double_as_longlong(m2)) * u2;
    }
};

// the segment of this wavefront, or nullptr past the group's last
__device__ __forceinline__ const GradSeg *wave_segment(const GradP &gp, int &gl) {
    const int64_t gblocks = ceil_div(gp.segcap, WAVES);
    const int64_t nblocks = gblocks * gp.ng;
    const int64_t blk = xcd_logical_block(launch_block(), nblocks);
    if (blk >= nblocks) return nullptr;
    gl = (int)(blk / gblocks);
    const int64_t si = (blk - gl * gblocks) * WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x / SSA_WAVE);
    if (si >= gp.nseg[gl]) return nullptr;
    return gp.segs + (int64_t)gl * gp.segcap + si;
}

// deterministic mode: the largest bounds of each key row's terms (integer maxima
// of float patterns, whose result does not depend on their order)
__global__ void __launch_bounds__(WAVES * SSA_WAVE) grad_bound_kernel(GradP gp) {
    int gl;
    const GradSeg *s = wave_segment(gp, gl);
    if (!s) return;
    const GradSeg sg = *s;
    uint32_t wk = 0, wv = 0;
    for (int i = lane_id(); i < sg.len; i += SSA_WAVE) {
        const uint32_t b = gp.bnd[sg.begin + i];
        wk = max(wk, b >> 16);
        wv = max(wv, b & 0xffffu);
    }
    wk = wave_max_u(wk);
    wv = wave_max_u(wv);
    if (lane_id() == 0) {
        uint32_t *w = gp.wmax + 2 * ((int64_t)gl * gp.a.M + sg.key);
        atomicMax(w, wk);
        atomicMax(w + 1, wv);
    }
}

// The sum of a group's parts up to this one (a launch with all its rows: this
// launch's), in the order of the parts; kept for the next unless this is the last.
template <typename A>
__device__ __forceinline__ A add_part(const GradP &gp, A *acc, A sum) {
    if (!gp.first) sum += *acc;
    if (!gp.last) *acc = sum;
    return sum;
}

// One wavefront per segment of a key row's list; RPI entries a step, U steps
// in flight.  Bound: the L2 delivery of the q and dO rows (2 rows of d per
// entry: 8.6 GB in 473 us, 18.2 TB/s) and their FMAs.  Deterministic: fp64 issue
// and registers (1.27 M entries of d = 80: 114 us; 85 with one grid; four entries a
// lane in flight instead of two leave 2 waves a SIMD, 126 us; one, 124 us).
template <typename T, typename TD, int D, int U, bool DET>
__global__ void __launch_bounds__(WAVES * SSA_WAVE)
grad_keys_kernel(GradP gp) {
    using G = Geo<T, D>;
    using A = typename std::conditional<DET, double, float>::type;
    constexpr int VEC = G::VEC, LPR = G::LPR, RPI = G::RPI, STEP = RPI * U;
    const ApplyP &p = gp.a;
    int gl;
    const GradSeg *s = wave_segment(gp, gl);
    if (!s) return;
    const GradSeg sg = *s;
    const int lane = lane_id();
    const int sub = lane / LPR, li = lane % LPR;
    const bool live = li * VEC < p.d;
    const int lofs = live ? li * VEC : 0;
    const int grp = gp.g0 + gl, b = grp / p.Hkv, g = grp % p.Hkv;
    const T *qb = (const T *)p.q + b * p.qsb + (int64_t)g * p.rep * p.qsh + lofs;
    const TD *db = (const TD *)gp.dout + b * gp.dosb + (int64_t)g * p.rep * gp.dosh + lofs;
    const int64_t ki = (int64_t)gl * p.M + sg.key;

    const uint32_t cnt = DET ? gp.klen[ki] : 0u;
    const GridSum sk(cnt, DET ? gp.wmax[2 * ki] : 0u), sv(cnt, DET ? gp.wmax[2 * ki + 1] : 0u);

    A ak[VEC], av[VEC];
    constexpr int LV = DET ? VEC : 1;      // the second grids' sums
    uint64_t nk[LV], nv[LV];
#pragma unroll
    for (int e = 0; e < VEC; ++e) { ak[e] = DET ? (A)sk.m1 : (A)0; av[e] = DET ? (A)sv.m1 : (A)0; }
#pragma unroll
    for (int e = 0; e < LV; ++e) { nk[e] = 0; nv[e] = 0; }
    auto fetch = [&](int j0, uint4 (&en)[U]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = j0 + u * RPI + sub;
            en[u] = gp.ent[sg.begin + (j < sg.len ? j : sg.len - 1)];
        }
    };
    uint4 en[U];
    if (sg.len > 0) fetch(0, en);
    for (int j0 = 0; j0 < sg.len; j0 += STEP) {
        Raw<T, VEC> qr[U];
        Raw<TD, VEC> dr[U];
        float wk[U], wv[U];
        bool zero = false;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int64_t qo, dO;
            if (gp.shift >= 0) {
                qo = (int64_t)((uint64_t)en[u].x << gp.shift);
                dO = (int64_t)((uint64_t)en[u].y << gp.shift);
            } else {
                const int64_t r = gp.r0 + en[u].x, hl = r / p.N, n = r - hl * p.N;
                qo = hl * p.qsh + n * p.qsn;
                dO = hl * gp.dosh + n * gp.dosn;
            }
            qr[u] = load_raw<T, VEC>(qb + qo);
            dr[u] = load_raw<TD, VEC>(db + dO);
            const bool in = j0 + u * RPI + sub < sg.len;
            wk[u] = in ? __uint_as_float(en[u].z) : 0.f;
            wv[u] = in ? __uint_as_float(en[u].w) : 0.f;
            zero |= wk[u] == 0.f || wv[u] == 0.f;
        }
        if (j0 + STEP < sg.len) fetch(j0 + STEP, en);
        // a zero weight takes nothing from its row, whatever the row holds
        if (wave_ballot(zero)) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (wk[u] == 0.f) __builtin_memset(&qr[u], 0, sizeof(qr[u]));
                if (wv[u] == 0.f) __builtin_memset(&dr[u], 0, sizeof(dr[u]));
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                const float x = to_f32(qr[u].e[e]), y = to_f32(dr[u].e[e]);
                if constexpr (DET) {
                    sk.add(wk[u], x, ak[e], nk[e]);
                    sv.add(wv[u], y, av[e], nv[e]);
                } else {
                    ak[e] = fmaf(wk[u], x, ak[e]);
                    av[e] = fmaf(wv[u], y, av[e]);
                }
            }
    }
    A lk[LV], lv[LV];
    if constexpr (DET) {
        const int terms = (sg.len + STEP - 1) / STEP * U;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            ak[e] -= sk.m1;
            av[e] -= sv.m1;
            lk[e] = sk.second(nk[e], terms);
            lv[e] = sv.second(nv[e], terms);
        }
    }
#pragma unroll
    for (int o = LPR; o < SSA_WAVE; o <<= 1)
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            ak[e] += __shfl_xor(ak[e], o, SSA_WAVE);
            av[e] += __shfl_xor(av[e], o, SSA_WAVE);
            if constexpr (DET) {
                lk[e] += __shfl_xor(lk[e], o, SSA_WAVE);
                lv[e] += __shfl_xor(lv[e], o, SSA_WAVE);
            }
        }
    if (sub != 0 || !live) return;
    if (sg.part >= 0) {
        A *pa = (A *)gp.part + (int64_t)sg.part * (DET ? 4 : 2) * p.d + lofs;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            pa[e] = ak[e];
            pa[p.d + e] = av[e];
            if constexpr (DET) { pa[2 * p.d + e] = lk[e]; pa[3 * p.d + e] = lv[e]; }
        }
        return;
    }
    if constexpr (DET) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) { ak[e] += lk[e]; av[e] += lv[e]; }
    }
    const uint8_t f = gp.poison[ki];
    const int64_t ok = b * gp.dksb + g * gp.dksh + (int64_t)sg.key * gp.dksn + lofs;
    const int64_t ov = b * gp.dvsb + g * gp.dvsh + (int64_t)sg.key * gp.dvsn + lofs;
    A *acc = (A *)gp.acc + (int64_t)sg.key * 2 * p.d + lofs;
    float x[VEC], y[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
        const A k = add_part(gp, acc + e, (f & 1) ? (A)__builtin_nanf("") : ak[e]);
        const A v = add_part(gp, acc + p.d + e, (f & 2) ? (A)__builtin_nanf("") : av[e]);
        x[e] = (float)k;
        y[e] = (float)v;
        if (gp.accumulate && gp.last) {
            x[e] += ((const float *)gp.dk)[ok + e];
            y[e] += ((const float *)gp.dv)[ov + e];
        }
    }
    if (!gp.last) return;
    store_vec<T, VEC>(gp.dk, ok, x, gp.out32);
    store_vec<T, VEC>(gp.dv, ov, y, gp.out32);
}

// ---------------------------------------------------------------- 5. joins
// Key rows of several segments: one wavefront per key row, its partials in
// order (eight rows of each in flight).
template <typename T, bool DET>
__global__ void __launch_bounds__(WAVES * SSA_WAVE) grad_join_kernel(GradP gp) {
    using A = typename std::conditional<DET, double, float>::type;
    const ApplyP &p = gp.a;
    const int64_t ki = launch_block() * WAVES + threadIdx.x / SSA_WAVE;
    if (ki >= (int64_t)gp.ng * p.M) return;
    const int2 kp = gp.kpart[ki];
    if (kp.y == 0) return;
    const uint8_t f = gp.poison[ki];
    const int64_t gl = ki / p.M, x = ki % p.M;
    const int64_t grp = gp.g0 + gl, b = grp / p.Hkv, g = grp % p.Hkv;
    const int d2 = 2 * p.d, pd = DET ? 2 * d2 : d2;
    auto total = [&](const A *pa) __attribute__((always_inline)) {
        A sum = (A)0;
        for (int s0 = 0; s0 < kp.y; s0 += 8) {
            A v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = s0 + u < kp.y ? pa[(int64_t)(s0 + u) * pd] : (A)0;
#pragma unroll
            for (int u = 0; u < 8; ++u) sum += v[u];
        }
        return sum;
    };
    for (int i = lane_id(); i < d2; i += SSA_WAVE) {
        const A *pa = (const A *)gp.part + (int64_t)kp.x * pd + i;
        A sum = total(pa);
        if constexpr (DET) sum += total(pa + d2);
        const bool isv = i >= p.d;
        const int e = isv ? i - p.d : i;
        float r = (float)add_part(gp, (A *)gp.acc + x * d2 + i,
                                  (f & (isv ? 2 : 1)) ? (A)__builtin_nanf("") : sum);
        if (!gp.last) continue;
        void *out = isv ? gp.dv : gp.dk;
        const int64_t at = isv ? b * gp.dvsb + g * gp.dvsh + x * gp.dvsn + e
                               : b * gp.dksb + g * gp.dksh + x * gp.dksn + e;
        if (gp.accumulate) r += ((const float *)out)[at];
        store_grad<T>(out, at, r, gp.out32);
    }
}

// zeros over a (B, H, N, d) view (no query row or no slot reaches anything)
template <typename T>
__global__ void __launch_bounds__(256) grad_fill0_kernel(void *out, int64_t sb, int64_t sh, int64_t sn,
                                                         int H, int N, int d, int64_t rows, int f32) {
    const int64_t total = rows * d;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t r = i / d, e = i % d;
        const int64_t n = r % N, bh = r / N;
        store_grad<T>(out, (bh / H) * sb + (bh % H) * sh + n * sn + e, 0.f, f32);
    }
}

// ---------------------------------------------------------------- launches
constexpr int64_t GRAD_SLOTS = (int64_t)1 << 28;   // slots per launch: 5.4 GB of workspace
constexpr int64_t GRAD_KEYS = (int64_t)1 << 25;    // key rows per launch: 2 GB

int64_t align256(int64_t x) { return (x + 255) / 256 * 256; }

struct GradLayout {
    int64_t ent, rank, tab, kbegin, klen, kfirst, kpart, bnd, wmax, poison, segs, nseg, part, acc, total;
};

// Groups and rows of each in one launch: whole (b, kv head) groups, so that few key
// rows' sums span launches, as many as hold GRAD_SLOTS slots and GRAD_KEYS key rows;
// of a group with more slots, the rows that hold GRAD_SLOTS.
void grad_launches(GradP &p) {
    const int64_t all = (int64_t)p.a.B * p.a.Hkv, rows = (int64_t)p.a.rep * p.a.N;
    const int64_t K = std::max(p.a.K, 1), slots = std::max<int64_t>(rows * K, 1);
    p.ng = (int)std::max<int64_t>(1, std::min(all, std::min(GRAD_SLOTS / slots, GRAD_KEYS / p.a.M)));
    p.grows = std::min(rows, std::max<int64_t>(1, GRAD_SLOTS / K));
    p.gslots = p.grows * p.a.K;
}

// Sizes of one launch over `ng` groups of `grows` rows, and the workspace they take.
//   * blocks of query rows: about 1,024 over the launch, but at least two
//     slots per counted key (the table costs 4 B per key and block)
//   * segments: about 32,768 over the launch, 256 to 4,096 entries
GradLayout grad_plan(GradP &p, int det) {
    const int64_t slots = (int64_t)p.ng * p.gslots, K = std::max(p.a.K, 1);
    const int64_t keys = (int64_t)p.ng * p.a.M;
    int64_t cr = std::max<int64_t>(ceil_div((int64_t)p.ng * p.grows, 1024), ceil_div(2 * (int64_t)p.a.M, K));
    p.crows = (int32_t)std::max<int64_t>(1, std::min(cr, p.grows));
    p.nc = (int32_t)ceil_div(p.grows, p.crows);
    int64_t sg = 256;
    while (sg < 4096 && sg * 32768 < slots) sg *= 2;
    p.seg = (int32_t)sg;
    p.segcap = p.a.M + p.gslots / sg;
    p.partcap = 2 * (p.gslots / sg);
    GradLayout L{};
    int64_t o = 0;
    auto take = [&](int64_t bytes) { const int64_t at = o; o += align256(bytes); return at; };
    L.ent = take(slots * 16);
    L.rank = take(slots * 4);
    L.tab = take((int64_t)p.ng * p.nc * p.a.M * 4);
    L.kbegin = take(keys * 8);
    L.klen = take(keys * 4);
    L.kfirst = take(keys * 4);
    L.kpart = take(keys * 8);
    L.bnd = take(det ? slots * 4 : 0);
    L.wmax = take(det ? keys * 8 : 0);
    L.poison = take(keys + 4);
    L.segs = take((int64_t)p.ng * p.segcap * (int64_t)sizeof(GradSeg));
    L.nseg = take((int64_t)p.ng * 4);
    const bool parts = p.grows < (int64_t)p.a.rep * p.a.N;
    L.acc = take(parts ? (int64_t)p.a.M * 2 * p.a.d * (det ? 8 : 4) : 0);
    L.part = take((int64_t)p.ng * p.partcap * 2 * p.a.d * (det ? 16 : 4));
    L.total = o;
    return L;
}

// K and V rows within 32-bit byte offsets of a wave-uniform base, rows
// addressed by 24-bit multiplies
bool grad_off32(const ApplyP &p, int elem, int D) {
    const int64_t lim = (int64_t)1 << 24;
    return p.M < lim && p.ksn * elem < lim && p.vsn * elem < lim &&
           ((int64_t)p.M * p.ksn + D) * elem < ((int64_t)1 << 31) &&
           ((int64_t)p.M * p.vsn + D) * elem < ((int64_t)1 << 31);
}

template <typename T, typename TD, int D, int U, bool OFF32>
int launch_rows(const GradP &p, dim3 grid, hipStream_t st) {
    constexpr int STEP = Geo<T, D>::RPI * U;
    const size_t lds = (size_t)WAVES * 3 * ceil_div(p.a.K, STEP) * STEP * 4;
    if (lds > 65536)
        SSA_CHECK_HIP(hipFuncSetAttribute((const void *)grad_rows_kernel<T, TD, D, U, OFF32>,
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((grad_rows_kernel<T, TD, D, U, OFF32>), grid, dim3(WAVES * SSA_WAVE), lds, st, p);
    SSA_CHECK_LAUNCH();
    return SSA_OK;
}

template <typename T, typename TD, int D>
int launch_grad(GradP p, int det, char *ws, hipStream_t st) {
    constexpr int U = grad_u<T, D>();
    const int all = p.a.B * p.a.Hkv;
    grad_launches(p);
    const int per = p.ng;
    const int64_t rows = (int64_t)p.a.rep * p.a.N, part = p.grows;
    const GradLayout L = grad_plan(p, det);
    p.ent = (uint4 *)(ws + L.ent);
    p.rank = (uint32_t *)(ws + L.rank);
    p.tab = (uint32_t *)(ws + L.tab);
    p.kbegin = (int64_t *)(ws + L.kbegin);
    p.klen = (uint32_t *)(ws + L.klen);
    p.kfirst = (int32_t *)(ws + L.kfirst);
    p.kpart = (int2 *)(ws + L.kpart);
    p.bnd = det ? (uint32_t *)(ws + L.bnd) : nullptr;
    p.wmax = det ? (uint32_t *)(ws + L.wmax) : nullptr;
    p.poison = (uint8_t *)(ws + L.poison);
    p.segs = (GradSeg *)(ws + L.segs);
    p.nseg = (int32_t *)(ws + L.nseg);
    p.acc = ws + L.acc;
    p.part = ws + L.part;
    const ApplyP &a = p.a;
    const size_t clds = (size_t)std::min(a.M, CNT_KEYS) * 4;
    // the launches of the groups and rows that p holds
    auto launch = [&]() -> int {
        hipLaunchKernelGGL(grad_count_kernel, launch_grid((int64_t)p.ng * p.nc), dim3(CNT_THREADS), clds,
                           st, p);
        SSA_CHECK_LAUNCH();
        const int64_t keys = (int64_t)p.ng * a.M;
        hipLaunchKernelGGL(grad_chunk_kernel, launch_grid(ceil_div(keys, 256)), dim3(256), 0, st, p);
        SSA_CHECK_LAUNCH();
        hipLaunchKernelGGL(grad_list_kernel, launch_grid(p.ng), dim3(1024), 0, st, p);
        SSA_CHECK_LAUNCH();
        hipLaunchKernelGGL(grad_segs_kernel, launch_grid(ceil_div(keys, 256)), dim3(256), 0, st, p);
        SSA_CHECK_LAUNCH();
        const dim3 grid = launch_grid(8 * ceil_div(ceil_div((int64_t)p.ng * p.grows, WAVES), 8));
        if (a.K > GRAD_KLDS) {
            hipLaunchKernelGGL((grad_rows_long_kernel<T, TD, D>), grid, dim3(WAVES * SSA_WAVE), 0, st, p);
            SSA_CHECK_LAUNCH();
        } else {
            const int rc = grad_off32(a, (int)sizeof(T), D) ? launch_rows<T, TD, D, U, true>(p, grid, st)
                                                            : launch_rows<T, TD, D, U, false>(p, grid, st);
            if (rc) return rc;
        }
        const dim3 kgrid = launch_grid(8 * ceil_div(ceil_div(p.segcap, WAVES) * p.ng, 8));
        constexpr int UK = U > 4 ? 4 : U;
        const dim3 jgrid = launch_grid(ceil_div(keys, WAVES));
        if (det) {
            hipLaunchKernelGGL(grad_bound_kernel, kgrid, dim3(WAVES * SSA_WAVE), 0, st, p);
            SSA_CHECK_LAUNCH();
            hipLaunchKernelGGL((grad_keys_kernel<T, TD, D, 2, true>), kgrid, dim3(WAVES * SSA_WAVE), 0, st,
                               p);
            SSA_CHECK_LAUNCH();
            hipLaunchKernelGGL((grad_join_kernel<T, true>), jgrid, dim3(WAVES * SSA_WAVE), 0, st, p);
        } else {
            hipLaunchKernelGGL((grad_keys_kernel<T, TD, D, UK, false>), kgrid, dim3(WAVES * SSA_WAVE), 0,
                               st, p);
            SSA_CHECK_LAUNCH();
            hipLaunchKernelGGL((grad_join_kernel<T, false>), jgrid, dim3(WAVES * SSA_WAVE), 0, st, p);
        }
        SSA_CHECK_LAUNCH();
        return SSA_OK;
    };
    for (int g0 = 0; g0 < all; g0 += per) {
        p.g0 = g0;
        p.ng = std::min(per, all - g0);
        for (int64_t r0 = 0; r0 < rows; r0 += part) {
            p.r0 = r0;
            p.row0 = g0 * rows + r0;
            p.grows = std::min(part, rows - r0);
            p.gslots = p.grows * a.K;
            p.first = r0 == 0;
            p.last = r0 + part >= rows;
            const int rc = launch();
            if (rc) return rc;
        }
    }
    return SSA_OK;
}

template <typename T, typename TD>
int grad_d(const GradP &p, int det, char *ws, hipStream_t st) {
    switch (ssa_pow2_instance(p.a.d)) {
        case 4: return launch_grad<T, TD, 4>(p, det, ws, st);
        case 8: return launch_grad<T, TD, 8>(p, det, ws, st);
        case 16: return launch_grad<T, TD, 16>(p, det, ws, st);
        case 32: return launch_grad<T, TD, 32>(p, det, ws, st);
        case 64: return launch_grad<T, TD, 64>(p, det, ws, st);
        case 128: return launch_grad<T, TD, 128>(p, det, ws, st);
        case 256: return launch_grad<T, TD, 256>(p, det, ws, st);
        case 512: return launch_grad<T, TD, 512>(p, det, ws, st);
        case 1024: return launch_grad<T, TD, 1024>(p, det, ws, st);
    }
    ssa_set_error("sparse_gather_attention_grad: head dim %d has no kernel instance", p.a.d);
    return SSA_E_UNSUP;
}

template <typename T>
int zero_outputs(const GradP &p, hipStream_t st) {
    const ApplyP &a = p.a;
    auto fill = [&](void *out, int64_t sb, int64_t sh, int64_t sn, int H, int N) -> int {
        const int64_t rows = (int64_t)a.B * H * N;
        if (rows == 0) return SSA_OK;
        hipLaunchKernelGGL((grad_fill0_kernel<T>), dim3((unsigned)std::min<int64_t>(ceil_div(rows * a.d, 256), 4096)),
                           dim3(256), 0, st, out, sb, sh, sn, H, N, a.d, rows, p.out32);
        SSA_CHECK_LAUNCH();
        return SSA_OK;
    };
    int rc = fill(p.dq, p.dqsb, p.dqsh, p.dqsn, a.Hq, a.N);
    if (!rc && !p.accumulate) rc = fill(p.dk, p.dksb, p.dksh, p.dksn, a.Hkv, a.M);
    if (!rc && !p.accumulate) rc = fill(p.dv, p.dvsb, p.dvsh, p.dvsn, a.Hkv, a.M);
    return rc;
}

int run_grad(const GradP &p, int dtype, int dodtype, int det, char *ws, hipStream_t st) {
    if (p.a.rows == 0 || p.a.K == 0) {
        switch (dtype) {
            case SSA_F32: return zero_outputs<float>(p, st);
            case SSA_BF16: return zero_outputs<bf16_t>(p, st);
            default: return zero_outputs<f16_t>(p, st);
        }
    }
    if (dtype == SSA_F32) return grad_d<float, float>(p, det, ws, st);
    if (dtype == SSA_BF16)
        return dodtype == SSA_F32 ? grad_d<bf16_t, float>(p, det, ws, st)
                                  : grad_d<bf16_t, bf16_t>(p, det, ws, st);
    return dodtype == SSA_F32 ? grad_d<f16_t, float>(p, det, ws, st)
                              : grad_d<f16_t, f16_t>(p, det, ws, st);
}

// checks the arguments and fills p; the workspace is left open
int grad_common(const ssa_apply_grad_args *a, GradP &p) {
    SSA_CHECK_ARG(a != nullptr, "sparse_gather_attention_grad: null args");
    p = GradP{};
    ssa_apply_args f = a->fwd;
    f.out = (void *)a->dq.ptr;                  // the forward's output is not written
    const int rc = apply_common(&f, p.a);
    if (rc) return rc;
    p.a.row_inv = nullptr;
    const int32_t dt = a->fwd.q.dtype;
    if (!ssa_head_dim_ok(a->fwd.d, dt)) {
        ssa_set_error("sparse_gather_attention_grad: head dim %d unsupported", a->fwd.d);
        return SSA_E_UNSUP;
    }
    SSA_CHECK_ARG(a->dout.ptr && a->dq.ptr && a->dk.ptr && a->dv.ptr,
                  "sparse_gather_attention_grad: null gradient");
    SSA_CHECK_ARG(a->dout.dtype == dt || a->dout.dtype == SSA_F32,
                  "sparse_gather_attention_grad: dout is q's type or fp32");
    SSA_CHECK_ARG(a->dq.dtype == a->dk.dtype && a->dk.dtype == a->dv.dtype &&
                      (a->dq.dtype == dt || a->dq.dtype == SSA_F32),
                  "sparse_gather_attention_grad: dq, dk and dv are all q's type or all fp32");
    p.dout = a->dout.ptr; p.dosb = a->dout.sb; p.dosh = a->dout.sh; p.dosn = a->dout.sn;
    p.dq = (void *)a->dq.ptr; p.dqsb = a->dq.sb; p.dqsh = a->dq.sh; p.dqsn = a->dq.sn;
    p.dk = (void *)a->dk.ptr; p.dksb = a->dk.sb; p.dksh = a->dk.sh; p.dksn = a->dk.sn;
    p.dv = (void *)a->dv.ptr; p.dvsb = a->dv.sb; p.dvsh = a->dv.sh; p.dvsn = a->dv.sn;
    p.out32 = a->dq.dtype == SSA_F32;
    // entries hold offsets of q and dO rows from their group's first in 32
    // bits, in the largest unit (up to 8 elements) that divides the strides
    const int64_t all = p.a.qsh | p.a.qsn | p.dosh | p.dosn;
    p.shift = (all & 1) ? 0 : (all & 2) ? 1 : (all & 4) ? 2 : 3;
    auto span = [&](int64_t sh, int64_t sn) { return (p.a.rep - 1) * sh + (int64_t)std::max(p.a.N - 1, 0) * sn; };
    const bool neg = p.a.qsh < 0 || p.a.qsn < 0 || p.dosh < 0 || p.dosn < 0;
    // (rows farther apart, or backwards: the entries hold the rows' numbers)
    if (neg || (std::max(span(p.a.qsh, p.a.qsn), span(p.dosh, p.dosn)) >> p.shift) >= ((int64_t)1 << 32))
        p.shift = -1;
    return SSA_OK;
}

int grad_run_checked(GradP &p, const ssa_apply_grad_args *a, void *ws, int64_t wsb, void *stream) {
    GradP q = p;
    grad_launches(q);
    const int64_t need = grad_plan(q, a->deterministic).total;
    SSA_CHECK_ARG(ws != nullptr && wsb >= need,
                  "sparse_gather_attention_grad: workspace of %lld bytes, %lld needed", (long long)wsb,
                  (long long)need);
    SSA_CHECK_ARG((uintptr_t)ws % 256 == 0,
                  "sparse_gather_attention_grad: workspace must be 256-byte aligned");
    return run_grad(p, a->fwd.q.dtype, a->dout.dtype, a->deterministic, (char *)ws, (hipStream_t)stream);
}

// ssa_apply_bwd_args (contiguous fp32 dout and gradients) as grad arguments
int from_bwd(const ssa_apply_bwd_args *b, ssa_apply_grad_args &a) {
    SSA_CHECK_ARG(b != nullptr, "sparse_gather_attention_bwd_det: null args");
    SSA_CHECK_ARG(b->dout && b->dq && b->dk && b->dv, "sparse_gather_attention_bwd: null grad");
    SSA_CHECK_ARG(b->fwd.neighbors32 == nullptr && b->fwd.neighbors != nullptr,
                  "sparse_gather_attention_bwd: needs the int64 neighbours");
    const int64_t d = b->fwd.d, N = b->fwd.N, M = b->fwd.M;
    a = ssa_apply_grad_args{};
    a.fwd = b->fwd;
    a.dout = {b->dout, SSA_F32, b->fwd.Hq * N * d, N * d, d};
    a.dq = {b->dq, SSA_F32, b->fwd.Hq * N * d, N * d, d};
    a.dk = {b->dk, SSA_F32, b->fwd.Hkv * M * d, M * d, d};
    a.dv = {b->dv, SSA_F32, b->fwd.Hkv * M * d, M * d, d};
    a.deterministic = 1;
    return SSA_OK;
}

}  // namespace

extern "C" int64_t ssa_sparse_gather_attention_grad_workspace_bytes(const ssa_apply_grad_args *a) {
    GradP p;
    const int rc = grad_common(a, p);
    if (rc) return rc;
    grad_launches(p);
    return grad_plan(p, a->deterministic).total;
}

extern "C" int ssa_sparse_gather_attention_grad(const ssa_apply_grad_args *a, void *workspace,
                                                int64_t workspace_bytes, void *stream) {
    GradP p;
    const int rc = grad_common(a, p);
    if (rc) return rc;
    return grad_run_checked(p, a, workspace, workspace_bytes, stream);
}

extern "C" int64_t ssa_sparse_gather_attention_bwd_det_workspace_bytes(const ssa_apply_bwd_args *b) {
    ssa_apply_grad_args a;
    const int rc = from_bwd(b, a);
    if (rc) return rc;
    return ssa_sparse_gather_attention_grad_workspace_bytes(&a);
}

extern "C" int ssa_sparse_gather_attention_bwd_det(const ssa_apply_bwd_args *b, void *workspace,
                                                   int64_t workspace_bytes, void *stream) {
    ssa_apply_grad_args a;
    int rc = from_bwd(b, a);
    if (rc) return rc;
    GradP p;
    rc = grad_common(&a, p);
    if (rc) return rc;
    p.accumulate = 1;
    return grad_run_checked(p, &a, workspace, workspace_bytes, stream);
}
