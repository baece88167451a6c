// ssa_apply.hip -- gather attention over a fixed neighbor graph (gfx950).
//
// Replaces sparse_gather_attention (sparse_attention.py:1096-1199).
//
// One wavefront per query row (b, h, n).  The row's neighbour ids are staged
// once in LDS as int32.  A row of d elements is covered by LPR lanes with
// 16-byte loads, so one load instruction brings RPI = 64/LPR whole K (or V)
// rows; with U rows in flight per lane the wave keeps U*RPI*row_bytes of
// gathers outstanding.  Scores go to LDS, the fp32 softmax is a wave
// reduction that turns them into the weights p in place (one exp per slot),
// and P.V accumulates in fp32 registers, reduced across the RPI row groups at
// the end.
//
// Numerics follow the reference: s = fp32(q.k) * fp32(scale); -inf where
// !valid; p = exp(s - max) / sum in fp32; 16-bit models round p to the value
// dtype before P.V (fp32_attn_weights keeps it fp32); P.V accumulates in fp32
// and is rounded once to the output dtype.
#include "ssa_apply_dev.h"

namespace {
template <typename T, int D, int U>
__global__ void __launch_bounds__(WAVES * SSA_WAVE)
apply_fwd_kernel(ApplyP p) {
    using G = Geo<T, D>;
    constexpr int VEC = G::VEC, LPR = G::LPR, RPI = G::RPI;
    extern __shared__ float smem[];
    const int64_t blk = xcd_logical_block(blockIdx.x, p.nblocks);
    if (blk >= p.nblocks) return;
    const int wid = threadIdx.x / SSA_WAVE;
    const int64_t row = blk * WAVES + wid;
    if (row >= p.rows) return;
    const int lane = lane_id();
    const int sub = lane / LPR, li = lane % LPR;
    constexpr int STEP = RPI * U;
    const int Kp = (p.K + STEP - 1) / STEP * STEP;                            // padded slots
    int32_t *ix = reinterpret_cast<int32_t *>(smem) + (int64_t)wid * 2 * Kp;    // key ids, -1 = masked
    float *sc = reinterpret_cast<float *>(ix + Kp);                           // scores, then p

    const int n = (int)(row % p.N);
    const int64_t bh = row / p.N;
    const int h = (int)(bh % p.Hq);
    const int b = (int)(bh / p.Hq);
    const int g = h / p.rep;

    const T *qrow = (const T *)p.q + b * p.qsb + h * p.qsh + (int64_t)n * p.qsn;
    const T *kb = (const T *)p.k + b * p.ksb + g * p.ksh;
    const T *vb = (const T *)p.v + b * p.vsb + g * p.vsh;
    const int64_t *nb = p.nb ? p.nb + row * p.K : nullptr;
    const uint8_t *va = p.valid ? p.valid + row * p.K : nullptr;

    // lanes whose elements lie past the head dim hold zeros and store nothing
    const bool live = li * VEC < p.d;
    const int lofs = live ? li * VEC : 0;
    // the q row is loaded first, beside the row's graph slots below
    float qf[VEC];
    load_vec<T, VEC>(qrow + lofs, qf);

    // neighbour ids once, as int32 in LDS; masked or out-of-range slots -> -1.
    // The row's padding count is the reference's (sparse_attention.py:1508):
    // slots the graph marks invalid (mask false, or a negative id in an int32
    // graph); an out-of-range id marked valid is skipped here but not counted
    int ninv = 0;
    auto slots = [&](auto i32) __attribute__((always_inline)) {
        for (int j0 = 0; j0 < Kp; j0 += APPLY_SLOT_BATCH * SSA_WAVE) {
            RowSlots<APPLY_SLOT_BATCH, decltype(i32)::value> rs;
            rs.load(p, row, nb, va, j0, lane);
#pragma unroll
            for (int u = 0; u < APPLY_SLOT_BATCH; ++u) {
                const int j = j0 + u * SSA_WAVE + lane;
                const bool in = j < p.K;
                const bool marked = in && rs.marked(u);
                const int64_t x = rs.y[u];
                if (j < Kp) ix[j] = (in && !marked && x >= 0 && x < p.M) ? (int)x : -1;
                ninv += __popcll(wave_ballot(marked));
            }
        }
    };
    if (p.nb32) slots(std::true_type{});
    else slots(std::false_type{});
    if (p.row_inv && lane == 0) p.row_inv[row] = ninv;
#pragma unroll
    for (int e = 0; e < VEC; ++e) qf[e] = live ? qf[e] : 0.f;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    // ---- scores (masked slots are set to -inf by the softmax); the lanes' sums
    // by DPP, whose tree is the shuffles' (no LDS round trips per row: 131 -> 96 us
    // at 73,488 fp32 rows of 54 slots, d = 64)
    for (int j0 = 0; j0 < Kp; j0 += STEP) {
        int xi[U];
#pragma unroll
        for (int u = 0; u < U; ++u) xi[u] = ix[j0 + u * RPI + sub];
        float kf[U][VEC];
#pragma unroll
        for (int u = 0; u < U; ++u)
            load_vec<T, VEC>(kb + (int64_t)(xi[u] < 0 ? 0 : xi[u]) * p.ksn + lofs, kf[u]);
        float part[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            part[u] = 0.f;
#pragma unroll
            for (int e = 0; e < VEC; ++e) part[u] = fmaf(qf[e], kf[u][e], part[u]);
        }
        rows_to_lds<LPR, RPI, U>(part, li, sub, sc + j0, p.scale);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    // ---- fp32 softmax, p computed once per slot (rounded to the value dtype
    // unless fp32_attn_weights; inverted dropout applied to p)
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
    const float inv = 1.f / l;
    for (int j = lane; j < Kp; j += SSA_WAVE) {
        float w = 0.f;
        if (j < p.K) {
            w = expf(sc[j] - m) * inv;
            if (!p.fp32w) w = Cvt<T>::round(w);
            if (p.drop_p > 0.f) {
                w = (drop_uniform(p.seed, row, j) < p.drop_p) ? 0.f : w * drop_scale_of<T>(p);
                if (!p.fp32w) w = Cvt<T>::round(w);
            }
        }
        sc[j] = w;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    // ---- P.V
    float acc[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc[e] = 0.f;
    for (int j0 = 0; j0 < Kp; j0 += STEP) {
        int xi[U];
        float pj[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            xi[u] = ix[j0 + u * RPI + sub];
            pj[u] = sc[j0 + u * RPI + sub];
        }
        float vf[U][VEC];
#pragma unroll
        for (int u = 0; u < U; ++u)
            load_vec<T, VEC>(vb + (int64_t)(xi[u] < 0 ? 0 : xi[u]) * p.vsn + lofs, vf[u]);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < VEC; ++e) acc[e] = fmaf(pj[u], vf[u][e], acc[e]);
    }
#pragma unroll
    for (int o = LPR; o < SSA_WAVE; o <<= 1)
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] += __shfl_xor(acc[e], o, SSA_WAVE);
    if (sub == 0 && live) {
        T *orow = (T *)p.out + b * p.osb + h * p.osh + (int64_t)n * p.osn + li * VEC;
#pragma unroll
        for (int e = 0; e < VEC; ++e) Cvt<T>::store(orow + e, acc[e]);
    }
}

template <typename T, int D>
__global__ void __launch_bounds__(WAVES * SSA_WAVE)
apply_fwd_long_kernel(ApplyP p) {
    using G = Geo<T, D>;
    constexpr int VEC = G::VEC, LPR = G::LPR, RPI = G::RPI;
    const int64_t blk = xcd_logical_block(blockIdx.x, p.nblocks);
    if (blk >= p.nblocks) return;
    const int wid = threadIdx.x / SSA_WAVE;
    const int64_t row = blk * WAVES + wid;
    if (row >= p.rows) return;
    const int lane = lane_id();
    const int sub = lane / LPR, li = lane % LPR;
    const int n = (int)(row % p.N);
    const int64_t bh = row / p.N;
    const int h = (int)(bh % p.Hq);
    const int b = (int)(bh / p.Hq);
    const int g = h / p.rep;
    const T *qrow = (const T *)p.q + b * p.qsb + h * p.qsh + (int64_t)n * p.qsn;
    const bool live = li * VEC < p.d;
    const LongRow<T, VEC, LPR> R{p, row, (const T *)p.k + b * p.ksb + g * p.ksh,
                                 (const T *)p.v + b * p.vsb + g * p.vsh,
                                 p.nb ? p.nb + row * p.K : nullptr,
                                 p.valid ? p.valid + row * p.K : nullptr, live ? li * VEC : 0};
    if (p.row_inv) {
        int ninv = 0;
        for (int j0 = 0; j0 < p.K; j0 += SSA_WAVE) {
            bool mk = false;
            if (j0 + lane < p.K) (void)R.id(j0 + lane, &mk);
            ninv += __popcll(wave_ballot(mk));
        }
        if (lane == 0) p.row_inv[row] = ninv;
    }
    float qf[VEC];
    load_vec<T, VEC>(qrow + R.lofs, qf);
#pragma unroll
    for (int e = 0; e < VEC; ++e) qf[e] = live ? qf[e] : 0.f;
    float m = -INFINITY, l = 0.f;
    for (int j0 = 0; j0 < p.K; j0 += RPI) {
        const int j = j0 + sub;
        const float sj = R.score(qf, j < p.K ? R.id(j) : -1);
        if (j < p.K) online_add(sj, m, l);
    }
    float mm, ll;
    online_merge(li == 0, m, l, mm, ll);
    const float inv = 1.f / ll;
    float acc[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) acc[e] = 0.f;
    for (int j0 = 0; j0 < p.K; j0 += RPI) {
        const int j = j0 + sub;
        const int x = j < p.K ? R.id(j) : -1;
        const float sj = R.score(qf, x);
        float w = expf(sj - mm) * inv;
        if (!p.fp32w) w = Cvt<T>::round(w);
        if (p.drop_p > 0.f) {
            w = (drop_uniform(p.seed, row, j) < p.drop_p) ? 0.f : w * drop_scale_of<T>(p);
            if (!p.fp32w) w = Cvt<T>::round(w);
        }
        w = j < p.K ? w : 0.f;
        float vf[VEC];
        load_vec<T, VEC>(R.vb + (int64_t)(x < 0 ? 0 : x) * p.vsn + R.lofs, vf);
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] = fmaf(w, vf[e], acc[e]);
    }
#pragma unroll
    for (int o = LPR; o < SSA_WAVE; o <<= 1)
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] += __shfl_xor(acc[e], o, SSA_WAVE);
    if (sub == 0 && live) {
        T *orow = (T *)p.out + b * p.osb + h * p.osh + (int64_t)n * p.osn + li * VEC;
#pragma unroll
        for (int e = 0; e < VEC; ++e) Cvt<T>::store(orow + e, acc[e]);
    }
}

// ---------------------------------------------------------------- 16-bit forward
// Packed 16-bit arithmetic for bf16 / fp16 models whose attention weights are
// rounded to the value dtype (fp32_attn_weights off):
//  * q.k: four v_dot2 (pairs of 16-bit products, fp32 accumulate) per lane,
//    then a sum over the LPR lanes of a row by DPP row permutations;
//  * P.V: the weights are exact in the value dtype, so two neighbours j, j'
//    go through one v_dot2 per element: {p_j, p_j'} . {v_j[e], v_j'[e]},
//    with the element pairs gathered by v_perm;
//  * rows are addressed by 32-bit byte offsets from a wave-uniform base.
template <typename T, int D, int U>
__global__ void __launch_bounds__(WAVES * SSA_WAVE)
apply_fwd16_kernel(ApplyP p) {
    constexpr int LPR = D / 8;                 // lanes per row, 16 bytes each
    constexpr int RPI = SSA_WAVE / LPR;        // rows per wave load
    constexpr int STEP = RPI * U;              // slots per loop step
    constexpr bool BFLY = 2 * U == LPR;        // head dims 64 and 128
    static_assert(sizeof(T) == 2 && D % 8 == 0 && LPR <= 32 && U % 2 == 0, "16-bit path");
    extern __shared__ float smem[];
    const int64_t blk = xcd_logical_block(blockIdx.x, p.nblocks);
    if (blk >= p.nblocks) return;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / SSA_WAVE);
    const int64_t row = blk * WAVES + wid;
    if (row >= p.rows) return;
    const int lane = lane_id();
    const int sub = lane / LPR, li = lane % LPR;
    const int Kp = (p.K + STEP - 1) / STEP * STEP;                               // padded slots
    // key ids; masked, out-of-range and padding slots hold INT_MIN, whose low
    // 24 bits (all a 24-bit multiply reads) address row 0
    int32_t *ix = reinterpret_cast<int32_t *>(smem) + (int64_t)wid * 2 * Kp;
    float *sc = reinterpret_cast<float *>(ix + Kp);                           // scores, then p

    const int n = (int)(row % p.N);
    const int64_t bh = row / p.N;
    const int h = (int)(bh % p.Hq);
    const int b = (int)(bh / p.Hq);
    const int g = h / p.rep;
    const T *qrow = (const T *)p.q + b * p.qsb + h * p.qsh + (int64_t)n * p.qsn;
    const char *kb = (const char *)((const T *)p.k + b * p.ksb + g * p.ksh);
    const char *vb = (const char *)((const T *)p.v + b * p.vsb + g * p.vsh);
    const uint32_t krb = (uint32_t)(p.ksn * 2), vrb = (uint32_t)(p.vsn * 2);   // row bytes < 2^24
    // lanes whose 8 elements lie past the head dim hold zeros and store nothing
    const bool live = li * 8 < p.d;
    const uint32_t lio = live ? (uint32_t)li * 16u : 0u;
    const int64_t *nb = p.nb ? p.nb + row * p.K : nullptr;
    const uint8_t *va = p.valid ? p.valid + row * p.K : nullptr;

    // the q row is loaded first, beside the row's graph slots below
    uint4 q4 = *reinterpret_cast<const uint4 *>(qrow + (live ? li * 8 : 0));

    // neighbour ids as int32 in LDS (ids < 2^24, checked at dispatch); the
    // padding count takes the slots the graph marks invalid, as above
    int ninv = 0;
    auto slots = [&](auto i32) __attribute__((always_inline)) {
        for (int j0 = 0; j0 < Kp; j0 += APPLY_SLOT_BATCH * SSA_WAVE) {
            RowSlots<APPLY_SLOT_BATCH, decltype(i32)::value> rs;
            rs.load(p, row, nb, va, j0, lane);
#pragma unroll
            for (int u = 0; u < APPLY_SLOT_BATCH; ++u) {
                const int j = j0 + u * SSA_WAVE + lane;
                const bool in = j < p.K;
                const bool marked = in && rs.marked(u);
                const int64_t y = rs.y[u];
                const int x = (in && !marked && y >= 0 && y < p.M) ? (int)y : INT32_MIN;
                if (j < Kp) ix[j] = x;
                ninv += __popcll(wave_ballot(marked));
            }
        }
    };
    if (p.nb32) slots(std::true_type{});
    else slots(std::false_type{});
    if (p.row_inv && lane == 0) p.row_inv[row] = ninv;
    if (!live) q4 = make_uint4(0, 0, 0, 0);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    // ---- scores q.k * scale (masked slots are set to -inf by the softmax)
    for (int j0 = 0; j0 < Kp; j0 += STEP) {
        int xi[U];
#pragma unroll
        for (int u = 0; u < U; ++u) xi[u] = ix[j0 + u * RPI + sub];
        uint4 kv[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            kv[u] = *reinterpret_cast<const uint4 *>(kb + (__umul24((uint32_t)xi[u], krb) + lio));
        float part[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            part[u] = Dot2<T>::dot(q4.x, kv[u].x, 0.f);
            part[u] = Dot2<T>::dot(q4.y, kv[u].y, part[u]);
            part[u] = Dot2<T>::dot(q4.z, kv[u].z, part[u]);
            part[u] = Dot2<T>::dot(q4.w, kv[u].w, part[u]);
        }
        if constexpr (BFLY) {
            const float tot = butterfly_rows<U>(part, li);
            const int r = (U == 8 ? 4 * (li >= 8) : 0) + 2 * ((li & 4) != 0) + ((li & 2) != 0);
            if ((li & 1) == 0) sc[j0 + r * RPI + sub] = tot * p.scale;
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float tot = group_sum<LPR>(part[u]);
                if (li == 0) sc[j0 + u * RPI + sub] = tot * p.scale;
            }
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    // the first P.V step's V rows (they need only the ids) load while the
    // softmax runs
    uint4 vv0[U];
    {
        int xi[U];
#pragma unroll
        for (int u = 0; u < U; ++u) xi[u] = ix[u * RPI + sub];
#pragma unroll
        for (int u = 0; u < U; ++u)
            vv0[u] = *reinterpret_cast<const uint4 *>(vb + (__umul24((uint32_t)xi[u], vrb) + lio));
    }

    // ---- fp32 softmax; p rounded to the value dtype (inverted dropout on p);
    // padding slots get p = 0
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
    const float inv = 1.f / l;
    for (int j = lane; j < Kp; j += SSA_WAVE) {
        float w = 0.f;
        if (j < p.K) {
            w = Cvt<T>::round(expf(sc[j] - m) * inv);
            if (p.drop_p > 0.f)
                w = (drop_uniform(p.seed, row, j) < p.drop_p) ? 0.f
                                                              : Cvt<T>::round(w * drop_scale_of<T>(p));
        }
        sc[j] = w;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    // ---- P.V, neighbours in pairs
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.f;
    auto vstep = [&](int j0, const uint4 (&vv)[U]) __attribute__((always_inline)) {
        float pj[U];
#pragma unroll
        for (int u = 0; u < U; ++u) pj[u] = sc[j0 + u * RPI + sub];
#pragma unroll
        for (int u = 0; u < U; u += 2) {
            const uint32_t pp = Dot2<T>::pack(pj[u], pj[u + 1]);
            const uint32_t a[4] = {vv[u].x, vv[u].y, vv[u].z, vv[u].w};
            const uint32_t c[4] = {vv[u + 1].x, vv[u + 1].y, vv[u + 1].z, vv[u + 1].w};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                acc[2 * r] = Dot2<T>::dot(pp, __builtin_amdgcn_perm(c[r], a[r], 0x05040100u),
                                          acc[2 * r]);
                acc[2 * r + 1] = Dot2<T>::dot(pp, __builtin_amdgcn_perm(c[r], a[r], 0x07060302u),
                                              acc[2 * r + 1]);
            }
        }
    };
    vstep(0, vv0);
    for (int j0 = STEP; j0 < Kp; j0 += STEP) {
        int xi[U];
#pragma unroll
        for (int u = 0; u < U; ++u) xi[u] = ix[j0 + u * RPI + sub];
        uint4 vv[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            vv[u] = *reinterpret_cast<const uint4 *>(vb + (__umul24((uint32_t)xi[u], vrb) + lio));
        vstep(j0, vv);
    }
#pragma unroll
    for (int o = LPR; o < SSA_WAVE; o <<= 1)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += __shfl_xor(acc[e], o, SSA_WAVE);
    if (sub == 0 && live) {
        T *orow = (T *)p.out + b * p.osb + h * p.osh + (int64_t)n * p.osn + li * 8;
        uint4 o4;
        o4.x = Dot2<T>::bits(acc[0]) | (Dot2<T>::bits(acc[1]) << 16);
        o4.y = Dot2<T>::bits(acc[2]) | (Dot2<T>::bits(acc[3]) << 16);
        o4.z = Dot2<T>::bits(acc[4]) | (Dot2<T>::bits(acc[5]) << 16);
        o4.w = Dot2<T>::bits(acc[6]) | (Dot2<T>::bits(acc[7]) << 16);
        *reinterpret_cast<uint4 *>(orow) = o4;
    }
}

// Backward: recompute p, then dp = dO.v, ds = p (dp - sum p dp), draw = ds*scale,
// dq = sum draw k (direct store), dk += draw q, dv += p' dO (fp32 atomics).
// The form without a workspace (ssa_sparse_gather_attention_bwd); ssa_grad.hip
// sums the key rows without atomics and is many times faster.
template <typename T, int D>
__global__ void __launch_bounds__(WAVES * SSA_WAVE)
apply_bwd_kernel(ApplyP p) {
    using G = Geo<T, D>;
    constexpr int VEC = G::VEC, LPR = G::LPR, RPI = G::RPI;
    extern __shared__ float smem[];
    const int64_t blk = xcd_logical_block(blockIdx.x, p.nblocks);
    if (blk >= p.nblocks) return;
    const int wid = threadIdx.x / SSA_WAVE;
    const int64_t row = blk * WAVES + wid;
    if (row >= p.rows) return;
    const int lane = lane_id();
    const int sub = lane / LPR, li = lane % LPR;
    float *sc = smem + wid * 2 * p.K;     // scores, then p'
    float *dpv = sc + p.K;                // dp per slot

    const int n = (int)(row % p.N);
    const int64_t bh = row / p.N;
    const int h = (int)(bh % p.Hq);
    const int b = (int)(bh / p.Hq);
    const int g = h / p.rep;
    const T *qrow = (const T *)p.q + b * p.qsb + h * p.qsh + (int64_t)n * p.qsn;
    const T *kb = (const T *)p.k + b * p.ksb + g * p.ksh;
    const T *vb = (const T *)p.v + b * p.vsb + g * p.vsh;
    const int64_t *nb = p.nb + row * p.K;
    const uint8_t *va = p.valid ? p.valid + row * p.K : nullptr;
    // gradients are (rows, d) fp32; lanes past the head dim hold zeros and
    // write nothing
    const bool live = li * VEC < p.d;
    const int lofs = live ? li * VEC : 0;
    const float *dorow = p.dout + row * p.d + lofs;

    float qf[VEC], dof[VEC];
    load_vec<T, VEC>(qrow + lofs, qf);
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
        dof[e] = live ? dorow[e] : 0.f;
        qf[e] = live ? qf[e] : 0.f;
    }

    for (int j0 = 0; j0 < p.K; j0 += RPI) {
        const int j = j0 + sub;
        int64_t x = 0;
        bool o = false;
        if (j < p.K) { x = nb[j]; o = va ? (va[j] != 0) : true; }
        if (x < 0 || x >= p.M) { x = 0; o = false; }
        float kf[VEC], vf[VEC];
        load_vec<T, VEC>(kb + x * p.ksn + lofs, kf);
        load_vec<T, VEC>(vb + x * p.vsn + lofs, vf);
        float s = 0.f, dp = 0.f;
#pragma unroll
        for (int e = 0; e < VEC; ++e) { s = fmaf(qf[e], kf[e], s); dp = fmaf(dof[e], vf[e], dp); }
#pragma unroll
        for (int off = LPR / 2; off > 0; off >>= 1) {
            s += __shfl_xor(s, off, SSA_WAVE);
            dp += __shfl_xor(dp, off, SSA_WAVE);
        }
        if (li == 0 && j < p.K) { sc[j] = o ? s * p.scale : -INFINITY; dpv[j] = dp; }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float m = -INFINITY;
    for (int j = lane; j < p.K; j += SSA_WAVE) m = fmaxf(m, sc[j]);
    m = wave_max(m);
    float l = 0.f;
    for (int j = lane; j < p.K; j += SSA_WAVE) l += expf(sc[j] - m);
    l = wave_sum(l);
    // dp w.r.t. softmax output includes the dropout mask/scale
    float pdp = 0.f;
    for (int j = lane; j < p.K; j += SSA_WAVE) {
        float pj = expf(sc[j] - m) / l;
        float mask = 1.f;
        if (p.drop_p > 0.f) mask = (drop_uniform(p.seed, row, j) < p.drop_p) ? 0.f : drop_scale_of<T>(p);
        float dpj = dpv[j] * mask;
        pdp += pj * dpj;
        sc[j] = pj;          // keep p
        dpv[j] = dpj;        // keep dp (softmax-output side)
    }
    pdp = wave_sum(pdp);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    float dqa[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) dqa[e] = 0.f;
    for (int j0 = 0; j0 < p.K; j0 += RPI) {
        const int j = j0 + sub;
        if (j >= p.K) continue;
        int64_t x = nb[j];
        if (x < 0 || x >= p.M) continue;
        const float pj = sc[j];
        const float draw = pj * (dpv[j] - pdp) * p.scale;
        float mask = 1.f;
        if (p.drop_p > 0.f) mask = (drop_uniform(p.seed, row, j) < p.drop_p) ? 0.f : drop_scale_of<T>(p);
        const float pw = pj * mask;
        float kf[VEC];
        load_vec<T, VEC>(kb + x * p.ksn + lofs, kf);
        const int64_t kr = ((int64_t)b * p.Hkv + g) * p.M + x;
        float *dkr = p.dk + kr * p.d + lofs;
        float *dvr = p.dv + kr * p.d + lofs;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            dqa[e] = fmaf(draw, kf[e], dqa[e]);
            if (live && draw != 0.f) unsafeAtomicAdd(dkr + e, draw * qf[e]);
            if (live && pw != 0.f) unsafeAtomicAdd(dvr + e, pw * dof[e]);
        }
    }
#pragma unroll
    for (int o = LPR; o < SSA_WAVE; o <<= 1)
#pragma unroll
        for (int e = 0; e < VEC; ++e) dqa[e] += __shfl_xor(dqa[e], o, SSA_WAVE);
    if (sub == 0 && live) {
        float *dqr = p.dq + row * p.d + lofs;
#pragma unroll
        for (int e = 0; e < VEC; ++e) dqr[e] = dqa[e];
    }
}

// Backward of rows beyond LDS: the softmax statistics online, then
// sum p dp, then each slot's draw and p' (the arithmetic of apply_bwd_kernel,
// with the scores and dout . v computed again in each pass).
template <typename T, int D>
__global__ void __launch_bounds__(WAVES * SSA_WAVE)
apply_bwd_long_kernel(ApplyP p) {
    using G = Geo<T, D>;
    constexpr int VEC = G::VEC, LPR = G::LPR, RPI = G::RPI;
    const int64_t blk = xcd_logical_block(blockIdx.x, p.nblocks);
    if (blk >= p.nblocks) return;
    const int wid = threadIdx.x / SSA_WAVE;
    const int64_t row = blk * WAVES + wid;
    if (row >= p.rows) return;
    const int lane = lane_id();
    const int sub = lane / LPR, li = lane % LPR;
    const int n = (int)(row % p.N);
    const int64_t bh = row / p.N;
    const int h = (int)(bh % p.Hq);
    const int b = (int)(bh / p.Hq);
    const int g = h / p.rep;
    const T *qrow = (const T *)p.q + b * p.qsb + h * p.qsh + (int64_t)n * p.qsn;
    const bool live = li * VEC < p.d;
    const LongRow<T, VEC, LPR> R{p, row, (const T *)p.k + b * p.ksb + g * p.ksh,
                                 (const T *)p.v + b * p.vsb + g * p.vsh, p.nb + row * p.K,
                                 p.valid ? p.valid + row * p.K : nullptr, live ? li * VEC : 0};
    const float *dorow = p.dout + row * p.d + R.lofs;
    float qf[VEC], dof[VEC];
    load_vec<T, VEC>(qrow + R.lofs, qf);
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
        dof[e] = live ? dorow[e] : 0.f;
        qf[e] = live ? qf[e] : 0.f;
    }
    // the ids are read from the graph in each pass (the graph's validity and
    // range rules of the forward; the backward takes int64 ids only)
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
    float dqa[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) dqa[e] = 0.f;
    for (int j0 = 0; j0 < p.K; j0 += RPI) {
        const int j = j0 + sub;
        if (j >= p.K) continue;
        const int64_t xr = R.nb[j];
        if (xr < 0 || xr >= p.M) continue;
        const int x = R.id(j);
        const float pj = expf(R.score(qf, x) - mm) / ll;
        const float mask = mask_of(j);
        const float draw = pj * (R.dotv(dof, x) * mask - pdp) * p.scale;
        const float pw = pj * mask;
        float kf[VEC];
        load_vec<T, VEC>(R.kb + xr * p.ksn + R.lofs, kf);
        const int64_t kr = ((int64_t)b * p.Hkv + g) * p.M + xr;
        float *dkr = p.dk + kr * p.d + R.lofs;
        float *dvr = p.dv + kr * p.d + R.lofs;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            dqa[e] = fmaf(draw, kf[e], dqa[e]);
            if (live && draw != 0.f) unsafeAtomicAdd(dkr + e, draw * qf[e]);
            if (live && pw != 0.f) unsafeAtomicAdd(dvr + e, pw * dof[e]);
        }
    }
#pragma unroll
    for (int o = LPR; o < SSA_WAVE; o <<= 1)
#pragma unroll
        for (int e = 0; e < VEC; ++e) dqa[e] += __shfl_xor(dqa[e], o, SSA_WAVE);
    if (sub == 0 && live) {
        float *dqr = p.dq + row * p.d + R.lofs;
#pragma unroll
        for (int e = 0; e < VEC; ++e) dqr[e] = dqa[e];
    }
}

// The 16-bit path needs weights in the value dtype, 16-byte aligned rows,
// byte offsets of every K / V row (and q row slice) within 32 bits, and key
// ids below 2^24 (rows are addressed by 24-bit multiplies).
bool fwd16_ok(const ApplyP &p, int elem, int D) {
    const int64_t v = 16 / elem;
    const bool aligned = ((uintptr_t)p.q % 16 == 0) && ((uintptr_t)p.k % 16 == 0) &&
                         ((uintptr_t)p.v % 16 == 0) && ((uintptr_t)p.out % 16 == 0) &&
                         p.qsb % v == 0 && p.qsh % v == 0 && p.qsn % v == 0 && p.ksb % v == 0 &&
                         p.ksh % v == 0 && p.ksn % v == 0 && p.vsb % v == 0 && p.vsh % v == 0 &&
                         p.vsn % v == 0 && p.osb % v == 0 && p.osh % v == 0 && p.osn % v == 0;
    const int64_t lim = (int64_t)1 << 24;
    const bool small = p.M < lim && p.ksn * elem < lim && p.vsn * elem < lim &&
                       ((int64_t)p.M * p.ksn + D) * elem < ((int64_t)1 << 31) &&
                       ((int64_t)p.M * p.vsn + D) * elem < ((int64_t)1 << 31);
    return !p.fp32w && aligned && small;
}

template <typename T, int D>
int launch_apply(const ApplyP &p, hipStream_t st, bool bwd) {
    const int64_t grid = 8 * ceil_div(p.nblocks, 8);
    const bool lng = p.K > APPLY_KLDS;
    if (lng && !bwd) {
        hipLaunchKernelGGL((apply_fwd_long_kernel<T, D>), dim3((unsigned)grid),
                           dim3(WAVES * SSA_WAVE), 0, st, p);
        SSA_CHECK_LAUNCH();
        return SSA_OK;
    }
    if (lng) {
        hipLaunchKernelGGL((apply_bwd_long_kernel<T, D>), dim3((unsigned)grid),
                           dim3(WAVES * SSA_WAVE), 0, st, p);
        SSA_CHECK_LAUNCH();
        return SSA_OK;
    }
    if (bwd) {
        const size_t lds = (size_t)WAVES * 2 * p.K * sizeof(float);
        if (lds > 65536)
            SSA_CHECK_HIP(hipFuncSetAttribute((const void *)apply_bwd_kernel<T, D>,
                                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL((apply_bwd_kernel<T, D>), dim3((unsigned)grid),
                           dim3(WAVES * SSA_WAVE), lds, st, p);
    } else {
        // slot batches of 8 row loads, 4 where a load covers 16 rows or more
        // (64 slots a step at 8 rows a load: 64-wide bf16 heads 1% faster)
        constexpr int U = (Geo<T, D>::RPI >= 16) ? 4 : 8;
        if constexpr (sizeof(T) == 2 && D >= 8 && D <= 256) {   // two rows per wave at least
            if (fwd16_ok(p, (int)sizeof(T), D)) {
                constexpr int STEP = (SSA_WAVE / (D / 8)) * U;
                const size_t lds16 = (size_t)WAVES * 2 * ceil_div(p.K, STEP) * STEP * sizeof(float);
                if (lds16 > 65536)
                    SSA_CHECK_HIP(hipFuncSetAttribute((const void *)apply_fwd16_kernel<T, D, U>,
                                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                                      (int)lds16));
                hipLaunchKernelGGL((apply_fwd16_kernel<T, D, U>), dim3((unsigned)grid),
                                   dim3(WAVES * SSA_WAVE), lds16, st, p);
                SSA_CHECK_LAUNCH();
                return SSA_OK;
            }
        }
        constexpr int UF = Geo<T, D>::RPI * U;
        const size_t ldsf = (size_t)WAVES * 2 * ceil_div(p.K, UF) * UF * sizeof(float);
        if (ldsf > 65536)
            SSA_CHECK_HIP(hipFuncSetAttribute((const void *)apply_fwd_kernel<T, D, U>,
                                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)ldsf));
        hipLaunchKernelGGL((apply_fwd_kernel<T, D, U>), dim3((unsigned)grid),
                           dim3(WAVES * SSA_WAVE), ldsf, st, p);
    }
    SSA_CHECK_LAUNCH();
    return SSA_OK;
}

template <typename T>
int dispatch_d(const ApplyP &p, int d, hipStream_t st, bool bwd) {
    if (!ssa_head_dim_ok(d, std::is_same<T, float>::value ? SSA_F32 : SSA_BF16)) {
        ssa_set_error("sparse_gather_attention: head dim %d unsupported (4..1024: a power of two "
                      "or a multiple of %d)", d, std::is_same<T, float>::value ? 4 : 8);
        return SSA_E_UNSUP;
    }
    switch (ssa_pow2_instance(d)) {
        case 4: return launch_apply<T, 4>(p, st, bwd);
        case 8: return launch_apply<T, 8>(p, st, bwd);
        case 16: return launch_apply<T, 16>(p, st, bwd);
        case 32: return launch_apply<T, 32>(p, st, bwd);
        case 64: return launch_apply<T, 64>(p, st, bwd);
        case 128: return launch_apply<T, 128>(p, st, bwd);
        case 256: return launch_apply<T, 256>(p, st, bwd);
        case 512: return launch_apply<T, 512>(p, st, bwd);
        case 1024: return launch_apply<T, 1024>(p, st, bwd);
        default:
            ssa_set_error("sparse_gather_attention: head dim %d has no kernel instance", d);
            return SSA_E_UNSUP;
    }
}

int run_apply(const ApplyP &p, int dtype, int d, hipStream_t st, bool bwd) {
    if (p.rows == 0) return SSA_OK;
    switch (dtype) {
        case SSA_F32: return dispatch_d<float>(p, d, st, bwd);
        case SSA_BF16: return dispatch_d<bf16_t>(p, d, st, bwd);
        case SSA_F16: return dispatch_d<f16_t>(p, d, st, bwd);
    }
    ssa_set_error("sparse_gather_attention: bad dtype %d", dtype);
    return SSA_E_ARG;
}

}  // namespace

extern "C" int ssa_sparse_gather_attention(const ssa_apply_args *a, void *stream) {
    ApplyP p;
    int rc = apply_common(a, p);
    if (rc) return rc;
    return run_apply(p, a->q.dtype, a->d, (hipStream_t)stream, false);
}

namespace {

int bwd_common(const ssa_apply_bwd_args *a, ApplyP &p) {
    SSA_CHECK_ARG(a != nullptr, "sparse_gather_attention_bwd: null args");
    int rc = apply_common(&a->fwd, p);
    if (rc) return rc;
    SSA_CHECK_ARG(a->dout && a->dq && a->dk && a->dv, "sparse_gather_attention_bwd: null grad");
    SSA_CHECK_ARG(a->fwd.neighbors32 == nullptr && a->fwd.neighbors != nullptr,
                  "sparse_gather_attention_bwd: needs the int64 neighbours");
    p.dout = a->dout; p.dq = a->dq; p.dk = a->dk; p.dv = a->dv;
    p.row_inv = nullptr;
    return SSA_OK;
}

}  // namespace

extern "C" int ssa_sparse_gather_attention_bwd(const ssa_apply_bwd_args *a, void *stream) {
    ApplyP p;
    const int rc = bwd_common(a, p);
    if (rc) return rc;
    return run_apply(p, a->fwd.q.dtype, a->fwd.d, (hipStream_t)stream, true);
}
