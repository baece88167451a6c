// ssa_apply_dev.h -- device helpers shared by the gather attention's forward
// (ssa_apply.hip) and its gradients (ssa_grad.hip).
#pragma once

#include <type_traits>

#include "ssa_common.h"

namespace {

struct ApplyP {
    int32_t B, Hq, Hkv, N, M, K, rep;
    int32_t d;             // head dim (<= the kernel's D; lanes past it load zeros, store nothing)
    const void *q, *k, *v;
    int64_t qsb, qsh, qsn, ksb, ksh, ksn, vsb, vsh, vsn;
    const int64_t *nb;
    const uint8_t *valid;
    const int32_t *nb32;   // or the graph as int32 ids, negative = invalid
    int32_t *row_inv;      // optional: per row, its count of invalid slots
    float scale;
    int32_t fp32w;
    float drop_p;
    float drop_scale;
    uint64_t seed;
    void *out;
    int64_t osb, osh, osn;
    int64_t rows;          // B*Hq*N
    int64_t nblocks;       // logical blocks
    // backward
    const float *dout;
    float *dq, *dk, *dv;
};

constexpr int WAVES = 4;   // waves per workgroup

template <typename T> struct VecOf;
template <> struct VecOf<float> { static constexpr int n = 4; };
template <> struct VecOf<bf16_t> { static constexpr int n = 8; };
template <> struct VecOf<f16_t> { static constexpr int n = 8; };

template <typename T, int D> struct Geo {
    // elements per lane: a 16-byte load, more when the row is wider than a
    // wave holds that way (fp32 beyond 256)
    static constexpr int VEC = (VecOf<T>::n < D) ? (VecOf<T>::n * SSA_WAVE < D ? D / SSA_WAVE
                                                                              : VecOf<T>::n)
                                                 : D;
    static constexpr int LPR = D / VEC;                                // lanes per row
    static constexpr int RPI = SSA_WAVE / LPR;                         // rows per wave load
    static_assert(D % VEC == 0, "head dim must be a multiple of the vector width");
    static_assert(LPR <= SSA_WAVE, "row wider than a wave");
};

template <typename T, int VEC>
__device__ __forceinline__ void load_vec(const T *p, float (&f)[VEC]) {
    if constexpr (sizeof(T) * VEC == 32) {
        uint4 u[2] = {reinterpret_cast<const uint4 *>(p)[0], reinterpret_cast<const uint4 *>(p)[1]};
        const T *e = reinterpret_cast<const T *>(u);
#pragma unroll
        for (int i = 0; i < VEC; ++i) f[i] = to_f32(e[i]);
    } else if constexpr (sizeof(T) * VEC == 16) {
        uint4 u = *reinterpret_cast<const uint4 *>(p);
        const T *e = reinterpret_cast<const T *>(&u);
#pragma unroll
        for (int i = 0; i < VEC; ++i) f[i] = to_f32(e[i]);
    } else if constexpr (sizeof(T) * VEC == 8) {
        uint2 u = *reinterpret_cast<const uint2 *>(p);
        const T *e = reinterpret_cast<const T *>(&u);
#pragma unroll
        for (int i = 0; i < VEC; ++i) f[i] = to_f32(e[i]);
    } else {
#pragma unroll
        for (int i = 0; i < VEC; ++i) f[i] = to_f32(p[i]);
    }
}

// counter-based uniform in [0, 1): 64-bit mix of (seed, row, slot)
__device__ __forceinline__ float drop_uniform(uint64_t seed, int64_t row, int j) {
    uint64_t x = seed ^ (uint64_t)row * 0x9E3779B97F4A7C15ull ^ ((uint64_t)j << 32);
    x ^= x >> 33; x *= 0xff51afd7ed558ccdull;
    x ^= x >> 33; x *= 0xc4ceb9fe1a85ec53ull;
    x ^= x >> 33;
    return (float)(x >> 40) * (1.0f / 16777216.0f);
}

// The factor kept weights are multiplied by: the reference's dropout runs on
// the weights in their own dtype (the value dtype, or fp32 with
// fp32_attn_weights), whose noise tensor holds 1 / (1 - p) rounded to that
// dtype (sparse_attention.py:1193-1194).
template <typename T>
__device__ __forceinline__ float drop_scale_of(const ApplyP &p) {
    return p.fp32w ? p.drop_scale : Cvt<T>::round(p.drop_scale);
}

// A query row's graph slots j0 + u * 64 + lane (u < NB): the ids (int32 graph,
// or int64 ids and the mask) of all NB groups are loaded before any is used,
// so the row pays one memory latency for them instead of one per group.  The
// loads are unconditional (lanes past the row read its last slot) and the
// graph's layout is a template parameter, so no branch separates a load from
// the others.
constexpr int APPLY_SLOT_BATCH = 4;
template <int NB, bool I32>
struct RowSlots {
    int64_t y[NB];
    uint8_t v[NB];
    __device__ __forceinline__ void load(const ApplyP &p, int64_t row, const int64_t *nb,
                                         const uint8_t *va, int j0, int lane) {
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int j = min(j0 + u * SSA_WAVE + lane, p.K - 1);
            if constexpr (I32) {
                y[u] = p.nb32[row * p.K + j];
            } else {
                y[u] = nb[j];
                v[u] = va ? va[j] : (uint8_t)1;
            }
        }
    }
    // the slot is marked invalid: mask false, or a negative id in an int32 graph
    __device__ __forceinline__ bool marked(int u) const {
        if constexpr (I32) return y[u] < 0;
        else return v[u] == 0;
    }
};

// ---------------------------------------------------------------- rows beyond LDS
// Rows of more than APPLY_KLDS slots (whose scores do not fit a wave's share
// of LDS): nothing is kept per slot.  The scores are computed again in each
// pass over the row (same products, same order, so the same values): first
// the softmax maximum and sum online (a slot raising the maximum rescales the
// sum), then the weights, whose arithmetic is the kernels' above.
constexpr int APPLY_KLDS = 4096;

template <typename T, int VEC, int LPR>
struct LongRow {
    const ApplyP &p;
    int64_t row;
    const T *kb, *vb;
    const int64_t *nb;
    const uint8_t *va;
    int lofs;
    // key id of slot j, -1 when masked or out of range
    __device__ int id(int j, bool *marked = nullptr) const {
        const int64_t x = p.nb32 ? (int64_t)p.nb32[row * p.K + j] : nb[j];
        const bool mk = p.nb32 ? x < 0 : (va ? va[j] == 0 : false);
        if (marked) *marked = mk;
        return (!mk && x >= 0 && x < p.M) ? (int)x : -1;
    }
    // score of slot j (key id x, -1: -inf), every lane of the slot's group
    __device__ float score(const float (&qf)[VEC], int x) const {
        float kf[VEC];
        load_vec<T, VEC>(kb + (int64_t)(x < 0 ? 0 : x) * p.ksn + lofs, kf);
        float part = 0.f;
#pragma unroll
        for (int e = 0; e < VEC; ++e) part = fmaf(qf[e], kf[e], part);
#pragma unroll
        for (int o = LPR / 2; o > 0; o >>= 1) part += __shfl_xor(part, o, SSA_WAVE);
        return x >= 0 ? part * p.scale : -INFINITY;
    }
    // dout . v of key x (row 0 for -1), every lane of the slot's group
    __device__ float dotv(const float (&dof)[VEC], int x) const {
        float vf[VEC];
        load_vec<T, VEC>(vb + (int64_t)(x < 0 ? 0 : x) * p.vsn + lofs, vf);
        float part = 0.f;
#pragma unroll
        for (int e = 0; e < VEC; ++e) part = fmaf(dof[e], vf[e], part);
#pragma unroll
        for (int o = LPR / 2; o > 0; o >>= 1) part += __shfl_xor(part, o, SSA_WAVE);
        return part;
    }
};

// online softmax statistics of one lane group, then merged over the wave
__device__ __forceinline__ void online_add(float s, float &m, float &l) {
    if (s == -INFINITY) return;
    if (s > m) { l = l * expf(m - s) + 1.f; m = s; }
    else l += expf(s - m);
}

__device__ __forceinline__ void online_merge(bool lead, float m, float l, float &mm, float &ll) {
    mm = wave_max(lead ? m : -INFINITY);
    ll = wave_sum((lead && m != -INFINITY) ? l * expf(m - mm) : 0.f);
}

template <typename T> struct Dot2;
template <> struct Dot2<bf16_t> {
    typedef __bf16 __attribute__((ext_vector_type(2))) v2;
    static __device__ __forceinline__ float dot(uint32_t a, uint32_t b, float c) {
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2, a), __builtin_bit_cast(v2, b),
                                               c, false);
    }
    // two bf16-exact fp32 values as a pair (a low, b high): their upper halves
    static __device__ __forceinline__ uint32_t pack(float a, float b) {
        return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
    }
    static __device__ __forceinline__ uint32_t bits(float v) { return f32_to_bf16_bits(v); }
};
template <> struct Dot2<f16_t> {
    typedef _Float16 __attribute__((ext_vector_type(2))) v2;
    static __device__ __forceinline__ float dot(uint32_t a, uint32_t b, float c) {
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(v2, a), __builtin_bit_cast(v2, b), c,
                                      false);
    }
    static __device__ __forceinline__ uint32_t pack(float a, float b) {
        const v2 h = {(_Float16)a, (_Float16)b};       // exact: both are fp16 values
        return __builtin_bit_cast(uint32_t, h);
    }
    static __device__ __forceinline__ uint32_t bits(float v) {
        const _Float16 h = (_Float16)v;
        return (uint32_t)__builtin_bit_cast(uint16_t, h);
    }
};

template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
    // every source lane of these patterns exists: old (0) is never used, and
    // an identity old lets the move fold into the add as a DPP operand
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF,
                                                          false));
}

// sum over the L lanes of each aligned group (L a power of two <= 32); every
// lane of the group gets the sum
template <int L>
__device__ __forceinline__ float group_sum(float v) {
    if constexpr (L >= 16) v = dpp_add<0x140>(v);   // row mirror
    if constexpr (L >= 8) v = dpp_add<0x141>(v);    // row half mirror
    if constexpr (L >= 2) v = dpp_add<0xB1>(v);     // quad perm [1,0,3,2]
    if constexpr (L >= 4) v = dpp_add<0x4E>(v);     // quad perm [2,3,0,1]
    if constexpr (L >= 32) v += __shfl_xor(v, 16, SSA_WAVE);
    return v;
}

template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}

// Reduce U per-lane partials (one per row) over the 2U lanes of a row group
// by a butterfly: at each step a lane pair splits its rows, each lane sending
// the half it drops and adding the half it keeps (row mirror, half mirror,
// quad swaps as the pairings).  Afterwards lanes li and li ^ 1 both hold the
// total of row r = 4 [li >= 8] + 2 [li & 4] + [li & 2] (U = 8), or
// r = 2 [li & 4] + [li & 2] (U = 4).
template <int U>
__device__ __forceinline__ float butterfly_rows(float (&v)[U], int li) {
    static_assert(U == 4 || U == 8, "butterfly over 8 or 16 lanes");
    float w[4];
    if constexpr (U == 8) {
        const bool hi = li >= 8;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float send = hi ? v[k] : v[k + 4], keep = hi ? v[k + 4] : v[k];
            w[k] = keep + dpp_move<0x140>(send);        // row mirror: li <-> 15 - li
        }
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) w[k] = v[k];
    }
    float x[2];
    {
        const bool hi = (li & 4) != 0;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const float send = hi ? w[k] : w[k + 2], keep = hi ? w[k + 2] : w[k];
            x[k] = keep + dpp_move<0x141>(send);        // half mirror: li <-> 7 - li (in 8)
        }
    }
    const bool hi = (li & 2) != 0;
    const float send = hi ? x[0] : x[1], keep = hi ? x[1] : x[0];
    float y = keep + dpp_move<0x4E>(send);              // quad perm [2,3,0,1]: li ^ 2
    return y + dpp_move<0xB1>(y);                       // quad perm [1,0,3,2]: li ^ 1
}

// Sum over the L lanes of each aligned group as xor shuffles by L / 2, .., 1
// add them (that tree's rounding, which long and unvectorised rows have too):
// once the step by 16 has run, rotating a row of 16 lanes by 8, 4, 2 and 1
// brings a lane the same partner value as the xor.
template <int L>
__device__ __forceinline__ float tree_sum(float v) {
    if constexpr (L > 32) return wave_sum(v);
    if constexpr (L >= 32) v += __shfl_xor(v, 16, SSA_WAVE);
    if constexpr (L >= 16) v = dpp_add<0x128>(v);        // row_ror:8
    if constexpr (L >= 16) v = dpp_add<0x124>(v);        // row_ror:4
    if constexpr (L == 8) v += dpp_move<0x1B>(dpp_move<0x141>(v));   // li ^ 7, then ^ 3
    if constexpr (L >= 4) v = dpp_add<0x4E>(v);          // li ^ 2
    if constexpr (L >= 2) v = dpp_add<0xB1>(v);          // li ^ 1
    return v;
}

// butterfly_rows with the pairings of tree_sum (li ^ 8, ^ 4, ^ 2, ^ 1), so each
// row's total is that tree's, bit for bit
template <int U>
__device__ __forceinline__ float tree_rows(float (&v)[U], int li) {
    static_assert(U == 4 || U == 8, "over 8 or 16 lanes");
    float w[4];
    if constexpr (U == 8) {
        const bool hi = li >= 8;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float send = hi ? v[k] : v[k + 4], keep = hi ? v[k + 4] : v[k];
            w[k] = keep + dpp_move<0x128>(send);         // row_ror:8
        }
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) w[k] = v[k];
    }
    float x[2];
    {
        const bool hi = (li & 4) != 0;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const float send = hi ? w[k] : w[k + 2], keep = hi ? w[k + 2] : w[k];
            x[k] = keep + dpp_move<0x1B>(dpp_move<0x141>(send));
        }
    }
    const bool hi = (li & 2) != 0;
    const float send = hi ? x[0] : x[1], keep = hi ? x[1] : x[0];
    float y = keep + dpp_move<0x4E>(send);
    return y + dpp_move<0xB1>(y);
}

// sums of v[u] over each row's LPR lanes, stored to dst[row slot u * RPI + sub]
template <int LPR, int RPI, int U>
__device__ __forceinline__ void rows_to_lds(float (&v)[U], int li, int sub, float *dst, float mul) {
    if constexpr (2 * U == LPR && (U == 4 || U == 8)) {
        const float t = tree_rows<U>(v, li);
        const int r = (U == 8 ? 4 * (li >= 8) : 0) + 2 * ((li & 4) != 0) + ((li & 2) != 0);
        if ((li & 1) == 0) dst[r * RPI + sub] = t * mul;
    } else {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float t = tree_sum<LPR>(v[u]);
            if (li == 0) dst[u * RPI + sub] = t * mul;
        }
    }
}

// checks the forward's arguments and fills p
inline int check_view(const ssa_tensor4 &t, int dtype, const char *name) {
    if (!t.ptr) { ssa_set_error("%s: null pointer", name); return SSA_E_ARG; }
    if (t.dtype != dtype) { ssa_set_error("%s: dtype mismatch", name); return SSA_E_ARG; }
    return SSA_OK;
}

inline int apply_common(const ssa_apply_args *a, ApplyP &p) {
    SSA_CHECK_ARG(a != nullptr, "sparse_gather_attention: null args");
    SSA_CHECK_ARG(a->B >= 0 && a->Hq > 0 && a->Hkv > 0 && a->N >= 0 && a->M > 0 && a->K >= 0,
                  "sparse_gather_attention: bad sizes B=%d Hq=%d Hkv=%d N=%d M=%d K=%d", a->B,
                  a->Hq, a->Hkv, a->N, a->M, a->K);
    SSA_CHECK_ARG(a->Hq % a->Hkv == 0, "sparse_gather_attention: Hq %% Hkv != 0");
    SSA_CHECK_ARG((int64_t)a->B * a->Hq * a->N * a->K < ((int64_t)1 << 62),
                  "sparse_gather_attention: too many slots");
    SSA_CHECK_ARG(a->q.dtype >= 0 && a->q.dtype <= 2, "sparse_gather_attention: bad dtype");
    int rc;
    if ((rc = check_view(a->q, a->q.dtype, "q"))) return rc;
    if ((rc = check_view(a->k, a->q.dtype, "k"))) return rc;
    if ((rc = check_view(a->v, a->q.dtype, "v"))) return rc;
    SSA_CHECK_ARG((a->neighbors != nullptr || a->neighbors32 != nullptr) && a->out != nullptr,
                  "sparse_gather_attention: null");
    SSA_CHECK_ARG(a->dropout_p >= 0.f && a->dropout_p < 1.f, "dropout p must be in [0, 1)");
    p = ApplyP{};
    p.B = a->B; p.Hq = a->Hq; p.Hkv = a->Hkv; p.N = a->N; p.M = a->M; p.K = a->K;
    p.rep = a->Hq / a->Hkv;
    p.d = a->d;
    p.q = a->q.ptr; p.k = a->k.ptr; p.v = a->v.ptr;
    p.qsb = a->q.sb; p.qsh = a->q.sh; p.qsn = a->q.sn;
    p.ksb = a->k.sb; p.ksh = a->k.sh; p.ksn = a->k.sn;
    p.vsb = a->v.sb; p.vsh = a->v.sh; p.vsn = a->v.sn;
    p.nb = a->neighbors; p.valid = a->valid; p.nb32 = a->neighbors32;
    p.row_inv = a->row_invalid;
    p.scale = a->scale; p.fp32w = a->fp32_weights;
    p.drop_p = a->dropout_p;
    // inverted dropout scales kept weights by 1 / (1 - p), the keep rate taken
    // in double and rounded to fp32 as torch's dropout divides its noise
    p.drop_scale = a->dropout_p > 0.f ? 1.f / (float)(1.0 - (double)a->dropout_p) : 1.f;
    p.seed = a->seed;
    p.out = a->out; p.osb = a->out_sb; p.osh = a->out_sh; p.osn = a->out_sn;
    p.rows = (int64_t)a->B * a->Hq * a->N;
    p.nblocks = ceil_div(p.rows, WAVES);
    return SSA_OK;
}

}  // namespace
