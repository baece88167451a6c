// ssa_graph_dense.h -- the graph build's dense form (included by ssa_graph.hip
// after its select helpers, inside its anonymous namespace).
//
// A query's candidates are the union of a few bucket lists.  With many lists
// over few keys (R x id sets x C of the order of M or more) the lists hold
// each key several times, and scoring, reading and deduplicating list members
// costs more than looking at every key once.  Then:
//
//   list_bits_kernel     each (kv head, round, bucket)'s members as a bitmap
//                        over the key ids, and the largest member
//   dense_mfma_kernel /  the code of every (query, key) score: a plain matrix
//   dense_valu_kernel    product, no lists
//   select_dense_kernel  a query's candidate set is the OR of its lists'
//                        bitmaps; the kk-th largest code under it is found by
//                        counting over the row's codes held in registers
//
// Scores, codes, exact keys and the tie rule are those of the list form
// (select_kernel), so both give the same graph.  Only FULL mode has this form:
// the LSH mode's output order follows the stream.

constexpr int DN_BLK = 128;            // keys per block of a score row
constexpr int DN_MAX_KEYS = 4096;      // keys a select row holds in registers
constexpr int DN_MAX_LISTS = 64;       // one lane per list
constexpr int DN_BITS_LDS = 65536;     // bytes of one round's bitmaps

// Score row of a query: Ms codes (M rounded up to DN_BLK, one block more where
// that is a multiple of 1,024 codes: rows a multiple of 2 KB apart would share
// few of the L2's channels), in 32-bit pairs:
// word 64 b + l holds keys 128 b + l (low half) and 128 b + 64 + l (high), so
// a wave's load of one word per lane brings two 64-key chunks in key order.
// Codes are clamped to at least 1; 0 marks a key that is no candidate.
struct DnP {
    const void *q, *k;
    int64_t qsb, qsh, qsn, ksb, ksh, ksn;
    uint32_t *S;           // (nbh * N, Ms / 2)
    const float *aux;      // MFMA: the query's code scale, last of NA floats
    // VALU: max |k|^2 per (batch, kv head), float bits, or the key hash's 16-row
    // maxima (kp_n per kv head)
    const uint32_t *knorm, *kpart;
    int kp_n;
    int NA;
    int N, M, Ms, Hq, Hkv, rep, bh0, nbh, causal, d;
    int qtiles, ktiles;    // workgroup tiles over queries and keys
};

// code of a score with at least 1: 65535 - min(neg code, 65534)
__device__ __forceinline__ uint32_t dn_neg(float s, float scale) {
    return (uint32_t)fminf(fmaxf(fmaf(-s, scale, 32767.f), 0.f), 65534.f);
}
__device__ __forceinline__ uint32_t dn_pair(float lo, float hi, float scale) {
    return ~(dn_neg(lo, scale) | (dn_neg(hi, scale) << 16));
}

// ---------------------------------------------------------------- bitmaps
struct LbP {
    const int32_t *perm, *bstart;
    const uint16_t *kid;
    uint64_t *bits;        // (rows, NB, nw)
    int32_t *lmax;         // (rows, NB) largest member, -1 without one
    int M, NB, C, R, nw;
    // the key hash's 16-row norm maxima, reduced per kv head (or null)
    const uint32_t *kpart;
    uint32_t *knorm;
    int kp_n;
};

// One workgroup per (kv head, round): the first C members of every bucket, in
// LDS, then written whole.  Latency bound (64 workgroups of 4 keys a thread at
// 4,096 keys).
__global__ void __launch_bounds__(1024) list_bits_kernel(LbP p) {
    extern __shared__ uint32_t lb_smem[];
    uint32_t *bits = lb_smem;                                // [NB * nw * 2]
    int32_t *mx = (int32_t *)(bits + (int64_t)p.NB * p.nw * 2);   // [NB]
    const int64_t row = blockIdx.x;
    const int nb2 = p.NB * p.nw * 2;
    for (int i = threadIdx.x; i < nb2; i += 1024) bits[i] = 0u;
    for (int i = threadIdx.x; i < p.NB; i += 1024) mx[i] = -1;
    __syncthreads();
    for (int i = threadIdx.x; i < p.M; i += 1024) {
        const int key = (int)SSA_IDX(p.perm[row * p.M + i], p.M, 12);
        const int u = (int)SSA_IDX(p.kid[row * p.M + key], p.NB, 13);
        if (i - p.bstart[row * p.NB + u] < p.C) {
            atomicOr(&bits[(u * p.nw + (key >> 6)) * 2 + ((key >> 5) & 1)], 1u << (key & 31));
            atomicMax(&mx[u], key);
        }
    }
    __syncthreads();
    uint32_t *out = (uint32_t *)(p.bits + row * p.NB * p.nw);
    for (int i = threadIdx.x; i < nb2; i += 1024) out[i] = bits[i];
    for (int i = threadIdx.x; i < p.NB; i += 1024) p.lmax[row * p.NB + i] = mx[i];
    if (p.kpart && row % p.R == 0 && threadIdx.x < SSA_WAVE) {
        const uint32_t *kt = p.kpart + row / p.R * p.kp_n;
        uint32_t m = 0u;
        for (int i = threadIdx.x; i < p.kp_n; i += SSA_WAVE) m = max(m, kt[i]);
        m = wave_max_u(m);
        if (threadIdx.x == 0) p.knorm[row / p.R] = m;
    }
}

// ---------------------------------------------------------------- scores
// 16-query operands per wave (QF): 4, or 2 where 4 leaves fewer than DM_TILES
// workgroups (64 x 2,048 queries over 512 keys, d = 64: 512 workgroups 69 us,
// 1,024 of half the queries 50 us).  Whole builds about the line, 4 / 2 operands:
// 512 workgroups of four 192 / 183 us (16 heads of 2,048, d = 64), 230 / 231 and 269 /
// 289 (64 heads of 1,024, d = 64 and 128); 1,024: 282 / 277 (32 heads of 2,048, d = 64)
constexpr int DM_QF = 4, DM_TILES = 1024;
constexpr int DM_K = 512;              // keys per workgroup: 4 blocks

// 16-bit q and k on the matrix cores, with the k steps, operand roles and so
// the sums of the list form's rescore.  A wave holds 16 QF queries as B operands
// and walks its keys in pairs of 16-row tiles 64 keys apart, whose results are
// the four 32-bit pairs a lane stores with one 16-byte store; the next pair's K
// rows load while this one multiplies.  K rows come straight from the L1 (the
// four waves walk the same rows).  Loads and stores of a wave retire in order,
// so a load issued behind a store waits for it: a block's stores go out together
// behind the next block's first loads.  Bound: the K fragments' way through the
// L1 (64 queries a wave instead of 32, which halves them: 95 -> 72 us at 16 heads
// of 2,999 causal rows, d = 96; 0.14 GB of codes).
template <typename T, int D, int QF>
__device__ __forceinline__ void dense_mfma_tile(const DnP &p, int64_t phys) {
    using V = typename Mfma16<T>::vec;
    constexpr int KS = (D + 31) / 32;
    const int64_t tiles = (int64_t)p.qtiles * p.ktiles;
    const int64_t blk = xcd_logical_block(phys, tiles * p.nbh);
    if (blk >= tiles * p.nbh) return;
    const int bhl = (int)(blk / tiles);
    const int t = (int)(blk % tiles);
    const int qt = t / p.ktiles, kt = t % p.ktiles;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / SSA_WAVE);
    const int n0 = qt * 64 * QF + 16 * QF * wid;
    const int k0 = kt * DM_K;
    // causal: keys up to the wave's last query
    int kend = min(k0 + DM_K, (p.M + DN_BLK - 1) / DN_BLK * DN_BLK);
    if (p.causal) kend = min(kend, (min(n0 + 16 * QF - 1, p.N - 1) / DN_BLK + 1) * DN_BLK);
    if (n0 >= p.N || k0 >= kend) return;
    const int bh = p.bh0 + bhl, b = bh / p.Hq, h = bh % p.Hq, g = h / p.rep;
    const int lane = lane_id(), li = lane % 16, lg = lane / 16;
    const T *qbase = (const T *)p.q + b * p.qsb + h * p.qsh;
    const T *kbase = (const T *)p.k + b * p.ksb + g * p.ksh;
    const V zero = __builtin_bit_cast(V, make_uint4(0, 0, 0, 0));
    V qf[QF][KS];
    float sc[QF];
#pragma unroll
    for (int i = 0; i < QF; ++i) {
        const int n = min(n0 + 16 * i + li, p.N - 1);
        sc[i] = p.aux[((int64_t)bhl * p.N + n) * p.NA + p.NA - 1];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int e0 = 32 * s + 8 * lg;
            const T *qe = qbase + (int64_t)n * p.qsn + e0;
            qf[i][s] = e0 < p.d ? __builtin_bit_cast(V, *reinterpret_cast<const uint4 *>(qe)) : zero;
        }
    }
    // A rows of the pair of tiles at key x: keys x + li and x + 64 + li
    auto load = [&](int x, V (&a)[2][KS]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const T *kr = kbase + (int64_t)min(x + 64 * i + li, p.M - 1) * p.ksn;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const int e0 = 32 * s + 8 * lg;
                a[i][s] = e0 < p.d ? __builtin_bit_cast(V, *reinterpret_cast<const uint4 *>(kr + e0)) : zero;
            }
        }
    };
    uint32_t *srow = p.S + ((int64_t)bhl * p.N + n0 + li) * (p.Ms / 2) + 4 * lg;
    uint4 w[4][QF];                     // the block's codes: tile pair, 16 queries
    auto score = [&](const V (&a)[2][KS], uint4 (&o)[QF]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < QF; ++i) {
            f32x4_t c0 = {0.f, 0.f, 0.f, 0.f}, c1 = c0;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                c0 = Mfma16<T>::mma(a[0][s], qf[i][s], c0);
                c1 = Mfma16<T>::mma(a[1][s], qf[i][s], c1);
            }
            // lane (li, lg): keys 4 lg + r (and 64 on) of the pair for query n0 + 16 i + li
            o[i] = make_uint4(dn_pair(c0[0], c1[0], sc[i]), dn_pair(c0[1], c1[1], sc[i]),
                              dn_pair(c0[2], c1[2], sc[i]), dn_pair(c0[3], c1[3], sc[i]));
        }
    };
    V a0[2][KS], a1[2][KS];
    load(k0, a0);
    for (int x = k0; x < kend; x += DN_BLK) {
        load(x + 16, a1);
        score(a0, w[0]);
        load(x + 32, a0);
        score(a1, w[1]);
        load(x + 48, a1);
        score(a0, w[2]);
        // the next block's first rows before this block's stores
        load(min(x + DN_BLK, kend - DN_BLK), a0);
        score(a1, w[3]);
#pragma unroll
        for (int i = 0; i < QF; ++i)
            if (n0 + 16 * i + li < p.N)
#pragma unroll
                for (int a = 0; a < 4; ++a)
                    *reinterpret_cast<uint4 *>(srow + (int64_t)16 * i * (p.Ms / 2) + x / 2 + 16 * a) = w[a][i];
    }
}

constexpr int DV_T = 128;              // queries and keys per workgroup tile
constexpr int DV_C = 32;               // head-dim columns staged at a time
constexpr int DV_LD = DV_T + 4;

// fp32 (and the 16-bit shapes the matrix-core form does not take): 128 x 128
// tiles, 8 queries x 8 keys per thread, each score one fmaf chain over the
// head dim in order, as the exact keys run it.  Bound: fp32 FMA issue (64 FMAs
// per four 16-byte LDS reads).
constexpr int DV_LDS = (2 * DV_C * DV_LD + DV_T) * 4;
template <typename T>
__device__ __forceinline__ void dense_valu_tile(const DnP &p, int64_t phys, float *lds) {
    float *Qs = lds, *Ks = Qs + DV_C * DV_LD, *q2s = Ks + DV_C * DV_LD;
    const int64_t tiles = (int64_t)p.qtiles * p.ktiles;
    const int64_t blk = xcd_logical_block(phys, tiles * p.nbh);
    if (blk >= tiles * p.nbh) return;
    const int bhl = (int)(blk / tiles);
    const int t = (int)(blk % tiles);
    const int n0 = t / p.ktiles * DV_T, k0 = t % p.ktiles * DV_T;
    if (p.causal && k0 > min(n0 + DV_T - 1, p.N - 1)) return;
    const int bh = p.bh0 + bhl, b = bh / p.Hq, h = bh % p.Hq, g = h / p.rep;
    const T *qbase = (const T *)p.q + b * p.qsb + h * p.qsh;
    const T *kbase = (const T *)p.k + b * p.ksb + g * p.ksh;
    const int tid = threadIdx.x, ty = tid / 16, tx = tid % 16;
    float acc[8][8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = 0.f;
    float q2 = 0.f;                    // thread r < 128: |q|^2 of query n0 + r
    for (int c0 = 0; c0 < p.d; c0 += DV_C) {
        const int cn = min(DV_C, p.d - c0);
        __syncthreads();
        // 128 rows x 32 columns of each: column tid % 32 of rows tid / 32 + 8 i
        for (int i = 0; i < DV_T / 8; ++i) {
            const int r = tid / DV_C + 8 * i, c = tid % DV_C;
            const bool in = c < cn;
            const int qn = min(n0 + r, p.N - 1), kn = min(k0 + r, p.M - 1);
            Qs[c * DV_LD + r] = in ? to_f32(qbase[(int64_t)qn * p.qsn + c0 + c]) : 0.f;
            Ks[c * DV_LD + r] = in ? to_f32(kbase[(int64_t)kn * p.ksn + c0 + c]) : 0.f;
        }
        __syncthreads();
        if (tid < DV_T)
            for (int c = 0; c < cn; ++c) q2 = fmaf(Qs[c * DV_LD + tid], Qs[c * DV_LD + tid], q2);
        for (int c = 0; c < cn; ++c) {
            const float4 qa = *reinterpret_cast<const float4 *>(&Qs[c * DV_LD + 8 * ty]);
            const float4 qb = *reinterpret_cast<const float4 *>(&Qs[c * DV_LD + 8 * ty + 4]);
            const float4 ka = *reinterpret_cast<const float4 *>(&Ks[c * DV_LD + 4 * tx]);
            const float4 kb = *reinterpret_cast<const float4 *>(&Ks[c * DV_LD + 64 + 4 * tx]);
            const float qv[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
            const float kv[8] = {ka.x, ka.y, ka.z, ka.w, kb.x, kb.y, kb.z, kb.w};
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[i][j] = fmaf(qv[i], kv[j], acc[i][j]);
        }
    }
    if (tid < DV_T) {
        uint32_t kn;
        if (p.kpart) {
            const uint32_t *kt = p.kpart + (int64_t)(b * p.Hkv + g) * p.kp_n;
            uint32_t m = 0u;
            for (int i = lane_id(); i < p.kp_n; i += SSA_WAVE) m = max(m, kt[i]);
            kn = wave_max_u(m);
        } else {
            kn = p.knorm[b * p.Hkv + g];
        }
        q2s[tid] = code_scale(q2, __uint_as_float(kn));
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int n = n0 + 8 * ty + i;
        if (n >= p.N) break;
        const float sc = q2s[8 * ty + i];
        uint4 w;
        w.x = dn_pair(acc[i][0], acc[i][4], sc);
        w.y = dn_pair(acc[i][1], acc[i][5], sc);
        w.z = dn_pair(acc[i][2], acc[i][6], sc);
        w.w = dn_pair(acc[i][3], acc[i][7], sc);
        *reinterpret_cast<uint4 *>(p.S + ((int64_t)bhl * p.N + n) * (p.Ms / 2) + k0 / 2 + 4 * tx) = w;
    }
}

// The score kernels alone (later head chunks), and the first chunk's beside the
// key sort's segments (the first nseg workgroups, a multiple of 8 so that the
// tiles keep their XCDs): the segments are a chain of dependent steps on a few
// CUs, and the scores need neither them nor what follows from them (segments 23
// us and scores 35 us one after the other, 45 us together, at 2 x 1,024 fp32 rows,
// 8 heads).
template <typename T, int D, int QF>
__global__ void __launch_bounds__(256) dense_mfma_kernel(DnP p, SortTopArgs s, int nseg) {
    extern __shared__ __align__(16) uint32_t dn_lds[];
    if ((int)blockIdx.x < nseg)
        sort_seg_blocks<uint16_t>(s.gkv, s.n, s.segs, s.segcount, s.perm, dn_lds, (int)blockIdx.x, nseg);
    else
        dense_mfma_tile<T, D, QF>(p, (int64_t)blockIdx.x - nseg);
}

template <typename T>
__global__ void __launch_bounds__(256) dense_valu_kernel(DnP p, SortTopArgs s, int nseg) {
    extern __shared__ __align__(16) uint32_t dn_lds[];
    if ((int)blockIdx.x < nseg)
        sort_seg_blocks<uint16_t>(s.gkv, s.n, s.segs, s.segcount, s.perm, dn_lds, (int)blockIdx.x, nseg);
    else
        dense_valu_tile<T>(p, (int64_t)blockIdx.x - nseg, (float *)dn_lds);
}

// ---------------------------------------------------------------- select
typedef uint16_t us2_t __attribute__((ext_vector_type(2)));

constexpr int DN_CAP = 256;            // boundary entries resolved in LDS
constexpr int DN_SCR = 2 * DN_CAP;     // LDS words of a row: their ids and exact keys

// x / d from magic = ceil(2^32 / d) (low 32 bits: 0 for d = 1): the high
// product is the quotient or one more
__device__ __forceinline__ uint32_t dn_div(uint32_t x, uint32_t d, uint32_t magic) {
    if (d == 1u) return x;
    const uint32_t q = __umulhi(x, magic);
    return q - (q * d > x ? 1u : 0u);
}

// the code scale of one query row, as dense_valu_kernel takes it
template <typename T>
__device__ float dn_row_scale(const SelP &p, int b, int h, int n) {
    const T *qr = (const T *)p.q + b * p.qsb + h * p.qsh + (int64_t)n * p.qsn;
    float q2 = 0.f;
    for (int c = 0; c < p.d; ++c) q2 = fmaf(to_f32(qr[c]), to_f32(qr[c]), q2);
    return code_scale(q2, __uint_as_float(p.knorm[b * p.Hkv + h / p.rep]));
}

// Blocks of a row are walked in groups of DN_GRP, the groups past its last
// block skipped (a causal row has half of them on average).
constexpr int DN_GRP = 4;
template <int NBK, class F>
__device__ __forceinline__ void dn_blocks(int nact, F &&f) {
#pragma unroll
    for (int b0 = 0; b0 < NBK; b0 += DN_GRP) {
        if (b0 == 0 || b0 < nact) {
#pragma unroll
            for (int b = b0; b < b0 + DN_GRP && b < NBK; ++b) f(b);
        }
    }
}

// codes at or above t (t >= 1) among the wave's packed pairs x[0, NBK)
template <int NBK>
__device__ __forceinline__ int dn_count(const uint32_t (&x)[NBK], int nact, uint32_t t) {
    const us2_t tm = {(uint16_t)(t - 1u), (uint16_t)(t - 1u)}, one = {1, 1};
    us2_t c = {0, 0};
    dn_blocks<NBK>(nact, [&](int b) __attribute__((always_inline)) {
        const us2_t v = __builtin_bit_cast(us2_t, x[b]);
        c += __builtin_elementwise_min(__builtin_elementwise_sub_sat(v, tm), one);
    });
    return __builtin_amdgcn_readlane(wave_incl_sum((int)c[0] + (int)c[1]), SSA_WAVE - 1);
}

// full_merge_emit for a selection held as 64-key words, one per lane: adds the
// window, the globals and the fallback key 0, removes the query and writes the
// union in ascending order, zero-padded.
__device__ __forceinline__ void dn_merge_emit(const SelP &p, uint64_t W, int n, int64_t row, int f) {
    const int lane = lane_id();
    const int nw = p.nw;
    if (lane >= nw) W = 0ull;
    if (!p.cross) {
        const int a = min(max(n - p.window, 0), p.M - 1) - 64 * lane;
        const int e = min(max(p.causal ? n : n + p.window, 0), p.M - 1) - 64 * lane;
        if (a < 64 && e >= 0)
            W |= (~0ull << max(a, 0)) & (~0ull >> (63 - min(e, 63)));
    }
    for (int j = 0; j < p.G; ++j) {
        const int v = (int)p.glob[j];
        if ((v >> 6) == lane) W |= 1ull << (v & 63);
    }
    if ((f > p.G ? f : p.G) < p.kk && lane == 0) W |= 1ull;
    const int self = p.cross ? 0 : 1;
    if (self && (n >> 6) == lane) W &= ~(1ull << (n & 63));
    const int ks = p.Kout - self;
    int total;
    const int pos = wave_excl_scan(__popcll(W), total);
    const int filled = total < ks ? total : ks;
    const int wlo = (int)(uint32_t)W, whi = (int)(uint32_t)(W >> 32);
    const int64_t o0 = SSA_IDX(row * p.Kout, p.rows_all * p.Kout, 4);
    int32_t *o32 = p.out_idx32 ? p.out_idx32 + o0 : nullptr;
    int64_t *o64 = p.out_idx + o0;
    uint8_t *ov = p.out_valid + o0;
    auto put = [&](int i, int v, bool valid) __attribute__((always_inline)) {
        if (o32) {
            o32[(uint32_t)i] = valid ? v : -1;
        } else {
            o64[(uint32_t)i] = valid ? (int64_t)v : 0;
            ov[(uint32_t)i] = valid ? 1 : 0;
        }
    };
    if (nw <= 8) {
        // few words: each word's keys straight to their slots
        for (int w = 0; w < nw; ++w) {
            const uint64_t m = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(whi, w) << 32) |
                               (uint32_t)__builtin_amdgcn_readlane(wlo, w);
            const int t = __builtin_amdgcn_readlane(pos, w) + lanes_below(m);
            if (in_mask(m) && t < ks) put(self + t, 64 * w + lane, true);
        }
    } else {
        // slot t: its word is the last one whose first slot is at or before t
        // (words without keys share their successor's)
        for (int t0 = 0; t0 < filled; t0 += SSA_WAVE) {
            const int t = t0 + lane;
            int w = 0;
#pragma unroll
            for (int step = 32; step > 0; step >>= 1) {
                const int ps = __shfl(pos, w + step, SSA_WAVE);
                if (ps <= t) w += step;
            }
            int r = t - __shfl(pos, w, SSA_WAVE);
            const uint32_t l = (uint32_t)__shfl(wlo, w, SSA_WAVE), h = (uint32_t)__shfl(whi, w, SSA_WAVE);
            const int c = __popc(l);
            const bool up = r >= c;
            r = up ? r - c : r;
            const int bit = nth_set_bit(up ? h : l, r) + (up ? 32 : 0);
            if (t < filled) put(self + t, 64 * w + bit, true);
        }
    }
    for (int i = self + filled + lane; i < p.Kout; i += SSA_WAVE) put(i, 0, false);
    if (self && lane == 0) put(0, n, true);
}

// One wavefront per query row (causal rows in descending position, as
// select_kernel).  NBK: blocks of 128 keys held, at least M / 128.
// What depends on the stream's order is settled as in select_kernel: the
// query's own key (earliest list holding a member at or past the query, or an
// overflow filler at or past it) and the overflow fillers (dropped unless a
// real occurrence precedes).
template <typename T, bool CAUSAL, int NBK>
__global__ void __launch_bounds__(SEL_WAVES * SSA_WAVE) select_dense_kernel(SelP p) {
    __shared__ uint32_t dn_scr[SEL_WAVES][DN_SCR];
    const int64_t blk = xcd_logical_block(blockIdx.x, p.nblocks);
    if (blk >= p.nblocks) return;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / SSA_WAVE);
    const int64_t rd = blk * SEL_WAVES + wid;
    if (rd >= p.rows) return;
    // row positions and heads by multiplication (the scalar unit has no divide)
    const uint32_t bhl = dn_div((uint32_t)rd, (uint32_t)p.N, p.magN);
    const int nr = (int)((uint32_t)rd - bhl * (uint32_t)p.N);
    const int n = CAUSAL ? p.N - 1 - nr : nr;
    const int64_t rloc = (int64_t)bhl * p.N + n;
    const int lane = lane_id();
    const int nl = p.nlists, nw = p.nw, kk = p.kk;
    uint32_t *scr = dn_scr[wid];
    const uint32_t bh = (uint32_t)p.bh0 + bhl;
    const int64_t row = (int64_t)p.bh0 * p.N + rloc;
    const int bq = (int)dn_div(bh, (uint32_t)p.Hq, p.magHq), hq = (int)bh - bq * p.Hq;
    const int prow0 = (int)dn_div(bh, (uint32_t)p.rep, p.magRep) * p.R;     // Hq = Hkv rep
    auto exact = [&](int v, bool want) {
        const T *qr = (const T *)p.q + bq * p.qsb + hq * p.qsh + (int64_t)n * p.qsn;
        const T *kb = (const T *)p.k + bq * p.ksb + (hq / p.rep) * p.ksh;
        return exact_keys<T>(p, qr, kb, v, want);
    };

    // ---- the row's codes, loaded while the candidate set is worked out
    const uint32_t *srow = p.S32 + rloc * (p.Ms / 2);
    int nact = CAUSAL ? n / DN_BLK + 1 : (p.M + DN_BLK - 1) / DN_BLK;   // blocks with scores
    uint32_t x[NBK];
#pragma unroll
    for (int b = 0; b < NBK; ++b) x[b] = 0u;
    dn_blocks<NBK>(nact, [&](int b) __attribute__((always_inline)) {
        if (b < nact) x[b] = srow[64 * b + lane];
    });

    // ---- lane l: list l
    const bool in = lane < nl;
    int li = 0, sz = 0, fk = 0, mx = -1;
    if (in) {
        const int r = (int)dn_div((uint32_t)lane, (uint32_t)p.NS, p.magNS);
        li = (prow0 + r) * p.NB + (int)SSA_IDX(p.qid[row * nl + lane], p.NB, 14);
        sz = p.bsize[li];
        mx = p.lmax[li];
        fk = p.perm[(int64_t)(prow0 + r) * p.M + p.M - 1];
    }
    const bool any_empty = wave_ballot(in && sz == 0) != 0ull;
    const int gl = min(p.G, p.C);
    // v is an entry of glob ++ 0 (all of them valid)
    auto in_glob = [&](int v) {
        bool hit = v == 0 && p.G < p.C;
        for (int j = 0; j < gl; ++j) hit |= (int)p.glob[j] == v;
        return hit;
    };
    bool nkeep = false;
    if (CAUSAL) {
        const bool gown = any_empty && in_glob(n);
        const bool real = sz > 0 ? mx >= n : gown;
        const uint64_t fm = wave_ballot(in && (real || (sz > 0 && sz < p.C && fk >= n)));
        if (fm) nkeep = (wave_ballot(real) >> (__ffsll((long long)fm) - 1)) & 1ull;
    }

    // ---- candidate words: lane w (mod nwp) holds keys 64 w .. 64 w + 63
    int nwp = 1;
    while (nwp < nw) nwp <<= 1;
    const int word = lane & (nwp - 1);
    const int per = SSA_WAVE / nwp;                    // lists per load
    uint64_t W = 0ull;
    auto list_word = [&](int l0) __attribute__((always_inline)) {
        const int l = l0 + lane / nwp;
        const int i = __shfl(li, l & (SSA_WAVE - 1), SSA_WAVE);
        return (l < nl && word < nw) ? p.lbits[(uint32_t)(i * nw + word)] : 0ull;
    };
    int l0 = 0;
    for (; l0 + 3 * per < nl; l0 += 4 * per) {
        const uint64_t w0 = list_word(l0), w1 = list_word(l0 + per), w2 = list_word(l0 + 2 * per),
                       w3 = list_word(l0 + 3 * per);
        W |= (w0 | w1) | (w2 | w3);
    }
    for (; l0 < nl; l0 += per) W |= list_word(l0);
    for (int o = nwp; o < SSA_WAVE; o <<= 1) W |= __shfl_xor((unsigned long long)W, o, SSA_WAVE);
    if (CAUSAL) {
        // members below the query
        const int below = n - 64 * word;
        W &= below >= 64 ? ~0ull : below <= 0 ? 0ull : (1ull << below) - 1ull;
    }
    if (any_empty) {
        const int nge = min(p.G + 1, p.C);
        const int nsc = nact;
        for (int j = 0; j < nge; ++j) {
            const int v = j < p.G ? (int)p.glob[j] : 0;
            if (CAUSAL && v == n) continue;            // settled
            if ((v >> 6) == word) W |= 1ull << (v & 63);
            if (CAUSAL && v / DN_BLK >= nsc) {
                nact = max(nact, v / DN_BLK + 1);
                // past the row's scored blocks: its code from its exact key
                const uint32_t key = (uint32_t)__builtin_amdgcn_readfirstlane((int)exact(v, lane == 0));
                const float sc = p.aux ? p.aux[rloc * p.NA + p.NA - 1] : dn_row_scale<T>(p, bq, hq, n);
                const uint32_t code = 65535u - dn_neg(key_score(key), sc);
                const int sh = (v & 64) ? 16 : 0;
#pragma unroll
                for (int b = 0; b < NBK; ++b)
                    if (b == v / DN_BLK && lane == (v & 63)) x[b] = (x[b] & ~(0xffffu << sh)) | (code << sh);
            }
        }
    }
    // overflow fillers below the query: dropped unless a real occurrence (or an
    // earlier list's filler of the same key, already dropped) comes first
    const bool fl = in && sz > 0 && sz < p.C && (!CAUSAL || fk < n);
    if (wave_ballot(fl)) {
        const int fv = fl ? fk : -1;
        if (lane < 2) scr[lane] = 0u;
        wave_lds_sync();
        const int np = nl * nl;
        for (int p0 = 0; p0 < np; p0 += SSA_WAVE) {
            const int pi = p0 + lane;
            const int L = min((int)__umulhi((uint32_t)pi, p.nl_magic), nl - 1);
            const int L2 = nl > 1 ? pi - L * nl : 0;
            const int v = __shfl(fv, L, SSA_WAVE);
            const int s2 = __shfl(sz, L2, SSA_WAVE), v2 = __shfl(fv, L2, SSA_WAVE);
            const int i2 = __shfl(li, L2, SSA_WAVE);
            if (pi < np && L2 <= L && v >= 0) {
                bool hit;
                if (s2 == 0) hit = in_glob(v);
                else
                    hit = (L2 < L && v2 == v) ||
                          ((p.lbits[(int64_t)i2 * nw + (SSA_IDX(v, p.M, 15) >> 6)] >> (v & 63)) & 1ull);
                if (hit) atomicOr(&scr[L >> 5], 1u << (L & 31));
            }
        }
        wave_lds_sync();
        uint64_t mark = wave_ballot(fl && !((scr[lane >> 5] >> (lane & 31)) & 1u));
        while (mark) {
            const int L = __ffsll((long long)mark) - 1;
            mark &= mark - 1ull;
            const int v = __builtin_amdgcn_readlane(fv, L);
            if ((v >> 6) == word) W &= ~(1ull << (v & 63));
        }
    }
    if (nkeep && (n >> 6) == word) W |= 1ull << (n & 63);
    const int nk = __builtin_amdgcn_readlane(wave_incl_sum(lane < nwp ? __popcll(W) : 0), SSA_WAVE - 1);

    if (nk > kk) {
        // ---- codes of the candidates only
        const int wlo = (int)(uint32_t)W, whi = (int)(uint32_t)(W >> 32);
        auto chunk = [&](int c) {                      // candidates among keys 64 c ..
            return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(whi, c & 63) << 32) |
                   (uint32_t)__builtin_amdgcn_readlane(wlo, c & 63);
        };
        us2_t tp = {0, 0};
        uint32_t s1 = 0u, s2 = 0u;                     // sums of codes, of (code / 128)^2
        dn_blocks<NBK>(nact, [&](int b) __attribute__((always_inline)) {
            const uint32_t m = (in_mask(2 * b < nwp ? chunk(2 * b) : 0ull) ? 0xffffu : 0u) |
                               (in_mask(2 * b + 1 < nwp ? chunk(2 * b + 1) : 0ull) ? 0xffff0000u : 0u);
            x[b] &= m;
            const us2_t v = __builtin_bit_cast(us2_t, x[b]), one = {1, 1};
            tp = __builtin_elementwise_max(tp, v);
            s1 = __builtin_amdgcn_udot2(v, one, s1, false);
            s2 = __builtin_amdgcn_udot2(v >> 7, v >> 7, s2, false);
        });
        const uint32_t top = max((uint32_t)tp[0], (uint32_t)tp[1]);
        // ---- kk-th largest: count(lo) >= kk > count(hi).  The first probe is
        // the place a normal distribution of the codes' mean and deviation has
        // its kk-th of nk, the next two step from the last count along that
        // distribution's tail, further ones interpolate the counts and, every
        // third, take the middle: 4 probes on normal scores, where bisection
        // takes 10.
        uint32_t lo = 1u, hi = wave_max_u(top) + 1u;
        int clo = nk, chi = 0;
        const float rn = __builtin_amdgcn_rcpf((float)nk);
        const float mean = (float)__builtin_amdgcn_readlane(wave_incl_sum((int)s1), SSA_WAVE - 1) * rn;
        const float m2 = (float)(uint32_t)__builtin_amdgcn_readlane(wave_incl_sum((int)s2), SSA_WAVE - 1) * rn;
        const float var = fmaxf(m2 - mean * mean * (1.f / 16384.f), 0.0625f);
        const float sd = 128.f * __builtin_amdgcn_sqrtf(var);
        // quantile (Tukey's lambda form) and hazard at the tail share kk / nk
        const float pk = (float)kk * rn;
        const float zq = (__builtin_amdgcn_exp2f(0.135f * __builtin_amdgcn_logf(1.f - pk)) -
                          __builtin_amdgcn_exp2f(0.135f * __builtin_amdgcn_logf(pk))) * 5.0633f;
        const float lk = __builtin_amdgcn_logf((float)kk);
        // sd / hazard, times ln 2 for counts in log2
        const float step = sd * 0.6931f * pk * 2.5066f * __builtin_amdgcn_exp2f(0.7213f * zq * zq);
        float at = mean + sd * zq;
        for (int it = 0; hi - lo > 1u && clo != kk; ++it) {
            if (it > 2) {
                at = it % 3 == 2 ? 0.5f * ((float)lo + (float)hi)
                                 : (float)lo + (float)(hi - lo) * ((float)(clo - kk) + 0.25f) *
                                                   __builtin_amdgcn_rcpf((float)(clo - chi));
            }
            uint32_t t = (uint32_t)fminf(fmaxf(at, (float)(lo + 1u)), (float)(hi - 1u));
            t = (uint32_t)__builtin_amdgcn_readfirstlane((int)t);
            const int c = dn_count<NBK>(x, nact, t);
            at = (float)t + (__builtin_amdgcn_logf(fmaxf((float)c, 0.5f)) - lk) * step;
            if (c >= kk) { lo = t; clo = c; }
            else { hi = t; chi = c; }
        }
        // codes >= lo when that is exactly kk; else those >= hi and `need` of
        // the code lo
        const bool tied = clo != kk;
        const uint32_t cut = tied ? hi : lo;
        uint64_t sel = 0ull, eq = 0ull;
        dn_blocks<NBK>(nact, [&](int b) __attribute__((always_inline)) {
            const uint64_t s0 = wave_ballot((x[b] & 0xffffu) >= cut), s1 = wave_ballot((x[b] >> 16) >= cut);
            if (lane == 2 * b) sel = s0;
            if (lane == 2 * b + 1) sel = s1;
        });
        if (tied) {
            int need = kk - chi;
            bool btie = false;
            dn_blocks<NBK>(nact, [&](int b) __attribute__((always_inline)) {
                const uint64_t e0 = wave_ballot((x[b] & 0xffffu) == lo), e1 = wave_ballot((x[b] >> 16) == lo);
                if (lane == 2 * b) eq = e0;
                if (lane == 2 * b + 1) eq = e1;
            });
            const int elo = (int)(uint32_t)eq, ehi = (int)(uint32_t)(eq >> 32);
            auto echunk = [&](int c) {
                return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(ehi, c) << 32) |
                       (uint32_t)__builtin_amdgcn_readlane(elo, c);
            };
            uint64_t nz = wave_ballot(eq != 0ull);
            if (clo - chi <= DN_CAP) {
                // their exact keys in LDS decide
                uint32_t *ids = scr, *keys = scr + DN_CAP;
                int ne = 0;
                for (uint64_t z = nz; z; z &= z - 1ull) {
                    const int c = __ffsll((long long)z) - 1;
                    const uint64_t m = echunk(c);
                    const int at = ne + lanes_below(m);
                    if (in_mask(m) && at < DN_CAP) ids[at] = (uint32_t)(64 * c + lane);
                    ne = min(ne + __popcll(m), DN_CAP);
                }
                wave_lds_sync();
                uint32_t kv[DN_CAP / SSA_WAVE];
                uint32_t kmx = 0u, kmn = 0xffffffffu;
#pragma unroll
                for (int i = 0; i < DN_CAP / SSA_WAVE; ++i) {
                    kv[i] = 0u;
                    const int e = i * SSA_WAVE + lane;
                    if (i * SSA_WAVE < ne) {
                        const bool w = e < ne;
                        const uint32_t k = exact(w ? (int)ids[e] : 0, w);
                        kv[i] = w ? k : 0u;
                        if (w) keys[e] = k;
                    }
                    kmx = max(kmx, kv[i]);
                    kmn = kv[i] != 0u ? min(kmn, kv[i]) : kmn;
                }
                const uint32_t thr = kth_search(kv, need, wave_min_u(kmn), wave_max_u(kmx), 0);
                int gt = 0, ge = 0;
#pragma unroll
                for (int i = 0; i < DN_CAP / SSA_WAVE; ++i) {
                    gt += __popcll(wave_ballot(kv[i] > thr));
                    ge += __popcll(wave_ballot(kv[i] >= thr));
                }
                btie = ge > need;
                wave_lds_sync();
                // above thr: all; equal: the first in key order until need are taken
                int left = need - gt;
                for (int e = 0; e < ne; ++e) {
                    const uint32_t k = keys[e];
                    const int v = (int)ids[e];
                    const bool take = k > thr || (k == thr && left > 0);
                    if (k == thr) --left;
                    if (take && lane == (v >> 6)) sel |= 1ull << (v & 63);
                }
            } else {
                // many candidates of one code: their exact keys again in every
                // pass, chunk by chunk
                uint32_t kmx = 0u, kmn = 0xffffffffu;
                for (uint64_t z = nz; z; z &= z - 1ull) {
                    const int c = __ffsll((long long)z) - 1;
                    const bool w = in_mask(echunk(c));
                    const uint32_t k = exact(64 * c + lane, w);
                    kmx = max(kmx, k);
                    kmn = w ? min(kmn, k) : kmn;
                }
                kmx = wave_max_u(kmx);
                kmn = wave_min_u(kmn);
                uint32_t thr = kmn;
                if (kmn < kmx) {
                    const int hb = 31 - __clz(kmn ^ kmx);
                    thr = hb >= 31 ? 0u : (kmn & ~((2u << hb) - 1u));
                    for (int bit = hb; bit >= 0; --bit) {
                        const uint32_t cand = thr | (1u << bit);
                        int c2 = 0;
                        for (uint64_t z = nz; z; z &= z - 1ull) {
                            const int c = __ffsll((long long)z) - 1;
                            const bool w = in_mask(echunk(c));
                            const uint32_t k = exact(64 * c + lane, w);
                            c2 += __popcll(wave_ballot(w && k >= cand));
                        }
                        if (c2 >= need) thr = cand;
                    }
                }
                int gt = 0, ge = 0;
                uint64_t sgt = 0ull, seq = 0ull;
                for (uint64_t z = nz; z; z &= z - 1ull) {
                    const int c = __ffsll((long long)z) - 1;
                    const bool w = in_mask(echunk(c));
                    const uint32_t k = exact(64 * c + lane, w);
                    const uint64_t mg = wave_ballot(w && k > thr), me = wave_ballot(w && k == thr);
                    gt += __popcll(mg);
                    ge += __popcll(mg | me);
                    if (lane == c) { sgt = mg; seq = me; }
                }
                btie = ge > need;
                // of the equal ones, the first in key order
                int left = need - gt;
                const int before = wave_incl_sum(__popcll(seq)) - __popcll(seq);
                uint64_t take = 0ull, rest = seq;
                for (int i = before; i < left && rest; ++i) {
                    take |= rest & (~rest + 1ull);
                    rest &= rest - 1ull;
                }
                sel |= sgt | take;
            }
            // a tied kk-th score: the exact replay decides
            if (btie && lane == 0) {
                if (p.ties) atomicAdd(p.ties, 1);
                if (p.tie_list) p.tie_list[atomicAdd(p.tie_count, 1)] = (int)row;
            }
        }
        W = sel;
    }
    dn_merge_emit(p, W, n, row, nk < kk ? nk : kk);
}
