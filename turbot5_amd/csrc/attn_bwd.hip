// Backward of the dense fused-bias attention forward for gfx950: dq, dk, dv and the gradient of the
// (num_buckets, H) bias table.  Replaces flash_attn_v2_bwd_bias of the reference
// (src/turbot5/ops/fused_bias_attention.py:397-820: _bwd_preprocess, _bwd_kv_bias_kernel with its atomics on the
// table gradient :617-619, _bwd_q_kernel).
//
// The general kernels do all arithmetic in fp32 (inputs of any of the three types are widened on their
// way into LDS; the products run on the fp32 matrix cores, v_mfma_f32_32x32x2_f32), so one code path serves fp32 and
// 16-bit tensors at head_dim 16, 32 and 64; 16-bit tensors at head_dim 64 and 128 have kernels of their own on the 16-bit
// matrix cores (bwd16_kernel, further down), and fp32 tensors at head_dim 64 theirs (attn_f32.hip), unless the caller asks
// for products on the fp32 matrix cores.  The general kernels:
//
//   bwd_rows_kernel   delta_i = sum_d o_id do_id and the log-sum-exp in base-2 units, per query row, both negated; also
//                     clears the table gradient
//   bwd_kernel<KV=0>  a workgroup owns 64 query rows (32 per wavefront) and walks the key tiles of 64 (32 of the 64 per
//                     wavefront): S^T = K Q^T, dP^T = V dO^T (key rows from LDS as the A operand, so a lane owns one
//                     query and its log-sum-exp and delta are lane scalars), P^T = exp2(c1 S^T + bias - lse),
//                     dS^T = P^T (dP^T - delta), dQ^T += K^T dS^T.  The table gradient is collected here: blocks whose
//                     distances are all saturated add their dS to one of two lane sums, the blocks around the
//                     diagonal are summed per distance through LDS; distances go to buckets at the end, and one
//                     global atomic per bucket and workgroup to the table.
//   bwd_kernel<KV=1>  a workgroup owns 64 keys and walks the query tiles of 64, the same products with the roles
//                     swapped (query rows from LDS; log-sum-exp and delta of the 64 queries staged in LDS):
//                     dV^T += dO^T P, dK^T += Q^T dS.
//
// With cu_seqlens the same kernels run a packed batch (varlen_fused_bias_attn.py:407-800): a workgroup looks up its
// sequence's first row and length and works on that sequence; the grid is sized for the longest one.
// Scores use the key position j and the query position i + N - M, as the forward does; rows whose log-sum-exp is
// -inf (no visible key) have no gradient.  Rows and keys past the end of a tensor are read as zeros and masked.
#include "lut_device.h"
#include "mfma16_device.h"
#include "t5a_internal.h"
#include "table_grad_device.h"

namespace t5a {

namespace {


constexpr int kBwdThreads = 256;
constexpr int kBwdOwn = 64;      // own rows per workgroup of the fp32 kernels (queries for dq, keys for dk / dv)
constexpr int kBwdOther = 64;    // rows of the other kind per tile
constexpr int kMaxBuckets = 4 * kMaxThresholds;     // of a table; the dq pass sums them in the memory of its tiles

template <typename T> __device__ __forceinline__ float to_f32(T x) { return static_cast<float>(x); }

// four consecutive elements of a row as floats (8 or 16 bytes, aligned: head_dim and strides are multiples of 8 / 4)
template <typename T> __device__ __forceinline__ f32x4 load4(const T* p) {
    if constexpr (sizeof(T) == 4) {
        return *reinterpret_cast<const f32x4*>(p);
    } else {
        typedef T t4 __attribute__((ext_vector_type(4)));
        const t4 x = *reinterpret_cast<const t4*>(p);
        return f32x4{to_f32(x[0]), to_f32(x[1]), to_f32(x[2]), to_f32(x[3])};
    }
}
template <typename T> __device__ __forceinline__ void store4(T* p, f32x4 x) {
    if constexpr (sizeof(T) == 4) {
        *reinterpret_cast<f32x4*>(p) = x;
    } else {
        typedef T t4 __attribute__((ext_vector_type(4)));
        *reinterpret_cast<t4*>(p) = t4{(T)x[0], (T)x[1], (T)x[2], (T)x[3]};
    }
}

// rows per block of bwd_rows_kernel: up to eight threads share a row, 16 bytes per load, so that a wavefront's loads
// cover whole rows (one thread per row reads with a stride of a row and takes twice as long)
template <typename T, int D> struct RowsGeom {
    static constexpr int CH = D * (int)sizeof(T) / 16;      // 16-byte chunks per row
    static constexpr int TPR = CH < 8 ? CH : 8;             // threads per row
    static constexpr int CPT = CH / TPR;                    // chunks per thread
    static constexpr int ROWS = 256 / TPR;                  // rows per block
    static constexpr int EPC = 16 / (int)sizeof(T);         // elements per chunk
};

template <typename T, int D>
__global__ __launch_bounds__(256) void bwd_rows_kernel(const BwdParams p) {
    using G = RowsGeom<T, D>;
    // dense: row = (b, h, i) flattened, statistics (B,H,M); packed: row = (token, h) flattened, statistics (total_q, H)
    const int sub = threadIdx.x % G::TPR;
    const int64_t row = (int64_t)blockIdx.x * G::ROWS + threadIdx.x / G::TPR;
    const bool packed = p.cu_q != nullptr;
    const int64_t rows = packed ? (int64_t)p.total_q * p.H : (int64_t)p.B * p.H * p.M;
    // the table gradient is accumulated with atomics by the dq kernel: clear it here, ahead of that launch
    if (p.dtable != nullptr) {
        const int64_t n = (int64_t)p.n_buckets * p.H;
        for (int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x; x < n; x += (int64_t)gridDim.x * 256) p.dtable[x] = 0.f;
    }
    float acc = 0.f;
    if (row < rows) {
        int64_t o_off, g_off;
        if (packed) {
            const int64_t tok = row / p.H;
            const int h = (int)(row - tok * p.H);
            o_off = tok * p.o_sr + (int64_t)h * p.o_sh;
            g_off = tok * p.do_sr + (int64_t)h * p.do_sh;
        } else {
            const int i = (int)(row % p.M);
            const int64_t bh = row / p.M;
            const int h = (int)(bh % p.H), b = (int)(bh / p.H);
            o_off = (int64_t)b * p.o_sb + (int64_t)h * p.o_sh + (int64_t)i * p.o_sr;
            g_off = (int64_t)b * p.do_sb + (int64_t)h * p.do_sh + (int64_t)i * p.do_sr;
        }
        const T* o = reinterpret_cast<const T*>(p.o) + o_off;
        const T* g = reinterpret_cast<const T*>(p.dout) + g_off;
#pragma unroll
        for (int c = 0; c < G::CPT; ++c)
#pragma unroll
            for (int q4 = 0; q4 < G::EPC / 4; ++q4) {
                const int at = (sub * G::CPT + c) * G::EPC + 4 * q4;
                const f32x4 x = load4(o + at), y = load4(g + at);
                acc += x[0] * y[0] + x[1] * y[1] + x[2] * y[2] + x[3] * y[3];
            }
    }
    // (every lane takes part in the exchange; the threads of a row are neighbours in one wavefront)
#pragma unroll
    for (int off = 1; off < G::TPR; off <<= 1) acc += __shfl_xor(acc, off, 64);
    if (row >= rows || sub != 0) return;
    p.delta[row] = -acc;     // negated: it is the start value of the dP accumulators
    const float l = p.lse[row];
    // negated as well; a row without a visible key: -inf makes every exp2(score + lse2) of the row 0
    p.lse2[row] = l == -INFINITY ? -INFINITY : l * -1.4426950408889634f;
}

// A workgroup owns 64 rows and walks tiles of 64, whose halves go to different wavefronts; their partial gradients are
// added through LDS at the end.  One 32 x 32 block of scores per wavefront leaves registers to fetch the next tile's rows
// under the current tile's products.  The fp32 matrix cores (64 cycles per product) bound it.  128 own rows and no
// prefetch took, with every table-gradient pair added to LDS by an atomic, 259 us where this takes 135 (fp32, B4 H8 L512 D64, the
// three kernels: 64-row blocks fill 256 compute units, 128-row blocks half of them), 674 / 515 at B4 H12 L1024 and
// 1210 / 925 at B8 H12 L1024; without the atomics 219, 615 and 1004, so the small blocks are the better at every size.
template <typename T, int D, bool CAUSAL, bool KV>
__global__ __launch_bounds__(kBwdThreads, 2) void bwd_kernel(const BwdParams p) {
    constexpr int STR = D + 1;              // fp32 tile rows padded by one float
    constexpr int DT = (D + 31) / 32;       // 32-row blocks of the transposed gradients
    constexpr int KS = D / 2;               // k-steps of a product over head_dim
    constexpr int OWNW = kBwdOwn / 32;
    constexpr int TILE = kBwdOther * STR + 32;
    constexpr int RED = OWNW * (KV ? 2 : 1) * DT * 16 * 64;
    constexpr int SKEW_ROWS = 8;
    static_assert(2 * TILE >= kMaxBuckets, "");
    __shared__ float tiles[2 * TILE > RED ? 2 * TILE : RED];
    float* const ta = tiles;               // K (dq) / Q (dk, dv) tile
    float* const tb = tiles + TILE;        // V (dq) / dO (dk, dv) tile
    __shared__ float rowstat[2 * kBwdOther];       // KV: lse2 and delta of the tile's queries
    __shared__ float lut_bias[2 * kMaxSaturation + 1];   // bias * log2(e) per clamped distance
    __shared__ float hist_rel[KV ? 1 : 2 * kMaxSaturation + 1];   // dS summed per clamped distance
    __shared__ float skew_all[KV ? 1 : 4 * SKEW_ROWS * 64];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 31, hh = lane >> 5;
    const int h = blockIdx.y, b = blockIdx.z;
    const int own_base = blockIdx.x * kBwdOwn;
    const int w_lo = own_base + (wave % OWNW) * 32, own_row = w_lo + lr;
    const int sub0 = (wave / OWNW) * 32;      // first tile row of this wavefront's block
    float* const skew = skew_all + (KV ? 0 : wave * SKEW_ROWS * 64);
    // packed batch: sequence b is the rows [cu[b], cu[b] + len) of the (total, H, D) tensors (len from seq_lens when
    // given, else up to cu[b + 1]); the batch strides are 0 and everything below works on that sequence
    int M = p.M, N = p.N;
    int64_t q_first = 0, k_first = 0;
    if (p.cu_q != nullptr) {
        q_first = p.cu_q[b]; k_first = p.cu_k[b];
        M = p.len_q != nullptr ? p.len_q[b] : p.cu_q[b + 1] - (int)q_first;
        N = p.len_k != nullptr ? p.len_k[b] : p.cu_k[b + 1] - (int)k_first;
        if (own_base >= (KV ? N : M)) return;     // (the grid is sized for the longest sequence)
    }
    const int n_own = KV ? N : M, n_other = KV ? M : N;
    const int P = N - M;                           // query i sits at key position i + P
    const bool has_bias = p.table != nullptr;
    const int sat = has_bias ? p.bs.sat : 0;

    const T* qp = reinterpret_cast<const T*>(p.q) + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh + q_first * p.q_sr;
    const T* kp = reinterpret_cast<const T*>(p.k) + (int64_t)b * p.k_sb + (int64_t)h * p.k_sh + k_first * p.k_sr;
    const T* vp = reinterpret_cast<const T*>(p.v) + (int64_t)b * p.v_sb + (int64_t)h * p.v_sh + k_first * p.v_sr;
    const T* gp = reinterpret_cast<const T*>(p.dout) + (int64_t)b * p.do_sb + (int64_t)h * p.do_sh + q_first * p.do_sr;
    // statistics of query i: index stat_base + i * stat_sr
    const int64_t stat_sr = p.cu_q != nullptr ? p.H : 1;
    const int64_t stat_base = p.cu_q != nullptr ? q_first * p.H + h : ((int64_t)b * p.H + h) * p.M;

    // bias (and bucket) per clamped distance
    if (has_bias) {
        for (int x = tid; x <= 2 * sat; x += kBwdThreads) {
            const int bk = bucket_of(p.bs, x - sat);
            lut_bias[x] = load_table(p.table, p.table_dtype, (int64_t)bk * p.t_sbucket + (int64_t)h * p.t_shead) * 1.4426950408889634f;
            if constexpr (!KV) hist_rel[x] = 0.f;
        }
        if constexpr (!KV)
            for (int x = lane; x < SKEW_ROWS * 64; x += 64) skew[x] = 0.f;
    }

    // own rows as B operands of the 32x32x2 products: lane (lr, hh) holds elements 2s + hh of its row
    const bool own_ok = own_row < n_own;
    float fa[KS], fb[KS];
    {
        const T* a = (KV ? kp + (int64_t)own_row * p.k_sr : qp + (int64_t)own_row * p.q_sr);
        const T* c = (KV ? vp + (int64_t)own_row * p.v_sr : gp + (int64_t)own_row * p.do_sr);
#pragma unroll
        for (int s4 = 0; s4 < D / 4; ++s4) {
            f32x4 x = {0.f, 0.f, 0.f, 0.f}, y = {0.f, 0.f, 0.f, 0.f};
            if (own_ok) { x = load4(a + 4 * s4); y = load4(c + 4 * s4); }
            fa[2 * s4] = hh ? x[1] : x[0]; fa[2 * s4 + 1] = hh ? x[3] : x[2];
            fb[2 * s4] = hh ? y[1] : y[0]; fb[2 * s4 + 1] = hh ? y[3] : y[2];
        }
    }
    float lse2_own = -INFINITY, delta_own = 0.f;
    if (!KV && own_ok) { lse2_own = p.lse2[stat_base + own_row * stat_sr]; delta_own = p.delta[stat_base + own_row * stat_sr]; }

    // tiles of the other kind that can hold a visible pair
    int t_lo = 0, t_hi = (n_other + kBwdOther - 1) / kBwdOther;
    if (CAUSAL) {
        if (!KV) t_hi = min(t_hi, max(0, (own_base + kBwdOwn - 1 + P) / kBwdOther + 1));   // keys j <= i + P
        else t_lo = max(0, own_base - P) / kBwdOther;                                      // queries i >= j - P
    }

    f32x16 acc_a[DT], acc_b[DT];     // dQ^T or dK^T; dV^T
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) { acc_a[dt][r] = 0.f; acc_b[dt][r] = 0.f; }
    float sum_lo = 0.f, sum_hi = 0.f;   // dS of the tiles saturated on the left / on the right of the diagonal

    // staging: thread -> 16-byte (of fp32) chunks of both tiles' rows, and with KV one row statistic
    constexpr int CHUNKS = kBwdOther * (D / 4) / kBwdThreads;
    f32x4 xa[CHUNKS], xb[CHUNKS];
    float stat = 0.f;
    auto fetch = [&](int o0) {
        const T* a = KV ? qp : kp;
        const T* c = KV ? gp : vp;
        const int64_t a_sr = KV ? p.q_sr : p.k_sr, c_sr = KV ? p.do_sr : p.v_sr;
#pragma unroll
        for (int n = 0; n < CHUNKS; ++n) {
            const int idx = tid + n * kBwdThreads, row = idx / (D / 4), c4 = idx % (D / 4);
            xa[n] = f32x4{0.f, 0.f, 0.f, 0.f}; xb[n] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (o0 + row < n_other) {
                xa[n] = load4(a + (int64_t)(o0 + row) * a_sr + 4 * c4);
                xb[n] = load4(c + (int64_t)(o0 + row) * c_sr + 4 * c4);
            }
        }
        if (KV && tid < 2 * kBwdOther) {
            const int row = tid & (kBwdOther - 1);
            stat = tid < kBwdOther ? -INFINITY : 0.f;
            if (o0 + row < n_other)
                stat = tid < kBwdOther ? p.lse2[stat_base + (o0 + row) * stat_sr] : p.delta[stat_base + (o0 + row) * stat_sr];
        }
    };
    if (t_lo < t_hi) fetch(t_lo * kBwdOther);

    for (int t = t_lo; t < t_hi; ++t) {
        const int o0 = t * kBwdOther;
        __syncthreads();     // the previous tile's readers are done (and the LUT is written, first time round)
#pragma unroll
        for (int n = 0; n < CHUNKS; ++n) {
            const int idx = tid + n * kBwdThreads, row = idx / (D / 4), c4 = idx % (D / 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) { ta[row * STR + 4 * c4 + e] = xa[n][e]; tb[row * STR + 4 * c4 + e] = xb[n][e]; }
        }
        if (KV && tid < 2 * kBwdOther) rowstat[tid] = stat;
        __syncthreads();
        if (t + 1 < t_hi) fetch(o0 + kBwdOther);

        f32x16 s, dp;
#pragma unroll
        for (int r = 0; r < 16; ++r) { s[r] = 0.f; dp[r] = 0.f; }
        const float* const row_a = ta + (sub0 + lr) * STR + hh;
        const float* const row_b = tb + (sub0 + lr) * STR + hh;
#pragma unroll
        for (int k2 = 0; k2 < KS; ++k2) {
            s = __builtin_amdgcn_mfma_f32_32x32x2f32(row_a[2 * k2], fa[k2], s, 0, 0, 0);
            dp = __builtin_amdgcn_mfma_f32_32x32x2f32(row_b[2 * k2], fb[k2], dp, 0, 0, 0);
        }

        float tile_sum = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int ol = sub0 + 8 * (r >> 2) + 4 * hh + (r & 3);   // row of the other kind inside the tile
            const int i = KV ? o0 + ol : own_row, j = KV ? own_row : o0 + ol;
            const int rel = j - (i + P);
            const bool valid = i < M && j < N && (!CAUSAL || rel <= 0);
            const float bias2 = has_bias ? lut_bias[min(max(rel, -sat), sat) + sat] : 0.f;
            const float l2 = KV ? rowstat[ol] : lse2_own;
            const float dl = KV ? rowstat[kBwdOther + ol] : delta_own;
            const float pv = valid ? __builtin_amdgcn_exp2f(__builtin_fmaf(p.c1, s[r], bias2) + l2) : 0.f;
            const float ds = valid ? pv * (dp[r] + dl) : 0.f;     // (a NaN of dP stays out of the sums over pairs that exist)
            s[r] = pv;
            dp[r] = ds;
            tile_sum += ds;
        }
        if constexpr (!KV) {
            // (wavefront-uniform) every pair of the block at a saturated distance on one side, or dS summed per
            // distance by way of LDS, as in bwd16_kernel: the pair of key kk and query lr at row lr, column
            // kk - lr + R - 1.  (One LDS atomic per pair took two thirds of the pass.)
            const int rel_min = o0 + sub0 - (w_lo + 31 + P), rel_max = rel_min + 62;
            if (has_bias) {
                if (rel_max <= -sat) sum_lo += tile_sum;
                else if (rel_min >= sat) sum_hi += tile_sum;
                else {
                    constexpr int R = SKEW_ROWS;
#pragma unroll
                    for (int round = 0; round < 32 / R; ++round) {
                        if (lr / R == round) {
                            float* w = skew + (lr % R) * 63 + (R - 1) + 4 * hh;
#pragma unroll
                            for (int r = 0; r < 16; ++r) w[8 * (r >> 2) + (r & 3)] = dp[r];
                        }
                        asm volatile("" ::: "memory");     // (LDS accesses of a wavefront keep their order)
                        float sum = 0.f;
#pragma unroll
                        for (int q = 0; q < R; ++q) sum += skew[q * 64 + lane];
                        asm volatile("" ::: "memory");
                        const int rel = rel_min + 31 - R * round + lane - (R - 1);
                        if (lane < 31 + R) atomicAdd(&hist_rel[min(max(rel, -sat), sat) + sat], sum);
                    }
                }
            }
        }

        // dQ^T += K^T dS^T   /   dK^T += Q^T dS, dV^T += dO^T P   (contraction over the block's 32 rows, two per product)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int ol = sub0 + 8 * (r >> 2) + 4 * hh + (r & 3);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                acc_a[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(ta[ol * STR + 32 * dt + lr], dp[r], acc_a[dt], 0, 0, 0);
                if constexpr (KV)
                    acc_b[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(tb[ol * STR + 32 * dt + lr], s[r], acc_b[dt], 0, 0, 0);
            }
        }
    }

    // the partial gradients of the other half's wavefronts, in lane order
    float* const red = tiles + (wave % OWNW) * ((KV ? 2 : 1) * DT * 16 * 64) + lane;
    __syncthreads();
    if (sub0 != 0) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                red[(dt * 16 + r) * 64] = acc_a[dt][r];
                if constexpr (KV) red[((DT + dt) * 16 + r) * 64] = acc_b[dt][r];
            }
    }
    __syncthreads();
    if (sub0 == 0) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc_a[dt][r] += red[(dt * 16 + r) * 64];
                if constexpr (KV) acc_b[dt][r] += red[((DT + dt) * 16 + r) * 64];
            }
    }

    // rows: lane (lr, hh) holds, for its own row, elements 32 dt + 8 g + 4 hh .. + 3 of the transposed gradients
    const float scale = p.c1 * 0.6931471805599453f;     // d score / d (q . k), natural units
    if (own_ok && sub0 == 0) {
        T* oa = KV ? reinterpret_cast<T*>(p.dk) + (int64_t)b * p.dk_sb + (int64_t)h * p.dk_sh + (k_first + own_row) * p.dk_sr
                   : reinterpret_cast<T*>(p.dq) + (int64_t)b * p.dq_sb + (int64_t)h * p.dq_sh + (q_first + own_row) * p.dq_sr;
        T* ob = KV ? reinterpret_cast<T*>(p.dv) + (int64_t)b * p.dv_sb + (int64_t)h * p.dv_sh + (k_first + own_row) * p.dv_sr : nullptr;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int d0 = 32 * dt + 8 * g + 4 * hh;
                if (d0 < D) {
                    store4(oa + d0, f32x4{acc_a[dt][4 * g] * scale, acc_a[dt][4 * g + 1] * scale,
                                          acc_a[dt][4 * g + 2] * scale, acc_a[dt][4 * g + 3] * scale});
                    if constexpr (KV)
                        store4(ob + d0, f32x4{acc_b[dt][4 * g], acc_b[dt][4 * g + 1], acc_b[dt][4 * g + 2], acc_b[dt][4 * g + 3]});
                }
            }
    }
    if constexpr (!KV) {
        if (has_bias && p.dtable != nullptr) {
            // the saturated tiles' sums: one value per wavefront and side, into the last bucket of that side
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                sum_lo += __shfl_xor(sum_lo, off, 64);
                sum_hi += __shfl_xor(sum_hi, off, 64);
            }
            float* const hist = tiles;     // (the tiles are done with)
            __syncthreads();
            for (int x = tid; x < p.n_buckets; x += kBwdThreads) hist[x] = 0.f;
            __syncthreads();
            if (lane == 0) {
                if (sum_lo != 0.f) atomicAdd(&hist[bucket_of(p.bs, -sat)], sum_lo);
                if (sum_hi != 0.f) atomicAdd(&hist[bucket_of(p.bs, sat)], sum_hi);
            }
            for (int x = tid; x <= 2 * sat; x += kBwdThreads)     // distances -> buckets
                if (hist_rel[x] != 0.f) atomicAdd(&hist[bucket_of(p.bs, x - sat)], hist_rel[x]);
            __syncthreads();
            for (int x = tid; x < p.n_buckets; x += kBwdThreads)
                if (hist[x] != 0.f) atomicAdd(&p.dtable[(int64_t)x * p.H + h], hist[x]);
        }
    }
}


// ------------------------------------------------------------------------------------------------------------------
// 16-bit inputs at head_dim 64 and 128: passes of the same kind on the 16-bit matrix cores
// (v_mfma_f32_32x32x16_bf16 / _f16).  PASS 0: dq and the table gradient; 1: dk and dv; 2: dk; 3: dv.
//
// The products over head_dim (S^T = K Q^T, dP^T = V dO^T and their counterparts of the dk / dv passes) take the inputs as
// they are; the probabilities and dS are rounded to the input type for the products over the tile's rows, as the
// reference does (fused_bias_attention.py:575-590: p.to(Q.dtype), ds.to(Q.dtype)); sums stay in fp32.  A tile of
// the other kind is rows of 128 or 256 bytes in LDS and serves both kinds of product from one copy: rows are read as they
// lie (A operand, contraction over head_dim), and the contraction over the tile's rows reads it through the
// transposing LDS read (ds_read_b64_tr_b16: four rows x 16 columns per group of 16 lanes), whose k-slot order --
// rows 4h .. 4h+3 and 8+4h .. 8+4h+3 of every 16 in lane half h -- is exactly the order in which a lane holds the rows
// of a 32x32 accumulator, so P and dS go from accumulator registers to B operands with a conversion and no shuffle.
// The 16-byte chunks of a row are XOR-swizzled with a pattern that keeps both kinds of read free of bank conflicts.
//
// What bounds it: no single pipe.  At B16 H12 L1024 D64 bf16 the matrix pipe is busy 40 % of the cycles, the vector
// port 50 %, LDS 45 %, with three wavefronts per SIMD.  Hence the choices below: one 32 x 32 block of scores per
// wavefront and step (144-168 registers; two blocks need two wavefronts per SIMD and copies between the code of the
// block classes), accumulators touched by one piece of code only (a class decides about arguments, never about products:
// with the products in the classes' branches the compiler kept a copy of every accumulator per branch and spilled), and
// as few instructions per score as the formulas allow.  Deeper staging (3 or 4 tile buffers) was slower: the LDS it
// takes costs more than the wait it saves.  Two blocks per wavefront and step / this one, us, the passes with
// bwd_rows_kernel, bf16: B16 H12 L1024 D64 283 / 238, the same causal 198 / 167, B4 H12 L4096 D64 810 / 764, B4 H6
// L4096 D128 1248 / 846, B2 H8 L1999 D128 causal 284 / 135.
// head_dim 128 (the T5-3B / 11B head shape): rows of 256 bytes, sixteen chunks
__device__ __forceinline__ int tile_swz128(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }

// Geometry of a 16-bit backward workgroup: wavefronts each on 32 own rows and 32 rows of the tile at a time (one
// 32 x 32 block of scores: 32 score registers, which is what lets three wavefronts share a SIMD at head_dim 64).
// SPLIT 1: four groups of own rows, tiles of 32.  SPLIT 2: two groups of own rows, tiles of 64 whose halves go to
// different wavefronts; the two partial gradients of a row are added through LDS at the end.  SPLIT 4: the same with eight
// wavefronts and tiles of 128, which halves the chain of tiles behind a block once more.
template <int D, int PASS, int SPLIT>
struct Bwd16Geom {
    static constexpr bool KV = PASS != 0;
    static constexpr int WAVES = SPLIT == 4 ? 8 : 4, THREADS = 64 * WAVES;
    static constexpr int OWNW = WAVES / SPLIT, OWN = 32 * OWNW, OTHER = 32 * SPLIT;
    static constexpr int TILE = OTHER * D * 2;                    // bytes of one staged tile
    static constexpr int SLABS = TILE / 1024 / WAVES;               // 1 KB requests per wavefront and tile
    static constexpr int RPS = 1024 / (2 * D);                    // rows per request
    static constexpr int STAGES = 2;                               // tile buffers
    static constexpr int REQS = 2 * SLABS + (KV ? 1 : 0);         // requests per wavefront and tile
    static constexpr int SKEW_ROWS = D == 128 && SPLIT >= 2 ? 8 : SPLIT == 4 ? 16 : 32;   // queries per round of the table gradient
    static constexpr int STAT_ROWS = OTHER > 64 ? OTHER : 64;      // of one statistic of a tile
    static constexpr int LUT_PAD16 = 64;                          // a 32 x 32 block spans 63 distances
    static constexpr int STAT = STAGES * 2 * TILE;                // byte offsets
    static constexpr int LUT = STAT + (KV ? STAGES * 2 * STAT_ROWS * 4 : 0);
    static __host__ __device__ int lut_floats(int sat) { return (2 * (sat + LUT_PAD16) + 4) & ~3; }
    static __host__ __device__ int hist(int sat) { return LUT + 4 * lut_floats(sat); }
    static __host__ __device__ int skew(int sat) { return hist(sat) + (KV ? 0 : 4 * WAVES * table_grad_floats(sat)); }
    static __host__ __device__ int bytes(int sat, bool bias) { return skew(sat) + (KV || !bias ? 0 : WAVES * SKEW_ROWS * 64 * 4); }
};

template <int D> __device__ __forceinline__ int row_swz(int row) { return D == 64 ? tile_swz(row) : tile_swz128(row); }

template <typename T, int D, bool CAUSAL, int PASS, int SPLIT>
__global__ __launch_bounds__(SPLIT == 4 ? 512 : kBwdThreads, SPLIT != 4 && (D == 64 || (PASS == 3 && SPLIT == 1)) ? 3 : 2) void bwd16_kernel(const BwdParams p, int nblk) {
    constexpr bool KV = PASS != 0, DS = PASS != 3, DA = PASS != 3, DV = PASS == 1 || PASS == 3;   // dS; dq or dk; dv
    using G = Bwd16Geom<D, PASS, SPLIT>;
    constexpr int DT = D / 32, KS = D / 16, OTHER = G::OTHER, CH = D / 8;
    using H16 = Half16<T>;
    using v8 = typename H16::v8;
    extern __shared__ __attribute__((aligned(16))) unsigned char bwd_smem[];

    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), ow = wave % G::OWNW, sub0 = (wave / G::OWNW) * 32;
    int own_block, h, b;
    bwd_place<CAUSAL, KV>(p.H, p.B, nblk, own_block, h, b);
    const int own_base = own_block * G::OWN;
    const int64_t slot = ((int64_t)h * p.B + b) * nblk + own_block;     // (of the table gradient)
    if constexpr (PASS == 1 || PASS == 2) {
        // (the last block: the shortest of a causal launch)
        if (p.slots != nullptr && p.table != nullptr && own_block == nblk - 1 && b == 0) table_grad_reduce<G::WAVES>(p, h, reinterpret_cast<float*>(bwd_smem));
    }
    const int w_lo = own_base + ow * 32, own_row = w_lo + lr;     // this wavefront's, this lane's own rows
    int M = p.M, N = p.N;
    int64_t q_first = 0, k_first = 0;
    if (p.cu_q != nullptr) {
        q_first = p.cu_q[b]; k_first = p.cu_k[b];
        M = p.len_q != nullptr ? p.len_q[b] : p.cu_q[b + 1] - (int)q_first;
        N = p.len_k != nullptr ? p.len_k[b] : p.cu_k[b + 1] - (int)k_first;
        if (own_base >= (KV ? N : M)) {     // (the grid is sized for the longest sequence)
            if constexpr (PASS == 0) table_grad_none<G::WAVES>(p, slot);
            return;
        }
    }
    const int n_own = KV ? N : M, n_other = KV ? M : N;
    const int P = N - M;
    const bool has_bias = p.table != nullptr;
    const int sat = has_bias ? p.bs.sat : 0;
    float* const lut = reinterpret_cast<float*>(bwd_smem + G::LUT);
    float* const dist = reinterpret_cast<float*>(bwd_smem + G::hist(sat)) + wave * table_grad_floats(sat);   // dS per distance
    float* const skew = reinterpret_cast<float*>(bwd_smem + G::skew(sat)) + wave * G::SKEW_ROWS * 64;

    const T* qp = reinterpret_cast<const T*>(p.q) + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh + q_first * p.q_sr;
    const T* kp = reinterpret_cast<const T*>(p.k) + (int64_t)b * p.k_sb + (int64_t)h * p.k_sh + k_first * p.k_sr;
    const T* vp = reinterpret_cast<const T*>(p.v) + (int64_t)b * p.v_sb + (int64_t)h * p.v_sh + k_first * p.v_sr;
    const T* gp = reinterpret_cast<const T*>(p.dout) + (int64_t)b * p.do_sb + (int64_t)h * p.do_sh + q_first * p.do_sr;
    const int64_t stat_sr = p.cu_q != nullptr ? p.H : 1;
    const int64_t stat_base = p.cu_q != nullptr ? q_first * p.H + h : ((int64_t)b * p.H + h) * p.M;

    // tiles that can hold a visible pair
    int t_lo = 0, t_hi = (n_other + OTHER - 1) / OTHER;
    if (CAUSAL) {
        if (!KV) t_hi = min(t_hi, max(0, own_base + G::OWN - 1 + P + OTHER) / OTHER);
        else t_lo = max(0, own_base - P) / OTHER;
    }

    // staging by LDS-DMA, 1 KB per request; each wavefront requests its share of the slabs of both tiles.  The chunk
    // swizzle is applied on the source side: the lane that writes physical chunk pc of row r fetches logical chunk
    // pc ^ swizzle(r).  Rows past the end of the tensor are out of the descriptor's range and arrive as zeros.
    // (Slices stay below 2 GiB -- checked on the host -- so 32-bit offsets do.)
    const T* src_a = KV ? qp : kp;
    const T* src_b = KV ? gp : vp;
    const int a_srb = (int)(KV ? p.q_sr : p.k_sr) * 2, b_srb = (int)(KV ? p.do_sr : p.v_sr) * 2;     // row strides in bytes
    const u32x4 rs_a = dma_rsrc(src_a, n_other > 0 ? (unsigned)(n_other - 1) * (unsigned)a_srb + D * 2 : 0u);
    const u32x4 rs_b = dma_rsrc(src_b, n_other > 0 ? (unsigned)(n_other - 1) * (unsigned)b_srb + D * 2 : 0u);
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)bwd_smem;
    // dk / dv: minus the log-sum-exp and minus delta of the tile's queries, one request of 64 words each (a tile of 32
    // leaves the second half unused); wavefronts 2 and 3 repeat those of 0 and 1, so that all have the same count
    const u32x4 rs_s = dma_rsrc((wave & 1 ? p.delta : p.lse2) + stat_base, n_other > 0 ? (unsigned)(n_other - 1) * (unsigned)(stat_sr * 4) + 4 : 0u);
    auto request = [&](int t, int buf) {     // tile t into buffer buf
#pragma unroll
        for (int c = 0; c < G::SLABS; ++c) {
            const int slab = G::SLABS * wave + c, row = slab * G::RPS + lane / CH, ch = (lane % CH) ^ row_swz<D>(row);
            const unsigned at = (unsigned)buf * (2 * G::TILE) + slab * 1024u;
            const int other = min(t * OTHER + row, n_other);     // (a row past the end: one that cannot wrap around)
            dma_16(rs_a, lds0 + at, other * a_srb + ch * 16);
            dma_16(rs_b, lds0 + at + G::TILE, other * b_srb + ch * 16);
        }
        if constexpr (KV) {
            const int half = G::STAT_ROWS > 64 ? (wave >> 1 & 1) * 64 : 0;
            dma_4(rs_s, lds0 + G::STAT + (buf * 2 + (wave & 1)) * (G::STAT_ROWS * 4) + half * 4, (t * OTHER + half + lane) * (int)stat_sr * 4);
        }
    };
    const BiasColumn bias(p, h, lane);
    // Tile t + STAGES - 1 is requested when the barrier at the top of tile t has shown that every wavefront is done with
    // the buffer it goes into (tile t - 1's): it has STAGES - 1 tiles' work to arrive in.
#pragma unroll
    for (int c = 0; c < G::STAGES - 1; ++c)
        if (t_lo + c < t_hi) request(t_lo + c, c);

    // own rows as B operands: lane (lr, hh) holds elements 16 s + 8 hh .. + 7 of its row
    const bool own_ok = own_row < n_own;
    v8 fa[KS], fb[KS];
    {
        const T* a = (KV ? kp + (int64_t)own_row * p.k_sr : qp + (int64_t)own_row * p.q_sr);
        const T* c = (KV ? vp + (int64_t)own_row * p.v_sr : gp + (int64_t)own_row * p.do_sr);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
#pragma unroll
            for (int e = 0; e < 8; ++e) { fa[s][e] = (T)0.0f; fb[s][e] = (T)0.0f; }
            if (own_ok) {
                fa[s] = *reinterpret_cast<const v8*>(a + 16 * s + 8 * hh);
                if constexpr (DS) fb[s] = *reinterpret_cast<const v8*>(c + 16 * s + 8 * hh);
            }
        }
    }
    // (rows past the end: -inf makes every probability of the row 0)
    float nlse2_own = -INFINITY, ndelta_own = 0.f;
    if (!KV && own_ok) { nlse2_own = p.lse2[stat_base + own_row * stat_sr]; ndelta_own = p.delta[stat_base + own_row * stat_sr]; }

    // bias per distance, ascending with the tile's row index in both passes (dk / dv: by -rel), so that consecutive
    // rows are consecutive words; padded by 64 on both sides, more than the distances of a lane's rows span
    float bias_lo = 0.f, bias_hi = 0.f;     // ... and of the two saturated sides
    {
        const int mid = sat + G::LUT_PAD16;
        for (int x0 = 0; x0 <= 2 * mid; x0 += G::THREADS) {
            const int x = x0 + tid;
            const float v = bias.at(KV ? mid - x : x - mid);
            if (x <= 2 * mid) lut[x] = v;
        }
        if (has_bias) {
            bias_lo = bias.at(-sat); bias_hi = bias.at(sat);
            if constexpr (!KV) {
                for (int x = lane; x <= 2 * sat; x += 64) dist[x] = 0.f;
                for (int x = lane; x < G::SKEW_ROWS * 64; x += 64) skew[x] = 0.f;
            }
        }
    }

    // row reads: element offsets of this lane's chunk (2 s + hh) of row lr; the 32-row halves of a tile differ by a constant
    int row_off[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) row_off[s] = (sub0 + lr) * D + (((2 * s + hh) ^ row_swz<D>(lr)) * 8);
    // transposing reads: within a group of 16 lanes, lane 4 j + a supplies the address of elements 4 a' .. of row j
    // and receives, for column (lane % 16) of the group's 16 columns, the rows j = 0 .. 3.  Group g covers the
    // columns 32 dt + 16 (g & 1) .. + 15 and the rows 4 (g >> 1) .. + 3 (first read) and 8 more (second read).
    int tr_lo[DT], tr_hi[DT];
    {
        const int g = lane >> 4, r = lane & 15, jj = r >> 2, aa = r & 3;
        const int row = 4 * (g >> 1) + jj, x = 2 * (g & 1) + (aa >> 1);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            tr_lo[dt] = (sub0 + row) * D + (((4 * dt + x) ^ row_swz<D>(row)) * 8) + (aa & 1) * 4;
            tr_hi[dt] = (sub0 + row + 8) * D + (((4 * dt + x) ^ row_swz<D>(row + 8)) * 8) + (aa & 1) * 4;
        }
    }
    auto tr_frag = [&](const T* tile, int g16, int dt) {   // columns 32 dt .. + 31 x rows 16 g16 .. + 15 of the block, as an A operand
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(tile + tr_lo[dt] + 16 * g16 * D));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(tile + tr_hi[dt] + 16 * g16 * D));
        return __builtin_bit_cast(v8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };

    f32x16 acc_a[DA ? DT : 1], acc_b[DV ? DT : 1];     // dQ^T or dK^T; dV^T
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) { if constexpr (DA) acc_a[dt][r] = 0.f; if constexpr (DV) acc_b[dt][r] = 0.f; }
    float sum_lo = 0.f, sum_hi = 0.f;
    const float c1 = p.c1;

    for (int t = t_lo, buf = 0; t < t_hi; ++t, buf = buf + 1 == G::STAGES ? 0 : buf + 1) {
        // this wavefront's requests for tile t have landed (those of the STAGES - 2 tiles behind it may be in flight) ...
        if (G::STAGES > 2 && t + G::STAGES - 2 < t_hi) wait_vmcnt<(G::STAGES - 2) * G::REQS>(); else wait_vmcnt<0>();
        __syncthreads();     // ... and everybody's; the buffer of tile t - 1 is free (and, first time round, the LUT written)
        if (t + G::STAGES - 1 < t_hi) request(t + G::STAGES - 1, buf == 0 ? G::STAGES - 1 : buf - 1);
        const T* ta = reinterpret_cast<const T*>(bwd_smem + buf * 2 * G::TILE);
        const T* tb = reinterpret_cast<const T*>(bwd_smem + buf * 2 * G::TILE + G::TILE);
        const float* rowstat = reinterpret_cast<const float*>(bwd_smem + G::STAT) + buf * 2 * G::STAT_ROWS + sub0 + 4 * hh;
        (void)rowstat;

        const int s0 = t * OTHER + sub0;        // first tile row of this wavefront's block
        // rel = j - (i + P): dq pass j in the tile, i own; dk / dv pass i in the tile, j own
        const int rel_min = KV ? w_lo - (s0 + 31 + P) : s0 - (w_lo + 31 + P), rel_max = rel_min + 62;
        if (s0 < n_other && (!CAUSAL || rel_min <= 0)) {
            f32x16 s, dp;
#pragma unroll
            for (int r = 0; r < 16; ++r) { s[r] = 0.f; dp[r] = 0.f; }
            if constexpr (KV && DS) {      // (dP starts at -delta: the matrix core subtracts it for free)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    const f32x4 d4 = *reinterpret_cast<const f32x4*>(rowstat + G::STAT_ROWS + 8 * r4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) dp[4 * r4 + e] = d4[e];
                }
            }
            // (the two chains in turn: 2 % faster than one behind the other)
#pragma unroll
            for (int k2 = 0; k2 < KS; ++k2) {
                s = H16::mfma(*reinterpret_cast<const v8*>(ta + row_off[k2]), fa[k2], s);
                if constexpr (DS) dp = H16::mfma(*reinterpret_cast<const v8*>(tb + row_off[k2]), fb[k2], dp);
            }

            // base-2 arguments of the probabilities; two classes of block (wavefront-uniform): every pair at a saturated
            // distance on one side (one bias), or a look-up per pair
            const bool sat_lo = rel_max <= -sat, sat_hi = rel_min >= sat;
            if (sat_lo || sat_hi) {
                const float bias_c = sat_lo ? bias_lo : bias_hi;
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    f32x4 l4 = {nlse2_own, nlse2_own, nlse2_own, nlse2_own};
                    if constexpr (KV) l4 = *reinterpret_cast<const f32x4*>(rowstat + 8 * r4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[4 * r4 + e] = __builtin_fmaf(c1, s[4 * r4 + e], bias_c + l4[e]);
                }
            } else {
                const float* lp = lut + (KV ? s0 + P - own_row : s0 - P - own_row) + 4 * hh + sat + G::LUT_PAD16;
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    f32x4 l4 = {nlse2_own, nlse2_own, nlse2_own, nlse2_own};
                    if constexpr (KV) l4 = *reinterpret_cast<const f32x4*>(rowstat + 8 * r4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[4 * r4 + e] = __builtin_fmaf(c1, s[4 * r4 + e], lp[8 * r4 + e]) + l4[e];
                }
            }
            // blocks with an invisible pair (own rows past the end need no test: a query's probabilities are 0, a
            // key's gradients are not stored)
            if (s0 + 32 > n_other || (CAUSAL && rel_max > 0)) {
                // (row 8 (r >> 2) + (r & 3) of the lane's half: visible from `first` on, up to `last`)
                const int first = CAUSAL && KV ? own_row - P - s0 - 4 * hh : 0;
                const int last = min(n_other - 1 - s0 - 4 * hh, CAUSAL && !KV ? own_row + P - s0 - 4 * hh : 32);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int ol = 8 * (r >> 2) + (r & 3);
                    s[r] = (!(CAUSAL && KV) || ol >= first) && ol <= last ? s[r] : -INFINITY;
                }
            }
            // probabilities and dS, rounded to the input type for the products that contract over the block's rows:
            //   dQ^T += K^T dS^T   /   dV^T += dO^T P, dK^T += Q^T dS
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s[r] = __builtin_amdgcn_exp2f(s[r]);
                if constexpr (KV) dp[r] *= s[r];
                else dp[r] = (dp[r] + ndelta_own) * s[r];
            }
            if constexpr (DV) {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const v8 pb = to_frag<v8>(s, u);
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) acc_b[dt] = H16::mfma(tr_frag(tb, u, dt), pb, acc_b[dt]);
                }
            }
            if constexpr (DA) {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const v8 dsb = to_frag<v8>(dp, u);
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) acc_a[dt] = H16::mfma(tr_frag(ta, u, dt), dsb, acc_a[dt]);
                }
            }
            if constexpr (!KV) {
                if (has_bias) {
                    if (sat_lo || sat_hi) {
                        const float sum = ((dp[0] + dp[1]) + (dp[2] + dp[3])) + ((dp[4] + dp[5]) + (dp[6] + dp[7])) +
                                          ((dp[8] + dp[9]) + (dp[10] + dp[11])) + ((dp[12] + dp[13]) + (dp[14] + dp[15]));
                        if (sat_lo) sum_lo += sum; else sum_hi += sum;
                    } else {
                        table_grad_block<G::SKEW_ROWS>(skew, dist, dp, lane, s0 - (w_lo + P), sat, sum_lo, sum_hi);
                    }
                }
            }
        }
    }

    if constexpr (SPLIT > 1) {
        // the partial gradients of the other wavefronts on the same rows, in lane order through the tile buffers
        constexpr int AT_B = DA ? DT * 16 : 0, REGS = ((DA ? 1 : 0) + (DV ? 1 : 0)) * DT * 16;
        const int part = wave / G::OWNW;
        static_assert(SPLIT / 2 * G::OWNW * REGS * 256 <= G::STAGES * 2 * G::TILE, "");
#pragma unroll
        for (int n = SPLIT / 2; n > 0; n /= 2) {
            float* const red = reinterpret_cast<float*>(bwd_smem) + ((part & (n - 1)) * G::OWNW + ow) * (REGS * 64) + lane;
            __syncthreads();
            if (part >= n && part < 2 * n) {
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        if constexpr (DA) red[(dt * 16 + r) * 64] = acc_a[dt][r];
                        if constexpr (DV) red[(AT_B + dt * 16 + r) * 64] = acc_b[dt][r];
                    }
            }
            __syncthreads();
            if (part < n) {
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        if constexpr (DA) acc_a[dt][r] += red[(dt * 16 + r) * 64];
                        if constexpr (DV) acc_b[dt][r] += red[(AT_B + dt * 16 + r) * 64];
                    }
            }
        }
    }
    const float scale = p.c1 * 0.6931471805599453f;     // d score / d (q . k), natural units; dv has none
    if (own_ok && sub0 == 0) {
        T* oa = !KV ? reinterpret_cast<T*>(p.dq) + (int64_t)b * p.dq_sb + (int64_t)h * p.dq_sh + (q_first + own_row) * p.dq_sr
                    : reinterpret_cast<T*>(p.dk) + (int64_t)b * p.dk_sb + (int64_t)h * p.dk_sh + (k_first + own_row) * p.dk_sr;
        T* ob = DV ? reinterpret_cast<T*>(p.dv) + (int64_t)b * p.dv_sb + (int64_t)h * p.dv_sh + (k_first + own_row) * p.dv_sr : nullptr;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int d0 = 32 * dt + 8 * g + 4 * hh;
                if constexpr (DA)
                    store4(oa + d0, f32x4{acc_a[dt][4 * g] * scale, acc_a[dt][4 * g + 1] * scale,
                                          acc_a[dt][4 * g + 2] * scale, acc_a[dt][4 * g + 3] * scale});
                if constexpr (DV)
                    store4(ob + d0, f32x4{acc_b[dt][4 * g], acc_b[dt][4 * g + 1], acc_b[dt][4 * g + 2], acc_b[dt][4 * g + 3]});
            }
    }
    if constexpr (!KV) {
        // (the tiles are done with)
        if (has_bias && p.dtable != nullptr)
            table_grad_finish<G::WAVES>(p, h, slot, reinterpret_cast<const float*>(bwd_smem + G::hist(sat)), reinterpret_cast<float*>(bwd_smem), sat, sum_lo, sum_hi);
    }
}

// A pass's SPLIT.  2 (own blocks of 64 instead of 128 rows, each block of scores walked by two wavefronts) halves the longest
// chain and doubles the workgroups, at twice the fetches per product, so it pays where 128-row
// blocks leave the chip idle (256 compute units with room for three workgroups at head_dim 64, two at 128).  Both
// sides, us, three kernels, bf16: head_dim 64 full attention, 256 workgroups 245 / 190 (SPLIT 1 / 2), 384 294 / 276, 512
// 302 / 333; causal, where the longest block counts, 512 233 / 182, 1536 181 / 228; head_dim 128 256 440 / 325, 384
// 504 / 586, causal 256 208 / 140, 512 259 / 221, 1024 390 / 441.  Packed, head_dim 64 (workgroups counted from the
// tokens of the pass's own kind): 424 67 / 73, causal 58 / 58, 564 186 / 183, 1464 212 / 222; cross-attention of 16 x 32
// queries over 16 x 2048 keys, 12 heads, where only the key pass fills the chip: 115 us with both passes by the queries'
// count, 94 each by its own (head_dim 128, 8 heads 175 / 135; 2048 queries over 32 keys 136 / 111).
// 4 (eight wavefronts, tiles of 128) where blocks of 64 rows are one round of one workgroup per compute unit, which is what its
// LDS allows, and with a causal mask up to one and a half.  us, SPLIT 2 / 4: 64-row blocks of unpacked tensors, head_dim 64 128 (B1 H8 L1000)
// 46 / 39, 256 (B1 H8 L2000) 72 / 59, causal 71 / 55, 320 (B20 H8 L128) 28 / 41, causal 512 75 / 74, 864 82 / 116; head_dim 128
// 256 122 / 111, causal 378 (B1 H6 L4000) 226 / 178, 512 139 / 137, 1024 216 / 268.
// It needs more than one tile to walk: 8 heads of D128 B8 L47 25.9 / 31.4, B5 L128 causal 30.3 / 34.1, D64 B5 L100 20.6 / 21.0, B1 L200
// 24.2 / 23.5, 2000 queries over 128 keys 47.6 / 37.9.
int bwd16_split(const BwdParams& p, int D, bool causal, bool keys) {
    const int rows = keys ? p.N : p.M;
    const int64_t pairs = (int64_t)p.H * p.B;
    if (p.cu_q == nullptr && (keys ? p.M : p.N) > 128 && (rows + 63) / 64 * pairs <= (causal ? 384 : 256)) return 4;
    const int64_t blocks = p.cu_q != nullptr ? ((int64_t)(keys ? p.total_k : p.total_q) / 128 + p.B) * p.H : (rows + 127) / 128 * pairs;
    return blocks < (p.cu_q != nullptr ? 320 : causal ? 768 : D == 64 ? 512 : 320) ? 2 : 1;
}

template <typename T, int D, bool CAUSAL, int PASS, int SPLIT>
hipError_t launch_bwd16_pass(const BwdParams& p, hipStream_t stream) {
    using G = Bwd16Geom<D, PASS, SPLIT>;
    const int rows = PASS != 0 ? p.N : p.M;
    if (rows <= 0) return hipSuccess;
    const int nblk = (rows + G::OWN - 1) / G::OWN;
    const int64_t blocks = (int64_t)nblk * p.H * p.B;
    if (blocks > 0x7fffffff) return hipErrorInvalidConfiguration;
    const bool bias = p.table != nullptr;
    const int lds = G::bytes(bias ? p.bs.sat : 0, bias);
    auto kern = bwd16_kernel<T, D, CAUSAL, PASS, SPLIT>;
    static LdsLimit limit;     // (per instantiation; bytes with the widest bucketing, saturated at 1024: 115 280 at head_dim 128, 107 088 at 64; SPLIT 4 up to 160 KB)
    const hipError_t e = limit.allow(reinterpret_cast<const void*>(kern), lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(G::THREADS), lds, stream, p, nblk);
    return hipGetLastError();
}

template <typename T, int D, bool CAUSAL, int PASS>
hipError_t launch_bwd16_rows(const BwdParams& p, hipStream_t stream) {
    const int split = bwd16_split(p, D, CAUSAL, PASS != 0);
    // (bucketings that saturate past distance 901, 219 at head_dim 128, leave no room for the largest tiles next to the table gradient's sums)
    if (split == 4 && Bwd16Geom<D, PASS, 4>::bytes(p.table != nullptr ? p.bs.sat : 0, p.table != nullptr) <= 160 * 1024)
        return launch_bwd16_pass<T, D, CAUSAL, PASS, 4>(p, stream);
    return split > 1 ? launch_bwd16_pass<T, D, CAUSAL, PASS, 2>(p, stream) : launch_bwd16_pass<T, D, CAUSAL, PASS, 1>(p, stream);
}

template <typename T, int D, bool CAUSAL>
hipError_t launch_bwd16(BwdParams p, hipStream_t stream) {
    p.slots_per_head = p.B * (bwd16_split(p, D, CAUSAL, false) > 1 ? (p.M + 63) / 64 : (p.M + 127) / 128);
    if (p.N <= 0) p.slots = nullptr;      // (no pass that would add them)
    hipError_t e = launch_bwd16_rows<T, D, CAUSAL, 0>(p, stream);
    if (e != hipSuccess) return e;
    if constexpr (D == 64) {
        return launch_bwd16_rows<T, D, CAUSAL, 1>(p, stream);
    } else {
        // head_dim 128: a row's head_dim twice and two gradients of it do not fit 256 registers next to the scores
        // (the joint pass spills and takes 721 us where the two take 592: B4 H6 L4096)
        if ((e = launch_bwd16_rows<T, D, CAUSAL, 2>(p, stream)) != hipSuccess) return e;
        return launch_bwd16_rows<T, D, CAUSAL, 3>(p, stream);
    }
}

template <typename T, int D>
hipError_t launch_bwd_d(const BwdParams& p, bool causal, hipStream_t stream) {
    const int64_t rows = p.cu_q != nullptr ? (int64_t)p.total_q * p.H : (int64_t)p.B * p.H * p.M;
    hipLaunchKernelGGL((bwd_rows_kernel<T, D>), dim3((unsigned)((rows + RowsGeom<T, D>::ROWS - 1) / RowsGeom<T, D>::ROWS)), dim3(256), 0, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if constexpr (sizeof(T) == 2 && (D == 64 || D == 128)) {
        if (p.fp32_math == 0) return causal ? launch_bwd16<T, D, true>(p, stream) : launch_bwd16<T, D, false>(p, stream);
    }
    if constexpr (sizeof(T) == 4 && D == 64) {
        if (p.fp32_math == 0) return launch_bwd_f32_64(p, causal, stream);
    }
    if constexpr (D == 128) {
        return hipErrorInvalidValue;     // (the fp32 kernels hold a row's head_dim in registers: up to 64)
    } else {
        const dim3 gq((p.M + kBwdOwn - 1) / kBwdOwn, p.H, p.B), gk((p.N + kBwdOwn - 1) / kBwdOwn, p.H, p.B);
        if (causal) {
            hipLaunchKernelGGL((bwd_kernel<T, D, true, false>), gq, dim3(kBwdThreads), 0, stream, p);
            if (p.N > 0) hipLaunchKernelGGL((bwd_kernel<T, D, true, true>), gk, dim3(kBwdThreads), 0, stream, p);
        } else {
            hipLaunchKernelGGL((bwd_kernel<T, D, false, false>), gq, dim3(kBwdThreads), 0, stream, p);
            if (p.N > 0) hipLaunchKernelGGL((bwd_kernel<T, D, false, true>), gk, dim3(kBwdThreads), 0, stream, p);
        }
        return hipGetLastError();
    }
}

template <typename T>
hipError_t launch_bwd_t(const BwdParams& p, int D, bool causal, hipStream_t s) {
    switch (D) {
        case 128:
            if constexpr (sizeof(T) == 2) return launch_bwd_d<T, 128>(p, causal, s);
            break;
        case 16: return launch_bwd_d<T, 16>(p, causal, s);
        case 32: return launch_bwd_d<T, 32>(p, causal, s);
        case 64: return launch_bwd_d<T, 64>(p, causal, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_bwd_dense(const BwdParams& p, int dtype, int D, bool causal, hipStream_t stream) {
    if (dtype == T5A_BF16) return launch_bwd_t<__bf16>(p, D, causal, stream);
    if (dtype == T5A_F16) return launch_bwd_t<_Float16>(p, D, causal, stream);
    if (dtype == T5A_F32) return launch_bwd_t<float>(p, D, causal, stream);
    return hipErrorInvalidValue;
}

}  // namespace t5a
