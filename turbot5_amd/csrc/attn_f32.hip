// Attention of fp32 tensors at head_dim 64 on the 16-bit matrix cores: the dense forward, the dense and the packed backward.
//
// Every product of fp32 numbers is formed from operands split into three bf16 parts (split_device.h): six
// v_mfma_f32_32x32x16_bf16 for sixteen indices in place of eight v_mfma_f32_32x32x2_f32, 192 cycles for 512.  Scores,
// probabilities, statistics and sums stay fp32; a probability or dS is split in its turn for the products over the tile's rows.
//
// Blocks and their order are those of attn_bwd.hip: a wavefront owns 32 rows and forms one 32 x 32 block of scores per step; a
// tile of the other kind is three planes of bf16 rows in LDS that serve the products over head_dim (rows as they lie) and the
// products over the tile's rows (transposing reads).  A tile is fetched into registers a step ahead and split into the other of
// two LDS buffers beside the products: one barrier per tile.
//
// What bounds it: large launches the matrix cores at the clock the card's power allows them (B3 H16 L2000, forward 265 us: 1110
// TFLOP/s of bf16 products, where a loop of nothing but such products on random numbers runs at 1870), small ones the chain of one
// wavefront per SIMD: products, exponentials, splits.  us, products on the fp32 matrix cores / this, forward and the backward's
// kernels: B4 H8 L512 47 / 25 and 127 / 73, B2 H6 L1999 causal 155 / 62 and 552 / 199, B8 H12 L1024 222 / 145 and 920 / 560, B3 H16
// L2000 424 / 265 and 1715 / 1020.  Errors against 64 bits are smaller: 4.5e-7 for 6.1e-7 (o, B4 H8 L512), 8.5e-7 for 1.05e-6 (dq, dk, dv).
//
// What is split is scaled (split_device.h), by exact powers of two that leave the sums again: a tile's rows and the probabilities by 2^16; own
// rows of a score's product by 2^-16, so that scores carry no factor and nothing is paid per score; own rows of dP's by 2^16, whose 2^32
// then stays on dS.  Without / with the scales, us, forward and backward (three kernels): B4 H8 L512 24.4 / 24.9 and 69 / 73,
// B2 H6 L1999 causal 67 / 62 (the bias is at hand ahead of the tile now) and 189 / 199, B8 H12 L1024 141 / 145 and 543 / 560.
// Scores scaled like dP, with 2^-32 in the factor of their bias's sum: the same times, and errors of o 5 % larger.
//
// Results that are not finite, and rows whose own values below 2^-94 the factor 2^-16 would take out of reach, are formed
// again by the same workgroup on the fp32 matrix cores (RAW): the parts of an infinity, or of a value close to the largest, are no numbers.
#include "split_device.h"
#include "t5a_internal.h"
#include "table_grad_device.h"

namespace t5a {

namespace {

constexpr int kThreads = 256;
constexpr int HD = 64, KS = HD / 16, DT = HD / 32;
constexpr int kPad = 64;                 // a 32 x 32 block spans 63 distances
constexpr int RSTR = HD + 1;             // RAW: fp32 rows padded by one float

// SPLIT 1: four groups of 32 own rows, tiles of 32 rows.  SPLIT 2: two groups of own rows, tiles of 64 whose halves go to
// different wavefronts; what the two hold of a row is put together through LDS at the end.
template <int SPLIT> struct Geom {
    static constexpr int OWNW = 4 / SPLIT, OWN = 32 * OWNW, OTHER = 32 * SPLIT;
    static constexpr int PLANE = OTHER * HD;                     // elements of a plane
    static constexpr int TENSOR = kPlanes * PLANE * 2;           // bytes of a tensor's tile
    static constexpr int BUF = 2 * TENSOR;
    static constexpr int PASSES = OTHER / 32;                    // eight values per thread, tensor and pass
    static constexpr int STAT = 2 * BUF;
    static constexpr int LUT = STAT + 2 * 2 * OTHER * 4 + 16;    // (16: the flag)
    static_assert(RSTR * OTHER * 4 <= TENSOR, "");
    static __host__ __device__ int lut_floats(int sat) { return (2 * (sat + kPad) + 4) & ~3; }
    static __host__ __device__ int hist(int sat) { return LUT + 4 * lut_floats(sat); }
    static constexpr int SKEW_ROWS = SPLIT == 2 ? 32 : 16;       // queries per round of the table gradient (two workgroups share the LDS with SPLIT 1)
    static __host__ __device__ int skew(int sat) { return hist(sat) + 4 * 4 * table_grad_floats(sat); }
    static __host__ __device__ int bytes(int sat, bool table_grad) { return table_grad ? skew(sat) + 4 * SKEW_ROWS * 64 * 4 : hist(sat); }
};

// dP and dS carry `ds`; the sums of P or dS times rows are multiplied by back_b and back_a
template <bool RAW> struct Scale {
    static constexpr float up = RAW ? 1.f : kSplitScale, down = RAW ? 1.f : kSplitBack;
    static constexpr float ds = up * up, ds_back = down * down, back_a = ds_back * down, back_b = ds_back;
};

// the tiles of the two tensors of the other kind
template <int SPLIT, bool RAW> struct Tiles {
    using G = Geom<SPLIT>;
    __amdgpu_buffer_rsrc_t rs[2];
    int stride[2], rows, row0, ch;
    f32x8 x[2][G::PASSES];
    __device__ __forceinline__ Tiles(const float* a, int64_t a_sr, const float* b, int64_t b_sr, int n, int tid) {
        stride[0] = (int)a_sr * 4; stride[1] = (int)b_sr * 4; rows = n; row0 = tid >> 3; ch = tid & 7;
        for (int e = 0; e < 2; ++e)
            rs[e] = __builtin_amdgcn_make_buffer_rsrc((void*)(e ? b : a), 0, n > 0 ? (n - 1) * stride[e] + HD * 4 : 0, 0x00020000);
    }
    __device__ __forceinline__ void fetch(int t) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int n = 0; n < G::PASSES; ++n) {
                const int row = t * G::OTHER + row0 + 32 * n;
                const int off = row < rows ? row * stride[e] + ch * 32 : 0x7fffffe0;     // (zeros past the end)
                u32x4* const d = reinterpret_cast<u32x4*>(&x[e][n]);
                d[0] = __builtin_amdgcn_raw_buffer_load_b128(rs[e], off, 0, 0);
                d[1] = __builtin_amdgcn_raw_buffer_load_b128(rs[e], off + 16, 0, 0);
            }
    }
    __device__ __forceinline__ void store(unsigned char* buf) const {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int n = 0; n < G::PASSES; ++n) {
                const int row = row0 + 32 * n;
                if constexpr (RAW) {
                    float* const to = reinterpret_cast<float*>(buf + e * G::TENSOR) + row * RSTR + ch * 8;
#pragma unroll
                    for (int i = 0; i < 8; ++i) to[i] = x[e][n][i];
                } else {
                    __bf16* const to = reinterpret_cast<__bf16*>(buf + e * G::TENSOR) + row * HD + (ch ^ tile_swz(row)) * 8;
                    bf16x8 s[kPlanes];
                    split3(x[e][n] * kSplitScale, s);
#pragma unroll
                    for (int q = 0; q < kPlanes; ++q) *reinterpret_cast<bf16x8*>(to + q * G::PLANE) = s[q];
                }
            }
    }
};

// A wavefront's own rows as B operands, and its products with a tile.
template <int SPLIT, bool RAW> struct Own;
template <int SPLIT> struct Own<SPLIT, false> {
    bf16x8 f[KS][kPlanes];
    // rows times factor, held times `scale`; the smallest magnitude but zero
    __device__ __forceinline__ unsigned load(const float* row, bool ok, int hh, float factor, float scale) {
        unsigned least = 0xffffffffu;        // twice a magnitude's bits, less one
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            f32x8 x = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (ok) x = *reinterpret_cast<const f32x8*>(row + 16 * s + 8 * hh);
            x *= factor;
#pragma unroll
            for (int e = 0; e < 8; ++e) least = min(least, (__builtin_bit_cast(unsigned, (float)x[e]) << 1) - 1u);
            split3(x * scale, f[s]);
        }
        return least;
    }
};
template <int SPLIT> struct Own<SPLIT, true> {
    float f[HD / 2];
    __device__ __forceinline__ unsigned load(const float* row, bool ok, int hh, float factor, float) {
#pragma unroll
        for (int s = 0; s < HD / 2; ++s) f[s] = ok ? row[2 * s + hh] * factor : 0.f;
        return 0xffffffffu;
    }
};
constexpr unsigned kTiny = 2u * 0x10800000u;      // 2^-94 as `least` counts

// lane constants of the tile reads of a block whose first tile row is sub0
template <int SPLIT, bool RAW> struct Reads;
template <int SPLIT> struct Reads<SPLIT, false> {
    using G = Geom<SPLIT>;
    int row[KS], lo[DT], hi[DT];
    __device__ __forceinline__ Reads(int sub0, int lane) {
        const int lr = lane & 31, hh = lane >> 5;
#pragma unroll
        for (int s = 0; s < KS; ++s) row[s] = (sub0 + lr) * HD + (((2 * s + hh) ^ tile_swz(lr)) * 8);
        const int g = lane >> 4, r = lane & 15, jj = r >> 2, aa = r & 3, rr = 4 * (g >> 1) + jj, x = 2 * (g & 1) + (aa >> 1);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            lo[dt] = (sub0 + rr) * HD + (((4 * dt + x) ^ tile_swz(rr)) * 8) + (aa & 1) * 4;
            hi[dt] = (sub0 + rr + 8) * HD + (((4 * dt + x) ^ tile_swz(rr + 8)) * 8) + (aa & 1) * 4;
        }
    }
    __device__ __forceinline__ void rows(const unsigned char* tensor, int s, bf16x8 (&out)[kPlanes]) const {
        const __bf16* const t = reinterpret_cast<const __bf16*>(tensor) + row[s];
#pragma unroll
        for (int q = 0; q < kPlanes; ++q) out[q] = *reinterpret_cast<const bf16x8*>(t + q * G::PLANE);
    }
    // columns 32 dt .. + 31 x rows 16 u .. + 15 of the block
    __device__ __forceinline__ void columns(const unsigned char* tensor, int u, int dt, bf16x8 (&out)[kPlanes]) const {
        const __bf16* const t = reinterpret_cast<const __bf16*>(tensor) + 16 * u * HD;
#pragma unroll
        for (int q = 0; q < kPlanes; ++q) {
            const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(t + q * G::PLANE + lo[dt]));
            const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(t + q * G::PLANE + hi[dt]));
            out[q] = __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    }
    // s += tile rows x own rows, over head_dim, for one or two tensors; a product of every chain in turn
    template <int N> __device__ __forceinline__ void over_dim(const unsigned char* const (&tensor)[N], const Own<SPLIT, false>* const (&own)[N], f32x16* const (&s)[N]) const {
        using H = Half16<__bf16>;
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            bf16x8 a[N][kPlanes];
#pragma unroll
            for (int e = 0; e < N; ++e) rows(tensor[e], k, a[e]);
#pragma unroll
            for (int q = 2; q >= 0; --q)
#pragma unroll
                for (int x = 0; x <= q; ++x)
#pragma unroll
                    for (int e = 0; e < N; ++e) *s[e] = H::mfma(a[e][x], own[e]->f[k][q - x], *s[e]);
        }
    }
    // acc[dt] += tile columns x (32 tile rows x own rows), over the block's tile rows
    __device__ __forceinline__ void over_rows(const unsigned char* tensor, const f32x16& x, f32x16 (&acc)[DT]) const {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            f32x8 y;
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] = x[8 * u + e];
            bf16x8 b[kPlanes];
            split3(y, b);
            bf16x8 a[DT][kPlanes];
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) columns(tensor, u, dt, a[dt]);
#pragma unroll
            for (int q = 2; q >= 0; --q)
#pragma unroll
                for (int c = 0; c <= q; ++c)
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) acc[dt] = Half16<__bf16>::mfma(a[dt][c], b[q - c], acc[dt]);
        }
    }
};
template <int SPLIT> struct Reads<SPLIT, true> {
    int row, col;
    __device__ __forceinline__ Reads(int sub0, int lane) : row((sub0 + (lane & 31)) * RSTR + (lane >> 5)), col((sub0 + 4 * (lane >> 5)) * RSTR + (lane & 31)) {}
    template <int N> __device__ __forceinline__ void over_dim(const unsigned char* const (&tensor)[N], const Own<SPLIT, true>* const (&own)[N], f32x16* const (&s)[N]) const {
#pragma unroll
        for (int e = 0; e < N; ++e) {
            const float* const t = reinterpret_cast<const float*>(tensor[e]) + row;
#pragma unroll
            for (int k = 0; k < HD / 2; ++k) *s[e] = __builtin_amdgcn_mfma_f32_32x32x2f32(t[2 * k], own[e]->f[k], *s[e], 0, 0, 0);
        }
    }
    __device__ __forceinline__ void over_rows(const unsigned char* tensor, const f32x16& x, f32x16 (&acc)[DT]) const {
        const float* const t = reinterpret_cast<const float*>(tensor) + col;
#pragma unroll
        for (int r = 0; r < 16; ++r)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
                acc[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(t[(8 * (r >> 2) + (r & 3)) * RSTR + 32 * dt], x[r], acc[dt], 0, 0, 0);
    }
};

__device__ __forceinline__ void clear(f32x16 (&acc)[DT]) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[dt][r] = 0.f;
}
// 0, or NaN if a value is not finite
__device__ __forceinline__ float odd(const f32x16 (&acc)[DT]) {
    float x = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) x += acc[dt][r] * 0.f;
    return x;
}
// whether any thread of the workgroup says so
__device__ __forceinline__ bool anybody(int* flag, bool mine) {
    __syncthreads();
    if (threadIdx.x == 0) *flag = 0;
    __syncthreads();
    if (mine) *flag = 1;
    __syncthreads();
    return *flag != 0;
}
// bias by distance, ascending with the tile's row index (down: by minus the distance), padded by kPad on both sides
template <bool DOWN> __device__ __forceinline__ void fill_bias(const BiasColumn& bias, float* lut, int sat, int tid) {
    const int mid = sat + kPad;
    for (int x0 = 0; x0 <= 2 * mid; x0 += kThreads) {
        const int x = x0 + tid;
        const float v = bias.at(DOWN ? mid - x : x - mid);
        if (x <= 2 * mid) lut[x] = v;
    }
}

// ------------------------------------------------------------------------------------------------------------ backward
// KV false: a workgroup owns query rows and walks the keys: dq and the table gradient.  KV true: it owns keys and walks the
// query rows: dk and dv.  Formulas, classes of block and the table gradient as in attn_bwd.hip; RAW leaves what is no pair out of
// the scores, dS and the table gradient.  (A row of the tile that is not finite still reaches every own row that shares a 32 x 32 block of
// pairs with one that sees it, by a product with zero, as in the general kernels.)
template <bool CAUSAL, bool KV, int SPLIT, bool RAW>
__device__ __forceinline__ bool bwd32_body(const BwdParams& p, int nblk, unsigned char* smem) {
    using G = Geom<SPLIT>;
    constexpr int OTHER = G::OTHER;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), ow = wave % G::OWNW, sub0 = (wave / G::OWNW) * 32;
    int own_block, h, b;
    bwd_place<CAUSAL, KV>(p.H, p.B, nblk, own_block, h, b);
    const int own_base = own_block * G::OWN, w_lo = own_base + ow * 32, own_row = w_lo + lr;
    const int64_t slot = ((int64_t)h * p.B + b) * nblk + own_block;     // (of the table gradient)
    if constexpr (KV && !RAW) {
        // (the last block: the shortest of a causal launch)
        if (p.slots != nullptr && p.table != nullptr && own_block == nblk - 1 && b == 0) table_grad_reduce<4>(p, h, reinterpret_cast<float*>(smem));
    }
    int M = p.M, N = p.N;
    int64_t q_first = 0, k_first = 0;
    if (p.cu_q != nullptr) {
        q_first = p.cu_q[b]; k_first = p.cu_k[b];
        M = p.len_q != nullptr ? p.len_q[b] : p.cu_q[b + 1] - (int)q_first;
        N = p.len_k != nullptr ? p.len_k[b] : p.cu_k[b + 1] - (int)k_first;
        if (own_base >= (KV ? N : M)) {     // (the grid is sized for the longest sequence)
            if constexpr (!KV) table_grad_none<4>(p, slot);
            return false;
        }
    }
    using X = Scale<RAW>;
    const int n_own = KV ? N : M, n_other = KV ? M : N, P = N - M;
    const bool has_bias = p.table != nullptr;
    const int sat = has_bias ? p.bs.sat : 0;
    float* const stats = reinterpret_cast<float*>(smem + G::STAT);
    int* const flag = reinterpret_cast<int*>(smem + G::LUT - 16);
    float* const lut = reinterpret_cast<float*>(smem + G::LUT);
    float* const dist = reinterpret_cast<float*>(smem + G::hist(sat)) + wave * table_grad_floats(sat);   // dS per distance
    float* const skew = reinterpret_cast<float*>(smem + G::skew(sat)) + wave * G::SKEW_ROWS * 64;

    auto slice = [&](const void* t, int64_t sb, int64_t sh, int64_t sr, int64_t first) {
        return reinterpret_cast<const float*>(t) + (int64_t)b * sb + (int64_t)h * sh + first * sr;
    };
    const float* const qp = slice(p.q, p.q_sb, p.q_sh, p.q_sr, q_first);
    const float* const kp = slice(p.k, p.k_sb, p.k_sh, p.k_sr, k_first);
    const float* const vp = slice(p.v, p.v_sb, p.v_sh, p.v_sr, k_first);
    const float* const gp = slice(p.dout, p.do_sb, p.do_sh, p.do_sr, q_first);
    const int64_t stat_sr = p.cu_q != nullptr ? p.H : 1;
    const int64_t stat_base = p.cu_q != nullptr ? q_first * p.H + h : ((int64_t)b * p.H + h) * p.M;

    int t_lo = 0, t_hi = (n_other + OTHER - 1) / OTHER;     // tiles that can hold a visible pair
    if (CAUSAL) {
        if (!KV) t_hi = min(t_hi, max(0, own_base + G::OWN - 1 + P + OTHER) / OTHER);
        else t_lo = max(0, own_base - P) / OTHER;
    }
    Tiles<SPLIT, RAW> tiles(KV ? qp : kp, KV ? p.q_sr : p.k_sr, KV ? gp : vp, KV ? p.do_sr : p.v_sr, n_other, tid);
    float stat = 0.f;       // KV: of the tile in registers, lse2 (threads 0 .. OTHER - 1) and delta (the next OTHER)
    auto fetch = [&](int t) {
        tiles.fetch(t);
        if (KV && tid < 2 * OTHER) {
            const int row = t * OTHER + (tid & (OTHER - 1));
            stat = tid < OTHER ? -INFINITY : 0.f;
            if (row < n_other) stat = (tid < OTHER ? p.lse2 : p.delta)[stat_base + row * stat_sr];
        }
    };
    auto store = [&](int buf) {
        tiles.store(smem + buf * G::BUF);
        if (KV && tid < 2 * OTHER) stats[buf * 2 * OTHER + tid] = tid < OTHER ? stat : stat * X::ds;
    };
    const BiasColumn bias(p, h, lane);
    if (t_lo < t_hi) fetch(t_lo);

    const bool own_ok = own_row < n_own;
    Own<SPLIT, RAW> fa, fb;
    unsigned least = fa.load(KV ? kp + (int64_t)own_row * p.k_sr : qp + (int64_t)own_row * p.q_sr, own_ok, hh, 1.f, X::down);
    fb.load(KV ? vp + (int64_t)own_row * p.v_sr : gp + (int64_t)own_row * p.do_sr, own_ok, hh, 1.f, X::up);
    float nlse2_own = -INFINITY, ndelta_own = 0.f;      // (rows past the end: every probability is 0)
    if (!KV && own_ok) { nlse2_own = p.lse2[stat_base + own_row * stat_sr]; ndelta_own = p.delta[stat_base + own_row * stat_sr]; }

    fill_bias<KV>(bias, lut, sat, tid);
    float bias_lo = 0.f, bias_hi = 0.f;
    if (has_bias) {
        bias_lo = bias.at(-sat); bias_hi = bias.at(sat);
        if constexpr (!KV) {
            for (int x = lane; x <= 2 * sat; x += 64) dist[x] = 0.f;
            for (int x = lane; x < G::SKEW_ROWS * 64; x += 64) skew[x] = 0.f;
        }
    }
    const Reads<SPLIT, RAW> reads(sub0, lane);
    f32x16 acc_a[DT], acc_b[DT];     // dQ^T or dK^T; dV^T
    clear(acc_a); clear(acc_b);
    float sum_lo = 0.f, sum_hi = 0.f;
    const float c1 = p.c1;

    if (t_lo < t_hi) { store(0); fetch(t_lo + 1); }
    asm volatile("" : "+v"(least));      // (formed here and not at the end, which would keep the rows in registers)
    ndelta_own *= X::ds;                 // (here and not where it is asked for, which would wait for it)
    for (int t = t_lo; t < t_hi; ++t) {
        const int buf = (t - t_lo) & 1;
        __syncthreads();      // tile t is written (and the LUT), the other buffer read
        const unsigned char* const ta = smem + buf * G::BUF;
        const unsigned char* const tb = ta + G::TENSOR;
        const float* const rowstat = stats + buf * 2 * OTHER + sub0 + 4 * hh;
        const int s0 = t * OTHER + sub0;
        // rel = j - (i + P): dq pass j in the tile, i own; dk / dv pass i in the tile, j own
        const int rel_min = KV ? w_lo - (s0 + 31 + P) : s0 - (w_lo + 31 + P), rel_max = rel_min + 62;
        // (the next tile is split beside the products over head_dim: one stretch of code without a branch)
        auto next = [&]() { store(buf ^ 1); fetch(t + 2); };
        if (!(s0 < n_other && (!CAUSAL || rel_min <= 0))) {
            next();
        } else {
            f32x16 s, dp;
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                f32x4 d4 = {0.f, 0.f, 0.f, 0.f};
                if constexpr (KV) d4 = *reinterpret_cast<const f32x4*>(rowstat + OTHER + 8 * r4);      // (dP starts at -delta)
#pragma unroll
                for (int e = 0; e < 4; ++e) { s[4 * r4 + e] = 0.f; dp[4 * r4 + e] = KV ? d4[e] : ndelta_own; }
            }
            reads.template over_dim<2>({ta, tb}, {&fa, &fb}, {&s, &dp});
            next();

            const bool sat_lo = rel_max <= -sat, sat_hi = rel_min >= sat;
            const bool flat = sat_lo || sat_hi;
            const float bias_c = sat_lo ? bias_lo : bias_hi;
            const float* lp = lut + (KV ? s0 + P - own_row : s0 - P - own_row) + 4 * hh + sat + kPad;
            if (flat) {
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    f32x4 l4 = {nlse2_own, nlse2_own, nlse2_own, nlse2_own};
                    if constexpr (KV) l4 = *reinterpret_cast<const f32x4*>(rowstat + 8 * r4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[4 * r4 + e] = __builtin_fmaf(c1, s[4 * r4 + e], bias_c + l4[e]);
                }
            } else {
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    f32x4 l4 = {nlse2_own, nlse2_own, nlse2_own, nlse2_own};
                    if constexpr (KV) l4 = *reinterpret_cast<const f32x4*>(rowstat + 8 * r4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[4 * r4 + e] = __builtin_fmaf(c1, s[4 * r4 + e], lp[8 * r4 + e]) + l4[e];
                }
            }
            // (row 8 (r >> 2) + (r & 3) of the lane's half: a pair from `first` on, up to `last`)
            const int first = CAUSAL && KV ? own_row - P - s0 - 4 * hh : 0;
            const int last = min(n_other - 1 - s0 - 4 * hh, CAUSAL && !KV ? own_row + P - s0 - 4 * hh : 32);
            const bool cut = RAW || s0 + 32 > n_other || (CAUSAL && rel_max > 0);
            if (cut) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int ol = 8 * (r >> 2) + (r & 3);
                    s[r] = (!(CAUSAL && KV) || ol >= first) && ol <= last && (!RAW || own_ok) ? s[r] : -INFINITY;
                }
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float pv = __builtin_amdgcn_exp2f(s[r]);
                const int ol = 8 * (r >> 2) + (r & 3);
                const bool pair = !RAW || ((!(CAUSAL && KV) || ol >= first) && ol <= last && own_ok);
                dp[r] = pair ? dp[r] * pv : 0.f;
                s[r] = pv;
            }
            if constexpr (KV) {
                if constexpr (!RAW) s *= X::up;
                reads.over_rows(tb, s, acc_b);
            }
            reads.over_rows(ta, dp, acc_a);
            if constexpr (!KV) {
                if (has_bias) {
                    if (flat) {
                        const float sum = ((dp[0] + dp[1]) + (dp[2] + dp[3])) + ((dp[4] + dp[5]) + (dp[6] + dp[7])) +
                                          ((dp[8] + dp[9]) + (dp[10] + dp[11])) + ((dp[12] + dp[13]) + (dp[14] + dp[15]));
                        if (sat_lo) sum_lo += sum; else sum_hi += sum;
                    } else {
                        table_grad_block<G::SKEW_ROWS>(skew, dist, dp, lane, rel_min + 31, sat, sum_lo, sum_hi);
                    }
                }
            }
        }
    }

    if constexpr (SPLIT > 1) {
        // the partial gradients of the second half's wavefronts, in lane order
        float* const red = reinterpret_cast<float*>(smem) + ow * ((KV ? 2 : 1) * DT * 16 * 64) + lane;
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
    }
    if constexpr (!RAW) {
        float x = odd(acc_a);
        if constexpr (KV) x += odd(acc_b);
        else if (has_bias) {
            x += (sum_lo + sum_hi) * 0.f;
            for (int y = lane; y <= 2 * sat; y += 64) x += dist[y] * 0.f;
        }
        if (anybody(flag, least < kTiny || x != x)) return true;
    }
    const float scale = p.c1 * 0.6931471805599453f;     // d score / d (q . k), natural units; dv has none
    if (own_ok && sub0 == 0) {
        float* oa = !KV ? reinterpret_cast<float*>(p.dq) + (int64_t)b * p.dq_sb + (int64_t)h * p.dq_sh + (q_first + own_row) * p.dq_sr
                        : reinterpret_cast<float*>(p.dk) + (int64_t)b * p.dk_sb + (int64_t)h * p.dk_sh + (k_first + own_row) * p.dk_sr;
        float* ob = KV ? reinterpret_cast<float*>(p.dv) + (int64_t)b * p.dv_sb + (int64_t)h * p.dv_sh + (k_first + own_row) * p.dv_sr : nullptr;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int d0 = 32 * dt + 8 * g + 4 * hh;
                auto four = [&](const f32x16& acc) { return f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]}; };
                *reinterpret_cast<f32x4*>(oa + d0) = four(acc_a[dt]) * X::back_a * scale;
                if constexpr (KV) *reinterpret_cast<f32x4*>(ob + d0) = four(acc_b[dt]) * X::back_b;
            }
    }
    if constexpr (!KV) {
        // (the tiles are done with)
        if (has_bias && p.dtable != nullptr)
            table_grad_finish<4>(p, h, slot, reinterpret_cast<const float*>(smem + G::hist(sat)), reinterpret_cast<float*>(smem), sat, sum_lo, sum_hi, X::ds_back);
    }
    return false;
}

template <bool CAUSAL, bool KV, int SPLIT>
__global__ __launch_bounds__(kThreads, SPLIT == 2 || KV ? 1 : 2) void bwd32_kernel(const BwdParams p, int nblk) {
    extern __shared__ __attribute__((aligned(16))) unsigned char f32_smem[];
    if (bwd32_body<CAUSAL, KV, SPLIT, false>(p, nblk, f32_smem)) {
        __syncthreads();
        bwd32_body<CAUSAL, KV, SPLIT, true>(p, nblk, f32_smem);
    }
}

// ------------------------------------------------------------------------------------------------------------- forward
template <bool CAUSAL, int SPLIT, bool RAW>
__device__ __forceinline__ bool fwd32_body(const FwdParams& p, int nblk, unsigned char* smem) {
    using G = Geom<SPLIT>;
    constexpr int OTHER = G::OTHER;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), ow = wave % G::OWNW, sub0 = (wave / G::OWNW) * 32;
    int own_block, h, b;
    bwd_place<CAUSAL, false>(p.H, p.B, nblk, own_block, h, b);
    const int own_base = own_block * G::OWN, w_lo = own_base + ow * 32, own_row = w_lo + lr;
    using X = Scale<RAW>;
    const int M = p.M, N = p.N, P = N - M;
    const bool has_bias = p.table != nullptr;
    const int sat = has_bias ? p.bs.sat : 0;
    int* const flag = reinterpret_cast<int*>(smem + G::LUT - 16);
    float* const lut = reinterpret_cast<float*>(smem + G::LUT);

    auto slice = [&](const void* t, int64_t sb, int64_t sh) { return reinterpret_cast<const float*>(t) + (int64_t)b * sb + (int64_t)h * sh; };
    int t_hi = (N + OTHER - 1) / OTHER;
    if (CAUSAL) t_hi = min(t_hi, max(0, own_base + G::OWN - 1 + P + OTHER) / OTHER);
    Tiles<SPLIT, RAW> tiles(slice(p.k, p.k_sb, p.k_sh), p.k_sr, slice(p.v, p.v_sb, p.v_sh), p.v_sr, N, tid);
    const BiasColumn bias(p, h, lane);
    if (t_hi > 0) tiles.fetch(0);
    const bool own_ok = own_row < M;
    Own<SPLIT, RAW> own;
    unsigned least = own.load(slice(p.q, p.q_sb, p.q_sh) + (int64_t)own_row * p.q_sr, own_ok, hh, p.c1, X::down);
    fill_bias<false>(bias, lut, sat, tid);
    const float bias_lo = has_bias ? bias.at(-sat) : 0.f, bias_hi = has_bias ? bias.at(sat) : 0.f;
    const Reads<SPLIT, RAW> reads(sub0, lane);
    f32x16 acc[DT];      // O^T
    clear(acc);
    float top = -INFINITY, sum = 0.f;     // running maximum of the row (base-2 units), this lane's share of the sum

    if (t_hi > 0) { tiles.store(smem); tiles.fetch(1); }
    asm volatile("" : "+v"(least));
    __syncthreads();      // (the LUT is written)
    for (int t = 0; t < t_hi; ++t) {
        const unsigned char* const tk = smem + (t & 1) * G::BUF;
        const int s0 = t * OTHER + sub0;
        const int rel_min = s0 - (w_lo + 31 + P), rel_max = rel_min + 62;
        const bool active = s0 < N && (!CAUSAL || rel_min <= 0);
        // (the products start at bias - running maximum, which is at hand ahead of the tile)
        const float ref = top > -INFINITY ? top : 0.f;
        f32x16 s;
        if (active) {
            const bool sat_lo = rel_max <= -sat, sat_hi = rel_min >= sat;
            if (sat_lo || sat_hi) {
                const float c = (sat_lo ? bias_lo : bias_hi) - ref;
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = c;
            } else {
                const float* lp = lut + s0 - P - own_row + 4 * hh + sat + kPad;
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = lp[8 * (r >> 2) + (r & 3)] - ref;
            }
        }
        __syncthreads();      // (tile t is written, the other buffer read)
        auto next = [&]() { tiles.store(smem + ((t + 1) & 1) * G::BUF); tiles.fetch(t + 2); };
        if (!active) {
            next();
        } else {
            reads.template over_dim<1>({tk}, {&own}, {&s});
            next();
            if (s0 + 32 > N || (CAUSAL && rel_max > 0)) {
                const int last = min(N - 1 - s0 - 4 * hh, CAUSAL ? own_row + P - s0 - 4 * hh : 32);
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = 8 * (r >> 2) + (r & 3) <= last ? s[r] : -INFINITY;
            }
            float most = s[0];
#pragma unroll
            for (int r = 1; r < 16; ++r) most = fmaxf(most, s[r]);
            // the running maximum is raised when a score exceeds it by more than 2^24, or there was none (sums and rows are
            // divided by the same one)
            const float limit = top > -INFINITY ? 24.f : -INFINITY;
            if (__any(most > limit)) {
                most = fmaxf(most, __shfl_xor(most, 32, 64));
                const float up = most > limit ? most : 0.f, f = top > -INFINITY ? __builtin_amdgcn_exp2f(-up) : 0.f;
                top = most > limit ? ref + up : top;
                sum *= f;
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] -= up;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[dt][r] *= f;
            }
            float part = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) { s[r] = __builtin_amdgcn_exp2f(s[r]); part += s[r]; }
            sum += part;
            if constexpr (!RAW) s *= X::up;
            reads.over_rows(tk + G::TENSOR, s, acc);
        }
    }

    if constexpr (SPLIT > 1) {
        float* const red = reinterpret_cast<float*>(smem) + ow * ((DT * 16 + 2) * 64) + lane;
        __syncthreads();
        if (sub0 != 0) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) red[(dt * 16 + r) * 64] = acc[dt][r];
            red[DT * 16 * 64] = top; red[(DT * 16 + 1) * 64] = sum;
        }
        __syncthreads();
        if (sub0 == 0) {
            const float other = red[DT * 16 * 64], both = fmaxf(top, other), ref = both > -INFINITY ? both : 0.f;
            const float f = __builtin_amdgcn_exp2f(top - ref), g = __builtin_amdgcn_exp2f(other - ref);
            top = both;
            sum = sum * f + red[(DT * 16 + 1) * 64] * g;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[dt][r] = acc[dt][r] * f + red[(dt * 16 + r) * 64] * g;
        }
    }
    sum += __shfl_xor(sum, 32, 64);
    if constexpr (!RAW) {
        const float x = odd(acc) + sum * 0.f;
        if (anybody(flag, least < kTiny || x != x)) return true;
    }
    if (own_ok && sub0 == 0) {
        const float inv = (sum == 0.f ? 0.f : 1.0f / sum) * X::back_b;      // (a row without a visible key: zeros)
        float* const o = reinterpret_cast<float*>(p.o) + (int64_t)b * p.o_sb + (int64_t)h * p.o_sh + (int64_t)own_row * p.o_sr;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *reinterpret_cast<f32x4*>(o + 32 * dt + 8 * g + 4 * hh) =
                    f32x4{acc[dt][4 * g] * inv, acc[dt][4 * g + 1] * inv, acc[dt][4 * g + 2] * inv, acc[dt][4 * g + 3] * inv};
        if (p.lse != nullptr && hh == 0)
            p.lse[(int64_t)b * p.lse_sb + (int64_t)h * p.lse_sh + (int64_t)own_row * p.lse_sr] =
                sum == 0.f ? -INFINITY : (top + __builtin_amdgcn_logf(sum)) * 0.6931471805599453f;
    }
    return false;
}

template <bool CAUSAL, int SPLIT>
__global__ __launch_bounds__(kThreads, 2) void fwd32_kernel(const FwdParams p, int nblk) {
    extern __shared__ __attribute__((aligned(16))) unsigned char f32_smem[];
    if (fwd32_body<CAUSAL, SPLIT, false>(p, nblk, f32_smem)) {
        __syncthreads();
        fwd32_body<CAUSAL, SPLIT, true>(p, nblk, f32_smem);
    }
}

template <bool CAUSAL, bool KV, int SPLIT>
hipError_t launch_bwd(const BwdParams& p, hipStream_t stream) {
    const int rows = KV ? p.N : p.M;
    if (rows <= 0) return hipSuccess;
    const int nblk = (rows + Geom<SPLIT>::OWN - 1) / Geom<SPLIT>::OWN;
    const int64_t blocks = (int64_t)nblk * p.H * p.B;
    if (blocks > 0x7fffffff) return hipErrorInvalidConfiguration;
    const int lds = Geom<SPLIT>::bytes(p.table != nullptr ? p.bs.sat : 0, !KV && p.table != nullptr);
    auto kern = bwd32_kernel<CAUSAL, KV, SPLIT>;
    static LdsLimit limit;
    const hipError_t e = limit.allow(reinterpret_cast<const void*>(kern), lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kThreads), lds, stream, p, nblk);
    return hipGetLastError();
}
template <bool CAUSAL, int SPLIT>
hipError_t launch_fwd(const FwdParams& p, hipStream_t stream) {
    const int nblk = (p.M + Geom<SPLIT>::OWN - 1) / Geom<SPLIT>::OWN;
    const int64_t blocks = (int64_t)nblk * p.H * p.B;
    if (blocks > 0x7fffffff) return hipErrorInvalidConfiguration;
    const int lds = Geom<SPLIT>::bytes(p.table != nullptr ? p.bs.sat : 0, false);
    auto kern = fwd32_kernel<CAUSAL, SPLIT>;
    static LdsLimit limit;
    const hipError_t e = limit.allow(reinterpret_cast<const void*>(kern), lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kThreads), lds, stream, p, nblk);
    return hipGetLastError();
}

// Whether blocks of 64 rows are taken (SPLIT 2) in place of 128: where they are one round of one workgroup per compute unit
// (what their LDS allows), and with a causal mask, where the longest block counts, up to two and a half.  us, SPLIT 2 / 1,
// forward and backward (before the operands were scaled): blocks of 64 rows 256 (B4 H8 L512) 26 / 33 and 77 / 114; 320 (B5 H8 L512) 44 / 31 and 132 / 116; 384 (B2 H8
// L1500) 102 / 77 and 292 / 276; 192 (B32 H6 L64) 14 / 16 and 34 / 39; causal 512 (B4 H8 L1000) 46 / 54 and 142 / 198, 576 (B3 H6
// L2000) 96 / 98 and 284 / 362, 768 (B4 H12 L1000) 71 / 59 and 216 / 203.
bool few(int rows, int64_t pairs, bool causal) { return ((int64_t)(rows + 63) / 64) * pairs <= (causal ? 640 : 256); }

}  // namespace

hipError_t launch_fwd_f32_64(const FwdParams& p, bool causal, hipStream_t stream) {
    const bool split = few(p.M, (int64_t)p.H * p.B, causal);
    if (causal) return split ? launch_fwd<true, 2>(p, stream) : launch_fwd<true, 1>(p, stream);
    return split ? launch_fwd<false, 2>(p, stream) : launch_fwd<false, 1>(p, stream);
}

template <bool CAUSAL> static hipError_t launch_passes(BwdParams p, hipStream_t stream) {
    const int64_t pairs = (int64_t)p.H * p.B;
    // (bucketings that saturate past distance 779 leave no room for the larger tiles next to the table gradient's sums)
    const bool room = Geom<2>::bytes(p.table != nullptr ? p.bs.sat : 0, p.table != nullptr) <= 160 * 1024;
    const bool split = room && few(p.M, pairs, CAUSAL);
    p.slots_per_head = p.B * (split ? (p.M + 63) / 64 : (p.M + 127) / 128);
    if (p.N <= 0) p.slots = nullptr;      // (no pass that would add them)
    const hipError_t e = split ? launch_bwd<CAUSAL, false, 2>(p, stream) : launch_bwd<CAUSAL, false, 1>(p, stream);
    if (e != hipSuccess) return e;
    return few(p.N, pairs, CAUSAL) ? launch_bwd<CAUSAL, true, 2>(p, stream) : launch_bwd<CAUSAL, true, 1>(p, stream);
}
hipError_t launch_bwd_f32_64(BwdParams p, bool causal, hipStream_t stream) { return causal ? launch_passes<true>(p, stream) : launch_passes<false>(p, stream); }

}  // namespace t5a
