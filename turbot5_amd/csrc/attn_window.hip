// Sliding-window attention, with or without side tokens (the local and transient-global patterns), for 16-bit tensors at
// head_dim 64 with or without padding around the sequences: src/turbot5/model/attentions.py:583-638, :977-1052 as one kernel.
//
// A workgroup owns 128 query rows, 32 per wavefront, and walks key tiles of 32 or 64 rows: those within the window of any of
// its rows, then the side tokens.  Per 32 keys a wavefront whose window reaches them forms one block
//   S^T = K Q^T (a lane owns one query and 16 of the keys), P^T = exp2(S^T + bias - m), O^T += V^T P^T
// with V read through the transposing LDS read, whose row order is that of the accumulator: P goes from accumulator
// registers to the next operand by a conversion.  The bias is a word per distance in LDS, consecutive rows consecutive
// words; the window is folded into it (-inf from the window's edge on), so only the last tile of a sequence is masked per
// element.  Side tokens at saturated distances take a constant instead.
//
// The row maximum m is raised only when a score exceeds it by more than 2^14 (probabilities stay finite in either type,
// the sums are fp32, and dividing by the sum at the end undoes whatever m was), or at a row's first visible key; the wavefront
// asks that of all its rows with one vote per block and shifts what it has in a block of code that is rarely run.
//
// What bounds it: waits and the vector port.  At B1 H12 L16384, window 128, the wavefronts wait 51 % of their cycles, for each
// other at the barrier of a tile; the vector port is busy 54 % of the time, the matrix pipe 20 % (with side tokens every 16:
// 36, 57 and 30 %); per block and lane it is 16 x (fma, subtract, exp2, half a max3, half a conversion and half a dot
// product) against eight matrix products.  More wavefronts per SIMD (5) or more tile buffers (4) were slower.  The general
// kernel (fwd_kernel) walks rings of eight 64-key tiles per 128 rows with a scalar prologue that eight wavefronts per
// compute unit execute at one instruction a cycle; this one has next to none, and a window of 255 keys costs 9 or 10 blocks
// of 32 keys.  us, general kernel / this one, bf16, 12 heads, window 128: L16384 37.9 / 34.6, L32768 75 / 62, 8 x 1024 27 /
// 21; L16384 with window 64 32.0 / 27.4, 256 56.5 / 52.8.  With side tokens and where the line between the two kernels lies:
// takes_window_kernel.
#include "lut_device.h"
#include "mfma16_device.h"
#include "t5a_internal.h"

namespace t5a {

namespace {

constexpr int kWinThreads = 256, kWinOwn = 128, kWinD = 64;
// rows per key tile: 32, or 64 with side tokens, where a row of tiles is long enough for fewer barriers to pay (B1 H12
// L16384, window 128, aux 16: 125 us with 32, 97 with 64; without side tokens 35.8 and 37.5)
__host__ __device__ constexpr int win_tile(bool side) { return side ? 64 : 32; }
// byte offset of the LUTs: two buffers of a K and a V tile come first
__host__ __device__ constexpr int win_lut_at(bool side) { return 4 * win_tile(side) * kWinD * 2; }
constexpr float kWinRaise = 14.f;              // base-2 margin of the running maximum

// words of the window's LUT (distances of a block that touches the window) and of the side tokens' (padded by 64, more
// than a lane's rows of a block span)
__host__ __device__ inline int win_lut_words(int w) { return (2 * (w + 62) + 4) & ~3; }
__host__ __device__ inline int side_lut_words(int sat) { return (2 * (sat + 64) + 4) & ~3; }

template <typename T, bool SIDE>
__global__ __launch_bounds__(kWinThreads, 4) void window16_kernel(const FwdParams p, int nblk) {
    constexpr int kWinTile = win_tile(SIDE), kWinTileBytes = kWinTile * kWinD * 2;
    constexpr int D = kWinD, DT = D / 32, KS = D / 16;
    using H16 = Half16<T>;
    using v8 = typename H16::v8;
    extern __shared__ __attribute__((aligned(16))) unsigned char win_smem[];
    __shared__ int again;

    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int blk, h, b;
    // Workgroups go to the eight XCDs in turn; each takes one contiguous piece of the (head, sequence, rows) list, so that
    // neighbouring rows, whose windows share most of their keys, find them in one L2.
    {
        const int total = nblk * p.H * p.B, piece = (total + 7) >> 3, item = (blockIdx.x & 7) * piece + (blockIdx.x >> 3);
        if (item >= total) return;
        const int pair = item / nblk;
        blk = item - pair * nblk; h = pair / p.B; b = pair - h * p.B;
    }
    const int L = p.M, w = p.block_len;
    const int q0 = blk * kWinOwn, w_lo = q0 + wave * 32, own_row = w_lo + lr;
    const bool has_bias = p.table != nullptr;
    const int sat = has_bias ? p.bs.sat : 0;
    // A padded sequence's tokens are the rows [key_lo, key_hi); a token's position stays its row index.  Side tokens: one per
    // block end among the tokens, the rest of them joining the last one (src/turbot5/model/utils.py:191-237 for one run)
    int key_lo = 0, key_hi = L, n_side = SIDE ? p.n_side : 0;
    if (p.len_k != nullptr) {
        key_lo = p.start_k != nullptr ? max(0, min(L, p.start_k[b])) : 0;
        key_hi = max(key_lo, min(L, key_lo + max(0, p.len_k[b])));
        if (SIDE) n_side = min(n_side, key_hi / p.aux - key_lo / p.aux);
    }
    float* const lut = reinterpret_cast<float*>(win_smem + win_lut_at(SIDE));
    float* const lut_side = lut + win_lut_words(w);

    const T* qp = reinterpret_cast<const T*>(p.q) + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
    const T* kp = reinterpret_cast<const T*>(p.k) + (int64_t)b * p.k_sb + (int64_t)h * p.k_sh;
    const T* vp = reinterpret_cast<const T*>(p.v) + (int64_t)b * p.v_sb + (int64_t)h * p.v_sh;
    const T* skp = SIDE ? reinterpret_cast<const T*>(p.side_k) + (int64_t)b * p.sk_sb + (int64_t)h * p.sk_sh : kp;
    const T* svp = SIDE ? reinterpret_cast<const T*>(p.side_v) + (int64_t)b * p.sv_sb + (int64_t)h * p.sv_sh : vp;

    // tiles: n_win of the window, from row k0 on (tiles are counted from the sequence's first token), then the side tokens'
    const int k0 = key_lo + max(0, q0 - (w - 1) - key_lo) / kWinTile * kWinTile;
    const int n_win = max(0, min(key_hi, q0 + kWinOwn - 1 + w) - k0 + kWinTile - 1) / kWinTile;
    const int n_tiles = n_win + (n_side + kWinTile - 1) / kWinTile;

    // staging by LDS-DMA, one request of 1 KB (8 rows) per wavefront and tensor; the chunk swizzle is applied on the
    // source side, rows past the end of a tensor are out of the descriptor's range and arrive as zeros (slices stay
    // below 2 GiB -- checked on the host -- and the row is clamped to one past the end, so 32-bit offsets do)
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)win_smem;
    // (the swizzle repeats every 16 rows: a wavefront's further slabs are 32 rows on)
    const int dma_row = wave * 8 + (lane >> 3), dma_ch = ((lane & 7) ^ tile_swz(dma_row)) * 16;
    auto request = [&](int t, int buf) {
        const bool side = SIDE && t >= n_win;
        const int rows = side ? n_side : key_hi;
        const int row0 = side ? (t - n_win) * kWinTile : k0 + t * kWinTile;
        const int k_srb = (int)(side ? p.sk_sr : p.k_sr) * 2, v_srb = (int)(side ? p.sv_sr : p.v_sr) * 2;
        const u32x4 rs_k = dma_rsrc(side ? skp : kp, (unsigned)(rows - 1) * (unsigned)k_srb + D * 2);
        const u32x4 rs_v = dma_rsrc(side ? svp : vp, (unsigned)(rows - 1) * (unsigned)v_srb + D * 2);
#pragma unroll
        for (int c = 0; c < kWinTile / 32; ++c) {
            const int row = min(row0 + 32 * c + dma_row, rows);
            const unsigned at = lds0 + buf * (2 * kWinTileBytes) + c * 4096u + wave * 1024u;
            dma_16(rs_k, at, row * k_srb + dma_ch);
            dma_16(rs_v, at + kWinTileBytes, row * v_srb + dma_ch);
        }
    };
    if (n_tiles > 0) request(0, 0);
    if (SIDE && tid == 0) again = 0;

    // the query row as B operands: lane (lr, hh) holds elements 16 s + 8 hh .. + 7; multiplied by the score factor and
    // rounded back unless the factor is to be applied to the product
    v8 fq[KS];
    {
        const T* q = qp + (int64_t)own_row * p.q_sr;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
#pragma unroll
            for (int e = 0; e < 8; ++e) fq[s][e] = (T)0.0f;
            if (own_row < L) fq[s] = *reinterpret_cast<const v8*>(q + 16 * s + 8 * hh);
        }
        if (!p.exact_scale)
#pragma unroll
            for (int s = 0; s < KS; ++s)
#pragma unroll
                for (int e = 0; e < 8; ++e) fq[s][e] = (T)((float)fq[s][e] * p.c1);
    }
    const float c1 = p.exact_scale ? p.c1 : 1.0f;

    auto bias_at = [&](int rel) {
        return has_bias ? load_table(p.table, p.table_dtype, (int64_t)bucket_of(p.bs, rel) * p.t_sbucket + (int64_t)h * p.t_shead) * 1.4426950408889634f : 0.f;
    };
    for (int x = tid; x <= 2 * (w + 62); x += kWinThreads) {
        const int rel = x - (w + 62);
        lut[x] = rel > -w && rel < w ? bias_at(rel) : -INFINITY;
    }
    const int mid = sat + 64;
    float bias_lo = 0.f, bias_hi = 0.f;
    // side tokens: this row's own one, and the wavefront's first and last
    int own_side = 0, side_lo = 0, side_hi = 0;
    if (SIDE && n_side > 0) {
        for (int x = tid; x <= 2 * mid; x += kWinThreads) lut_side[x] = bias_at(x - mid);
        bias_lo = bias_at(-sat); bias_hi = bias_at(sat);
        own_side = min(own_row / p.aux, n_side - 1);
        side_lo = min(w_lo / p.aux, n_side - 1);
        side_hi = min((w_lo + 31) / p.aux, n_side - 1);
    }

    // row reads: element offsets of this lane's chunk (2 s + hh) of row lr; transposing reads as in attn_bwd.hip
    int row_off[KS], tr_lo[DT], tr_hi[DT];
#pragma unroll
    for (int s = 0; s < KS; ++s) row_off[s] = lr * D + (((2 * s + hh) ^ tile_swz(lr)) * 8);
    {
        const int g = lane >> 4, r = lane & 15, jj = r >> 2, aa = r & 3;
        const int row = 4 * (g >> 1) + jj, x = 2 * (g & 1) + (aa >> 1);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            tr_lo[dt] = row * D + (((4 * dt + x) ^ tile_swz(row)) * 8) + (aa & 1) * 4;
            tr_hi[dt] = (row + 8) * D + (((4 * dt + x) ^ tile_swz(row + 8)) * 8) + (aa & 1) * 4;
        }
    }
    auto tr_frag = [&](const T* tile, int g16, int dt) {
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(tile + tr_lo[dt] + 16 * g16 * D));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(tile + tr_hi[dt] + 16 * g16 * D));
        return __builtin_bit_cast(v8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };

    f32x16 acc[DT];
    float m, sums[2];      // what is subtracted from the row's scores; this lane half's sum, in two parts
    float limit;            // a shifted score above it raises m (any, until the row's first visible key)
    // A key row of NaN or infinity is not outweighed by the folded -inf.  With side tokens it has to stay with the rows that see
    // it (the general kernel masks that pattern per element, and folds the local one as this does): a workgroup with a NaN
    // among its sums goes over its tiles once more with every window block masked per element.  (The mask in every block at
    // a window's edge, or asked for by the block's own sums, took 2 us of launches of 25 to 75.)
    bool masked = false;
again_masked:
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[dt][r] = 0.f;
    m = 0.f; sums[0] = 0.f; sums[1] = 0.f;
    limit = -INFINITY;

    // (kept a loop: unrolled by two it takes 128 registers and 39.9 us where this takes 110 and 35.8)
#pragma unroll 1
    for (int t = 0, buf = 0; t < n_tiles; ++t, buf ^= 1) {
        wait_vmcnt<0>();     // this wavefront's requests for tile t have landed
        __syncthreads();                        // ... and everybody's; the other buffer is free (and, first time round, the LUTs written)
        if (t + 1 < n_tiles) request(t + 1, buf ^ 1);
        const bool side = SIDE && t >= n_win;
        const int rows = side ? n_side : key_hi;
#pragma unroll 1
        for (int nt = 0; nt < kWinTile / 32; ++nt) {
            const T* tk = reinterpret_cast<const T*>(win_smem + buf * 2 * kWinTileBytes) + nt * 32 * D;
            const T* tv = tk + kWinTileBytes / 2;
            const int s0 = (side ? (t - n_win) * kWinTile : k0 + t * kWinTile) + 32 * nt;
            // (wavefront-uniform) rows past the sequence have nothing to do, nor has a tile outside the wavefront's window
            if (w_lo < L && (!SIDE || s0 < rows) && (side || (s0 + 31 > w_lo - w && s0 < w_lo + 31 + w))) {
                f32x16 s;
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
                for (int k = 0; k < KS; ++k) s = H16::mfma(*reinterpret_cast<const v8*>(tk + row_off[k]), fq[k], s);
                const bool sat_lo = side && s0 + 31 - side_lo <= -sat, sat_hi = side && s0 - side_hi >= sat;
                if (sat_lo || sat_hi) {
                    const float bm = (sat_lo ? bias_lo : bias_hi) - m;
#pragma unroll
                    for (int r = 0; r < 16; ++r) s[r] = __builtin_fmaf(c1, s[r], bm);
                } else {
                    // (a lane whose distances are all saturated reads the pad, which holds that side's last bucket)
                    const float* lp = side ? lut_side + min(max(s0 - own_side + 4 * hh + mid, 0), 2 * mid - 32)
                                           : lut + s0 - own_row + 4 * hh + w + 62;
#pragma unroll
                    for (int r = 0; r < 16; ++r) s[r] = __builtin_fmaf(c1, s[r], lp[8 * (r >> 2) + (r & 3)]) - m;
                }
                if (masked || s0 + 32 > rows) {
                    const int ends = rows - s0 - 4 * hh;
                    const int first = SIDE && !side ? own_row - w + 1 - s0 - 4 * hh : 0;
                    const int last = SIDE && !side ? min(ends, own_row + w - s0 - 4 * hh) : ends;
#pragma unroll
                    for (int r = 0; r < 16; ++r) s[r] = (!SIDE || 8 * (r >> 2) + (r & 3) >= first) && 8 * (r >> 2) + (r & 3) < last ? s[r] : -INFINITY;
                }
                float top = fmaxf(fmaxf(s[0], s[1]), s[2]);
#pragma unroll
                for (int r = 3; r < 15; r += 2) top = fmaxf(fmaxf(top, s[r]), s[r + 1]);
                top = fmaxf(top, s[15]);
                if (__builtin_amdgcn_ballot_w64(top > limit) != 0) {
                    top = fmaxf(top, __shfl_xor(top, 32, 64));      // the row's other 16 keys
                    const bool raise = top > limit;
                    const float shift = raise ? top : 0.f;
                    const float keep = !raise ? 1.f : limit == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(-shift);
                    limit = raise ? kWinRaise : limit;
                    m += shift;
                    sums[0] *= keep; sums[1] *= keep;
#pragma unroll
                    for (int r = 0; r < 16; ++r) s[r] -= shift;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                        for (int r = 0; r < 16; ++r) acc[dt][r] *= keep;
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = __builtin_amdgcn_exp2f(s[r]);
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const v8 pb = to_frag<v8>(s, u);
                    // (of the rounded probabilities: a row with one large one then divides by exactly what it was multiplied by)
#pragma unroll
                    for (int e = 0; e < 4; ++e) sums[e & 1] = H16::pair_sum(typename H16::v2{pb[2 * e], pb[2 * e + 1]}, sums[e & 1]);
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) acc[dt] = H16::mfma(tr_frag(tv, u, dt), pb, acc[dt]);
                }
            }
        }
    }

    float sum = sums[0] + sums[1];
    sum += __shfl_xor(sum, 32, 64);
    if (SIDE && !masked && n_tiles > 0) {
        if (__builtin_amdgcn_ballot_w64(sum != sum) != 0) again = 1;
        __syncthreads();      // (and every wavefront is done with the tile buffers)
        if (again != 0) {
            masked = true;
            request(0, 0);
            goto again_masked;
        }
    }
    const float inv = sum > 0.f || sum != sum ? 1.0f / sum : 0.f;      // (a row without a visible key: zeros)
    // A lane holds elements 8 g + 4 hh .. + 3 of its row, the lane 32 further on the other halves: they exchange, and each
    // writes 16 bytes of every second group of eight.
    typedef T t4 __attribute__((ext_vector_type(4)));
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    T* o = reinterpret_cast<T*>(p.o) + (int64_t)b * p.o_sb + (int64_t)h * p.o_sh + (int64_t)own_row * p.o_sr;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int g = 0; g < 4; g += 2) {
            u32x2 lo, hi;
            t4 x, y;
#pragma unroll
            for (int e = 0; e < 4; ++e) { x[e] = (T)(acc[dt][4 * g + e] * inv); y[e] = (T)(acc[dt][4 * g + 4 + e] * inv); }
            lo = __builtin_bit_cast(u32x2, x); hi = __builtin_bit_cast(u32x2, y);
            const auto a0 = __builtin_amdgcn_permlane32_swap(lo[0], hi[0], false, false);
            const auto a1 = __builtin_amdgcn_permlane32_swap(lo[1], hi[1], false, false);
            if (own_row < L)
                *reinterpret_cast<u32x4*>(o + 32 * dt + 8 * (g + hh)) = u32x4{a0[0], a1[0], a0[1], a1[1]};
        }
}

template <typename T>
hipError_t launch_window_t(const FwdParams& p, bool side, hipStream_t stream) {
    const int nblk = (p.M + kWinOwn - 1) / kWinOwn;
    const int64_t blocks = (int64_t)nblk * p.H * p.B;
    const int64_t grid = (blocks + 7) / 8 * 8;
    if (grid > 0x7fffffff) return hipErrorInvalidConfiguration;
    const int lds = win_lut_at(side) + 4 * (win_lut_words(p.block_len) + (side ? side_lut_words(p.table != nullptr ? p.bs.sat : 0) : 0));
    if (side) hipLaunchKernelGGL((window16_kernel<T, true>), dim3((unsigned)grid), dim3(kWinThreads), lds, stream, p, nblk);
    else hipLaunchKernelGGL((window16_kernel<T, false>), dim3((unsigned)grid), dim3(kWinThreads), lds, stream, p, nblk);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_window(const FwdParams& p, int dtype, bool side, hipStream_t stream) {
    if (dtype == T5A_BF16) return launch_window_t<__bf16>(p, side, stream);
    if (dtype == T5A_F16) return launch_window_t<_Float16>(p, side, stream);
    return hipErrorInvalidValue;
}

}  // namespace t5a
