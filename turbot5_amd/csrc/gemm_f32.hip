// Products of fp32 matrices on the 16-bit matrix cores: the linear layers of a training step with fp32 weights and their
// gradients.  What bounds them: at thousands of rows the matrix cores and, next to them, the vector instructions that split the
// operands, some 160 of a thread beside 24 products per step of the larger tile (8192 x 2048 x 512: 112 us, 6 matrix products in
// bf16 at 920 TFLOP/s; a library product in bf16 reaches 1214), below that the latency of a workgroup's steps.
// The factor 2^16 on the operands (split_device.h), one of those instructions per value, takes 1 to 3 %: 65.3 / 67.1 us without / with it at 4500 x 2048 x 512,
// 108 / 112 at 8192 x 2048 x 512.  A test for lost bits in its place, half an instruction per value, with the scaled products
// as its way out: 66.5 and 110, a training step of the T5-small encoder the same, for a second copy of the loop.
#include <type_traits>

#include "gemm_offsets.h"
#include "split_device.h"
#include "t5a_internal.h"

namespace t5a {

namespace {

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int BK = kGemmStep;   // depth of a staged tile

// An operand's tile in LDS: planes of bf16.  ROWS values along the output dimension, BK along the contraction.
// COL false: the matrix is (rows, contraction) with the contraction contiguous; the plane holds rows of 64 bytes, four chunks of
// eight values, read as they lie.  COL true: (contraction, rows) with the rows contiguous; the plane holds BK rows of 2 ROWS
// bytes and is read through the transposing LDS read.
template <typename T, bool COL, int ROWS>
struct Operand {
    static constexpr int NP = sizeof(T) == 4 ? 3 : 1;
    static constexpr int PLANE = ROWS * BK;                 // elements
    static constexpr int PASSES = ROWS / 64;                // eight values per thread and pass
    typedef T v8 __attribute__((ext_vector_type(8)));
    static constexpr int CPR = ROWS / 8;                    // COL: chunks per row of the plane

    // transposing reads hand lane half hh the plane rows 4 hh .. + 3 and 8 + 4 hh .. + 3 of every sixteen; row reads the
    // values 8 hh .. + 7.  Rows are placed so that both see the contraction in the same order.
    static __device__ __forceinline__ int plane_row(int k) { return (k & ~12) | ((k & 4) << 1) | ((k & 8) >> 1); }
    static __device__ __forceinline__ int swz(int row) {
        if constexpr (!COL) return (row >> 2) & 3;
        else if constexpr (ROWS == 128) return ((row & 3) << 2) | ((row >> 2) & 3);
        else return tile_swz(row);
    }

    // A lane's pieces of a tile, eight values each.  Read through a buffer descriptor, whose scalar offset advances with the
    // contraction; what lies past the contraction's end is asked for out of the descriptor's range and arrives as zero
    // (gemm_offsets.h).
    struct Tile { v8 x[PASSES]; };
    __amdgpu_buffer_rsrc_t rs;
    int at[PASSES], k[PASSES], step;
    __device__ __forceinline__ void start(const T* p, int64_t ld, int base, int rows, int K, int tid) {
        rs = __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, operand_bytes(COL ? K : rows, COL ? rows : K, ld, (int)sizeof(T)), 0x00020000);
        step = step_bytes(K, COL ? ld : 1, (int)sizeof(T));
#pragma unroll
        for (int n = 0; n < PASSES; ++n) {
            const int c = tid + n * kThreads;
            // (rows past the end: the last ones again; their results are not stored)
            const int row = COL ? min(base + (c % CPR) * 8, rows - 8) : min(base + (c >> 2), rows - 1);
            k[n] = COL ? c / CPR : (c & 3) * 8;
            at[n] = (COL ? min(k[n], K - 1) * (int)ld + row : row * (int)ld + k[n]) * (int)sizeof(T);
        }
    }
    // step kk of the contraction, of which K - kk BK indices are left
    __device__ __forceinline__ void fetch(Tile& t, int kk, int K) const {
        const int from = step_offset(kk, K, step);
#pragma unroll
        for (int n = 0; n < PASSES; ++n) {
            const int off = lane_offset(k[n], kk, K, at[n]);
            u32x4* const d = reinterpret_cast<u32x4*>(&t.x[n]);
#pragma unroll
            for (int e = 0; e < (int)sizeof(v8) / 16; ++e) d[e] = __builtin_amdgcn_raw_buffer_load_b128(rs, off + 16 * e, from, 0);
        }
    }
    static __device__ __forceinline__ void store(const Tile& t, __bf16* plane, int tid) {
#pragma unroll
        for (int n = 0; n < PASSES; ++n) {
            const int c = tid + n * kThreads;
            int to;
            if constexpr (!COL) { const int row = c >> 2; to = row * BK + ((c & 3) ^ swz(row)) * 8; }
            else { const int row = plane_row(c / CPR); to = row * ROWS + ((c % CPR) ^ swz(row)) * 8; }
            if constexpr (NP == 3) {
                bf16x8 s[3];
                split3(t.x[n] * kSplitScale, s);
#pragma unroll
                for (int q = 0; q < 3; ++q) *reinterpret_cast<bf16x8*>(plane + q * PLANE + to) = s[q];
            } else {
                *reinterpret_cast<v8*>(plane + to) = t.x[n];
            }
        }
    }
    // the 32 rows from r0 on, values 16 s .. + 15 of the contraction
    static __device__ __forceinline__ void frag(const __bf16* plane, int r0, int s, int lane, bf16x8 (&out)[NP]) {
        if constexpr (!COL) {
            const int row = r0 + (lane & 31), at = row * BK + ((2 * s + (lane >> 5)) ^ swz(row)) * 8;
#pragma unroll
            for (int q = 0; q < NP; ++q) out[q] = *reinterpret_cast<const bf16x8*>(plane + q * PLANE + at);
        } else {
            const int g = lane >> 4, jj = (lane >> 2) & 3, aa = lane & 3;
            const int row = 16 * s + 4 * (g >> 1) + jj, ch = r0 / 8 + 2 * (g & 1) + (aa >> 1);
            const int lo = row * ROWS + (ch ^ swz(row)) * 8 + (aa & 1) * 4;
            const int hi = (row + 8) * ROWS + (ch ^ swz(row + 8)) * 8 + (aa & 1) * 4;
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(plane + q * PLANE + lo));
                const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(plane + q * PLANE + hi));
                out[q] = __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
            }
        }
    }
    // one value, for the products in fp32
    static __device__ __forceinline__ float value(const T* p, int64_t ld, int row, int rows, int k, int K) {
        if (k >= K) return 0.f;
        row = min(row, rows - 1);
        return (float)(COL ? p[k * ld + row] : p[row * ld + k]);
    }
};

template <typename T, typename P> __device__ __forceinline__ T* pick(P* const (&p)[3], int g) {
    return reinterpret_cast<T*>(g == 0 ? p[0] : g == 1 ? p[1] : p[2]);
}

// What becomes of four results before they are rounded to the output's type.  The parameters are read once, ahead of the
// stores: read with each store they cost 10 us of a launch.
enum Finish { kPlain, kRelu, kPositive };
template <Finish F, typename TC>
__device__ __forceinline__ void finish4(TC* c, const float* positive, float alpha, f32x4 v) {
    v *= alpha;
    if constexpr (F == kRelu) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] < 0.f ? 0.f : v[e];       // (NaN stays)
    }
    if constexpr (F == kPositive) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(positive);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = x[e] <= 0.f ? 0.f : v[e];
    }
    typedef TC tc4 __attribute__((ext_vector_type(4)));
    *reinterpret_cast<tc4*>(c) = __builtin_convertvector(v, tc4);
}
// f(finish kind, type of c) for the call's kind and type
template <typename Fn> __device__ __forceinline__ void with_finish(const GemmParams& p, Fn f) {
    using std::integral_constant;
    auto typed = [&](auto kind) {
        if (p.c_dtype == T5A_F32) f(kind, float{});
        else if (p.c_dtype == T5A_BF16) f(kind, __bf16{});
        else f(kind, _Float16{});
    };
    if (p.positive != nullptr) typed(integral_constant<Finish, kPositive>{});
    else if (p.relu) typed(integral_constant<Finish, kRelu>{});
    else typed(integral_constant<Finish, kPlain>{});
}

// A workgroup of 2 x 2 wavefronts forms BM x 64 results in steps of 32 of the contraction: the step's products on one LDS
// buffer while the next step's values, fetched DEPTH steps ahead into registers, are split into the other.  With tens of steps
// per workgroup the latency of a step counts as much as its products: one barrier per step, and more steps ahead for the smaller
// tile.  4500 x 2048 x 512: 67 us = 141 TFLOP/s in fp32 terms, 845 on the bf16 matrix cores (before the operands were scaled 65, with
// a single buffer and two barriers 71; the fp32 library product 87); 1000 x 512 x 2048 25 us in four splits.
template <typename TA, typename TB, bool ACOL, bool BCOL, int BM>
__global__ __launch_bounds__(kThreads, BM == 128 ? 2 : 3) void gemm_kernel(const GemmParams p) {
    constexpr int BN = 64, DEPTH = BM == 128 ? 2 : 4;
    using OA = Operand<TA, ACOL, BM>;
    using OB = Operand<TB, BCOL, BN>;
    constexpr int MI = BM / 64, NI = BN / 64;        // 32 x 32 blocks per wavefront; wavefronts are 2 x 2
    constexpr int BUF = OA::NP * OA::PLANE + OB::NP * OB::PLANE;
    __shared__ __attribute__((aligned(16))) __bf16 tiles[2 * BUF];
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, hh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = (wave & 1) * (BM / 2), wn = (wave >> 1) * (BN / 2);

    // each XCD takes a contiguous piece of the list (split, group, row tile, column tile), whose rows its L2 then holds
    const int id = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (id >= p.items) return;
    int rest = id;
    const int tn = rest % p.tiles_n; rest /= p.tiles_n;
    const int tm = rest % p.tiles_m; rest /= p.tiles_m;
    const int go = rest % p.groups_out, split = rest / p.groups_out;
    const int m0 = tm * BM, n0 = tn * BN;
    // steps of this split: [it0, it_end) of the groups_k concatenated contractions
    const int it0 = split * p.steps_split, it_end = min(it0 + p.steps_split, p.groups_k * p.steps);

    f32x16 acc[NI][MI];
    auto each = [&](auto f) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < MI; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = f(acc[i][j][r]);
    };
    each([](float) { return 0.f; });

    // the steps of one group at a time
    for (int it = it0; it < it_end;) {
        const int g = it / p.steps, kk = it - g * p.steps, n = min(p.steps - kk, it_end - it);
        OA oa; OB ob;
        oa.start(pick<const TA>(p.a, go + g), p.lda, m0, p.M, p.K, tid);
        ob.start(pick<const TB>(p.b, go + g), p.ldb, n0, p.N, p.K, tid);
        typename OA::Tile xa[DEPTH];
        typename OB::Tile xb[DEPTH];
        // (steps past the last one, here or of the contraction, are fetched and not used)
        int at = kk;
        auto fetch = [&](typename OA::Tile& a, typename OB::Tile& b) { oa.fetch(a, at, p.K); ob.fetch(b, at, p.K); ++at; };
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) fetch(xa[d], xb[d]);
        __syncthreads();       // (the group before is done with the buffers)
        OA::store(xa[0], tiles, tid);
        OB::store(xb[0], tiles + OA::NP * OA::PLANE, tid);
        fetch(xa[0], xb[0]);
        for (int t0 = 0; t0 < n; t0 += DEPTH) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
                if (t0 + d >= n) break;
                const int next = (d + 1) % DEPTH;
                __bf16* const cur = tiles + (d & 1) * BUF;
                __bf16* const nxt = tiles + ((d + 1) & 1) * BUF;
                __syncthreads();
                bf16x8 fa[2][MI][OA::NP], fb[2][NI][OB::NP];
                auto frags = [&](int s) {
#pragma unroll
                    for (int j = 0; j < MI; ++j) OA::frag(cur, wm + 32 * j, s, lane, fa[s][j]);
#pragma unroll
                    for (int i = 0; i < NI; ++i) OB::frag(cur + OA::NP * OA::PLANE, wn + 32 * i, s, lane, fb[s][i]);
                };
                auto products = [&](int s) {
                    using H = Half16<__bf16>;
                    // smallest products first; a product of every block in turn
#pragma unroll
                    for (int q = 2; q >= 0; --q)
#pragma unroll
                        for (int qa = 0; qa < OA::NP; ++qa) {
                            const int qb = q - qa;
                            if (qb < 0 || qb >= OB::NP) continue;
#pragma unroll
                            for (int i = 0; i < NI; ++i)
#pragma unroll
                                for (int j = 0; j < MI; ++j) acc[i][j] = H::mfma(fb[s][i][qb], fa[s][j][qa], acc[i][j]);
                        }
                };
                frags(0);
                frags(1);
                products(0);
                OA::store(xa[next], nxt, tid);
                OB::store(xb[next], nxt + OA::NP * OA::PLANE, tid);
                fetch(xa[next], xb[next]);
                products(1);
            }
        }
        if (p.groups_k > 1 && g == 0) each([&](float x) { return x * p.alpha; });     // (the factor is the first group's)
        it += n;
    }

    // A sum that is not finite (split_device.h): the products again on the fp32 matrix cores, straight from memory.
    float odd = 0.f;                     // NaN if any is not finite
    each([&](float x) { odd += x * 0.f; return x; });
    if (__any(odd != odd)) {
        each([](float) { return 0.f; });
        for (int it = it0; it < it_end; ++it) {
            const int g = it / p.steps, kk = it - g * p.steps;
            const TA* const a = pick<const TA>(p.a, go + g);
            const TB* const b = pick<const TB>(p.b, go + g);
            for (int s2 = 0; s2 < BK / 2; ++s2) {
                const int k = kk * BK + 2 * s2 + hh;
                float fa[MI], fb[NI];
#pragma unroll
                for (int j = 0; j < MI; ++j) fa[j] = OA::value(a, p.lda, m0 + wm + 32 * j + lr, p.M, k, p.K);
#pragma unroll
                for (int i = 0; i < NI; ++i) fb[i] = OB::value(b, p.ldb, n0 + wn + 32 * i + lr, p.N, k, p.K);
#pragma unroll
                for (int i = 0; i < NI; ++i)
#pragma unroll
                    for (int j = 0; j < MI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[i], fa[j], acc[i][j], 0, 0, 0);
            }
            if (p.groups_k > 1 && g == 0 && (kk + 1 == p.steps || it + 1 == it_end)) each([&](float x) { return x * p.alpha; });
        }
    } else {
        constexpr float back = (OA::NP == 3 ? kSplitBack : 1.f) * (OB::NP == 3 ? kSplitBack : 1.f);
        each([](float x) { return x * back; });
    }

    // lane (lr, hh): row lr of the block, columns 8 (r >> 2) + 4 hh + (r & 3)
    auto quads = [&](auto put) {
#pragma unroll
        for (int j = 0; j < MI; ++j) {
            const int m = m0 + wm + 32 * j + lr;
            if (m >= p.M) continue;
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int n = n0 + wn + 32 * i + 8 * q + 4 * hh;
                    if (n < p.N) put(m, n, f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]});
                }
        }
    };
    if (p.nsplit > 1) {
        float* const part = p.part + ((int64_t)split * p.groups_out + go) * p.M * p.N;
        quads([&](int m, int n, f32x4 v) { *reinterpret_cast<f32x4*>(part + (int64_t)m * p.N + n) = v; });
    } else {
        const float alpha = go == 0 && p.groups_k == 1 ? p.alpha : 1.f;
        with_finish(p, [&](auto kind, auto zero) {
            using TC = decltype(zero);
            TC* const c = pick<TC>(p.c, go);
            quads([&](int m, int n, f32x4 v) {
                finish4<decltype(kind)::value, TC>(c + (int64_t)m * p.ldc + n, p.positive + (int64_t)m * p.ldpos + n, alpha, v);
            });
        });
    }
}

// the splits' sums, in their order
__global__ __launch_bounds__(kThreads) void gemm_reduce_kernel(const GemmParams p) {
    const int64_t quads = (int64_t)p.groups_out * p.M * p.N / 4;
    const f32x4* const part = reinterpret_cast<const f32x4*>(p.part);
    const unsigned nq = p.N / 4;
    with_finish(p, [&](auto kind, auto zero) {
        using TC = decltype(zero);
        for (int64_t x = (int64_t)blockIdx.x * kThreads + threadIdx.x; x < quads; x += (int64_t)gridDim.x * kThreads) {
            f32x4 v = part[x];
            for (int s = 1; s < p.nsplit; ++s) v += part[x + s * quads];
            const int64_t row = x / nq;
            const int group = (int)(row / p.M), m = (int)(row - (int64_t)group * p.M), n = (int)(x - row * nq) * 4;
            finish4<decltype(kind)::value, TC>(pick<TC>(p.c, group) + (int64_t)m * p.ldc + n, p.positive + (int64_t)m * p.ldpos + n,
                                               group == 0 && p.groups_k == 1 ? p.alpha : 1.f, v);
        }
    });
}

struct Shape { int bm, nsplit; };      // rows of a tile (of 64 columns), splits of the contraction

// A tile of 128 x 64 reads its operands less often, one of 64 x 64 fills the chip with fewer rows, and so does a contraction in
// several splits, at the price of a second kernel that adds them.  The estimate in us: a step of a tile takes `alone` on a
// compute unit of its own, `busy` where several workgroups share one (two of 128 x 64, three of 64 x 64 fit into its LDS), the
// rest are one workgroup's start and the second kernel.  Fitted to both tiles with 1 to 24 splits over products of 300 to 8192
// rows by 512 / 2048 and 768 / 3072 (84 products, root mean square error 9 %); its choice is 1.3 % off the best on average.
// 4500 rows, us (128 x 64 / 64 x 64): 512 -> 2048 64 / 68; 2048 -> 512 85 / 76 in one split, 73 / 75 in four; gradient of a
// 2048 x 512 weight 73 / 74 in two splits, 67 / 75 in four, 72 / 82 in eight; 1000 rows 512 -> 512 12.8 in 64 x 64, 14.9 in 128 x 64.
Shape gemm_shape(const GemmParams& p, bool sixfold) {
    constexpr int kComputeUnits = 256;
    const double product = sixfold ? 1.0 : 0.56;       // (with a bf16 operand: three matrix products for six)
    const int64_t steps = (int64_t)((p.K + BK - 1) / BK) * p.groups_k;
    const double mb = 4e-6 * p.groups_out * p.M * (double)p.N;
    Shape best = {64, 1};
    double least = 0.;
    for (int bm = 64; bm <= 128; bm += 64) {
        const int slots = bm == 128 ? 2 : 3;
        const double alone = bm == 128 ? 0.73 : 0.44, busy = bm == 128 ? 0.63 : 0.39;
        const int64_t tiles = (int64_t)((p.M + bm - 1) / bm) * ((p.N + 63) / 64) * p.groups_out;
        for (int s = 1; s <= 16 && s <= steps; ++s) {
            const int64_t each = (steps + s - 1) / s, on_unit = (tiles * s + kComputeUnits - 1) / kComputeUnits;
            const int64_t rounds = (on_unit + slots - 1) / slots;
            const double step = rounds * alone > on_unit * busy ? rounds * alone : on_unit * busy;
            const double us = each * product * step + 1.3 * rounds + (s > 1 ? 4.5 + (s + 1) * mb / 4.8 : 0.);
            if (least == 0. || us < least) { least = us; best = {bm, s}; }
        }
    }
    return best;
}

template <typename TA, typename TB, bool ACOL, bool BCOL>
hipError_t launch(GemmParams p, const Shape& t, hipStream_t stream) {
    p.tiles_m = (p.M + t.bm - 1) / t.bm;
    p.tiles_n = (p.N + 63) / 64;
    p.steps = (p.K + BK - 1) / BK;
    p.nsplit = t.nsplit;
    p.steps_split = (p.steps * p.groups_k + t.nsplit - 1) / t.nsplit;
    const int64_t items = (int64_t)p.tiles_m * p.tiles_n * p.groups_out * t.nsplit;
    if (items > 0x7ffffff0) return hipErrorInvalidConfiguration;
    p.items = (int)items;
    const dim3 grid((unsigned)((items + 7) / 8 * 8));
    if (t.bm == 128) hipLaunchKernelGGL((gemm_kernel<TA, TB, ACOL, BCOL, 128>), grid, dim3(kThreads), 0, stream, p);
    else hipLaunchKernelGGL((gemm_kernel<TA, TB, ACOL, BCOL, 64>), grid, dim3(kThreads), 0, stream, p);
    if (t.nsplit > 1) {
        const int64_t blocks = ((int64_t)p.groups_out * p.M * p.N / 4 + kThreads - 1) / kThreads;
        hipLaunchKernelGGL(gemm_reduce_kernel, dim3((unsigned)(blocks < 2048 ? blocks : 2048)), dim3(kThreads), 0, stream, p);
    }
    return hipGetLastError();
}

}  // namespace

static Shape shape_of(const GemmParams& p, int a_dtype, int b_dtype) { return gemm_shape(p, a_dtype != T5A_BF16 && b_dtype != T5A_BF16); }

int64_t gemm_f32_workspace_bytes(const GemmParams& p, int a_dtype, int b_dtype) {
    const Shape t = shape_of(p, a_dtype, b_dtype);
    return t.nsplit > 1 ? (int64_t)t.nsplit * p.groups_out * p.M * p.N * (int64_t)sizeof(float) : 0;
}

hipError_t launch_gemm_f32(const GemmParams& p, int a_dtype, int b_dtype, bool a_trans, bool b_trans, hipStream_t stream) {
    const Shape t = shape_of(p, a_dtype, b_dtype);
    const bool ab = a_dtype == T5A_BF16, bb = b_dtype == T5A_BF16;
    if (!a_trans && !b_trans && !bb) return ab ? launch<__bf16, float, false, false>(p, t, stream) : launch<float, float, false, false>(p, t, stream);
    if (!a_trans && b_trans && !bb) return ab ? launch<__bf16, float, false, true>(p, t, stream) : launch<float, float, false, true>(p, t, stream);
    if (a_trans && b_trans && !(ab && bb))
        return ab ? launch<__bf16, float, true, true>(p, t, stream) : bb ? launch<float, __bf16, true, true>(p, t, stream) : launch<float, float, true, true>(p, t, stream);
    return hipErrorInvalidValue;
}

}  // namespace t5a
