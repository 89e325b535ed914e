// Device helpers of the kernels built from 32 x 32 blocks of scores on the 16-bit matrix cores (attn_bwd.hip,
// attn_window.hip): operand types, tile swizzle, LDS-DMA requests, workgroup placement.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "lut_device.h"

namespace t5a {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

template <typename T> struct Half16;
template <> struct Half16<__bf16> {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    static __device__ __forceinline__ f32x16 mfma(v8 a, v8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
    typedef __bf16 v2 __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ float pair_sum(v2 x, float acc) {      // acc + x[0] + x[1]
        return __builtin_amdgcn_fdot2_f32_bf16(x, v2{(__bf16)1.0f, (__bf16)1.0f}, acc, false);
    }
};
template <> struct Half16<_Float16> {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    static __device__ __forceinline__ f32x16 mfma(v8 a, v8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
    typedef _Float16 v2 __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ float pair_sum(v2 x, float acc) {
        return __builtin_amdgcn_fdot2(x, v2{(_Float16)1.0f, (_Float16)1.0f}, acc, false);
    }
};

// chunk swizzle of a tile row: 16 consecutive rows put a chunk into 16 different 16-byte slots of a 256-byte bank
// line (row reads), and rows 2, 3 (mod 4) swap their 64-byte halves (the transposing read touches four consecutive
// rows x 64 bytes at a time)
__device__ __forceinline__ int tile_swz(int row) { return ((row >> 1) & 7) ^ (((row >> 1) & 1) << 2); }

// LDS-DMA: a wavefront instruction fetches 64 x 16 bytes at per-lane byte offsets of a buffer (zeros past its end) and
// writes them to 1 KB of consecutive LDS addresses in lane order, without passing through registers.  Issued from
// assembly, so the wait for it (vmcnt) is the kernel's own.
__device__ __forceinline__ u32x4 dma_rsrc(const void* base, unsigned bytes) {
    const unsigned long long a = reinterpret_cast<unsigned long long>(base);
    return u32x4{(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)a),
                 (unsigned)__builtin_amdgcn_readfirstlane((int)((unsigned)(a >> 32) & 0xffffu)),
                 (unsigned)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}
__device__ __forceinline__ void dma_16(u32x4 rs, unsigned lds_addr, int voffset) {
    const u32x4 rsrc = {(unsigned)__builtin_amdgcn_readfirstlane((int)rs[0]), (unsigned)__builtin_amdgcn_readfirstlane((int)rs[1]),
                        (unsigned)__builtin_amdgcn_readfirstlane((int)rs[2]), (unsigned)__builtin_amdgcn_readfirstlane((int)rs[3])};
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :: "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voffset), "s"(rsrc) : "memory", "m0");
}
// the same with 4 bytes per lane (256 consecutive bytes of LDS)
__device__ __forceinline__ void dma_4(u32x4 rs, unsigned lds_addr, int voffset) {
    const u32x4 rsrc = {(unsigned)__builtin_amdgcn_readfirstlane((int)rs[0]), (unsigned)__builtin_amdgcn_readfirstlane((int)rs[1]),
                        (unsigned)__builtin_amdgcn_readfirstlane((int)rs[2]), (unsigned)__builtin_amdgcn_readfirstlane((int)rs[3])};
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds"
                 :: "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voffset), "s"(rsrc) : "memory", "m0");
}
// waits until at most N of this wavefront's memory requests are outstanding (they complete in order)
template <int N> __device__ __forceinline__ void wait_vmcnt() {
    static_assert(N < 64, "");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// rows 16 u .. + 15 of a 32-row accumulator as a B operand
template <typename v8> __device__ __forceinline__ v8 to_frag(const f32x16& x, int u) {
    f32x8 y;
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = x[8 * u + e];
    return __builtin_convertvector(y, v8);
}

// Workgroup -> (own block, head, sequence).  Workgroups go to the eight XCDs in turn; all own blocks of a (head,
// sequence) pair go to one XCD, whose L2 then holds the pair's rows of the other kind for all of them.  Where the
// pairs do not divide by eight they are dealt out in turn instead.  With a causal mask the own blocks differ in length
// (a query block sees the keys up to its own end, a key block the queries from its own start on), and whatever is
// dispatched last should be short: the blocks are then the slowest index, longest first.
template <bool CAUSAL, bool KV>
__device__ __forceinline__ void bwd_place(int H, int B, int nblk, int& blk, int& h, int& b) {
    const int pairs = H * B, id = blockIdx.x;
    int pair, level;
    if ((pairs & 7) == 0) {
        const int pp = pairs >> 3, slot = id >> 3;
        if (CAUSAL) { level = slot / pp; pair = (id & 7) * pp + (slot - level * pp); }
        else { const int q = slot / nblk; level = slot - q * nblk; pair = (id & 7) * pp + q; }
    } else {
        level = id / pairs; pair = id - level * pairs;
    }
    blk = (CAUSAL && !KV) ? nblk - 1 - level : level;
    h = pair / B; b = pair - h * B;
}

// The bias of one head by distance, times log2(e).  With up to 64 buckets lane b of every wavefront holds bucket b: one
// load, and a look-up is an exchange between lanes instead of a round trip to memory.  `at` is for all lanes at once.
struct BiasColumn {
    const BucketSpec& bs;
    const void* table; int dtype; int64_t first, step;
    bool in_lanes;
    float mine;
    template <typename P> __device__ __forceinline__ BiasColumn(const P& p, int h, int lane)
        : bs(p.bs), table(p.table), dtype(p.table_dtype), first((int64_t)h * p.t_shead), step(p.t_sbucket), mine(0.f) {
        const int n = p.bs.bidirectional ? 2 * p.bs.nb : p.bs.nb;
        in_lanes = n <= 64;
        if (table != nullptr && in_lanes && lane < n) mine = load_table(table, dtype, first + lane * step) * 1.4426950408889634f;
    }
    __device__ __forceinline__ float at(int rel) const {
        if (table == nullptr) return 0.f;
        const int b = bucket_of(bs, rel);
        if (in_lanes) return __int_as_float(__builtin_amdgcn_ds_bpermute(b << 2, __float_as_int(mine)));
        return load_table(table, dtype, first + b * step) * 1.4426950408889634f;
    }
};

}  // namespace t5a
