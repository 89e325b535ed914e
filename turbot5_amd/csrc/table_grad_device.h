// The bias table's gradient in a backward pass over query rows: dS summed per distance, distances summed per bucket.
//
// A wavefront keeps sums of its own for the distances below saturation in LDS and in two registers for the rest; the
// wavefronts' sums meet once, at the end.  A workgroup's buckets then go to a slot of the workspace, and the pass over the keys, which
// follows in the stream, adds the slots of a head in a fixed order.  Atomics, on LDS per distance and on the table per bucket and
// workgroup, are what this avoids; all workgroups of a head met at the same 32 addresses.  us, the backward's kernels with
// atomics / now, bf16 D64: B16 H12 L1024 244 / 234, the same causal 170 / 164, B3 H12 L1500 causal 90 / 81, B4 H8 L512 39 / 34, B8 H8
// L512 causal 43 / 35.  (One LDS atomic per score, no skewed block: 434 at B16 H12 L1024.)
#pragma once
#include "lut_device.h"
#include "mfma16_device.h"

namespace t5a {

// floats of a wavefront's sums, index distance + sat
__host__ __device__ inline int table_grad_floats(int sat) { return (2 * sat + 4) & ~3; }

// Adds a block of dS: lane (lr, hh) holds, for query lr, the keys 8 (r >> 2) + 4 hh + (r & 3); `rel` is the distance of key 0 and
// query 0.  The block goes to LDS skewed, the pair of key kk and query lr at row lr, column kk - lr + R - 1, so that a column
// holds one distance, R queries at a time; a lane then sums a column.  What lies outside the skewed band is zero and never written.
// 16 words written and 32 / R times R read per lane at constant offsets, without bank conflicts.
template <int R>
__device__ __forceinline__ void table_grad_block(float* skew, float* sums, const f32x16& ds, int lane, int rel, int sat, float& lo, float& hi) {
    const int lr = lane & 31, hh = lane >> 5;
#pragma unroll
    for (int round = 0; round < 32 / R; ++round) {
        if (R == 32 || lr / R == round) {
            float* w = skew + (lr % R) * 63 + (R - 1) + 4 * hh;
#pragma unroll
            for (int r = 0; r < 16; ++r) w[8 * (r >> 2) + (r & 3)] = ds[r];
        }
        asm volatile("" ::: "memory");     // (LDS accesses of a wavefront keep their order)
        const int x = rel - R * round + lane - (R - 1);
        const bool inside = lane < 31 + R && x > -sat && x < sat;
        float* const at = sums + x + sat;
        float c0 = 0.f, c1 = 0.f, c2 = 0.f, c3 = 0.f;
        if (inside) c3 = *at;
#pragma unroll
        for (int q = 0; q < R; q += 4) {
            c0 += skew[q * 64 + lane]; c1 += skew[(q + 1) * 64 + lane];
            c2 += skew[(q + 2) * 64 + lane]; c3 += skew[(q + 3) * 64 + lane];
        }
        asm volatile("" ::: "memory");
        const float c = (c0 + c1) + (c2 + c3);
        if (inside) *at = c;
        else if (lane < 31 + R) { if (x < 0) lo += c; else hi += c; }
    }
}

// All threads: the wavefronts' sums into the workgroup's slot, or without slots into the head's column of the table's gradient.
// `scratch`: 2 WAVES floats; `unit`: what the sums are multiplied by.  Eight lanes share a bucket, whose distances are one run on one side of the diagonal.
template <int WAVES>
__device__ __forceinline__ void table_grad_finish(const BwdParams& p, int h, int64_t slot, const float* sums, float* scratch, int sat, float lo, float hi, float unit = 1.f) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, stride = table_grad_floats(sat);
    const BucketSpec& bs = p.bs;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        lo += __shfl_xor(lo, off, 64);
        hi += __shfl_xor(hi, off, 64);
    }
    __syncthreads();       // (the scratch may lie in memory that was still in use)
    if (lane == 0) { scratch[2 * wave] = lo; scratch[2 * wave + 1] = hi; }
    __syncthreads();
    const int last_lo = bucket_of(bs, -sat), last_hi = bucket_of(bs, sat);
    const int sub = tid & 7;
    for (int b0 = 0; b0 < p.n_buckets; b0 += 8 * WAVES) {      // (uniform: the exchange below needs every lane)
        const int b = b0 + (tid >> 3);
        const bool up = bs.bidirectional && b >= bs.nb;
        const int k = up ? b - bs.nb : b, t = k - bs.max_exact;
        float s = 0.f;
        if (b < p.n_buckets && k < bs.nb) {
            const int from = t <= 0 ? k : bs.thr[t - 1];
            const int to = min(t < 0 ? k + 1 : t < bs.n_thr ? bs.thr[t] : sat, sat);
            for (int d = from + sub; d < to; d += 8)
                if (!up || d > 0) {
                    const float* at = sums + (up ? d : -d) + sat;
#pragma unroll
                    for (int w = 0; w < WAVES; ++w) s += at[w * stride];
                }
        }
#pragma unroll
        for (int off = 1; off < 8; off <<= 1) s += __shfl_xor(s, off, 64);
        if (sub == 0 && b < p.n_buckets) {
#pragma unroll
            for (int w = 0; w < WAVES; ++w) {
                if (b == last_lo) s += scratch[2 * w];
                if (b == last_hi) s += scratch[2 * w + 1];
            }
            s *= unit;
            if (p.slots != nullptr) p.slots[slot * p.n_buckets + b] = s;
            else if (s != 0.f) atomicAdd(&p.dtable[(int64_t)b * p.H + h], s);
        }
    }
}

// A workgroup without rows: its slot is zero.
template <int WAVES>
__device__ __forceinline__ void table_grad_none(const BwdParams& p, int64_t slot) {
    if (p.slots == nullptr || p.table == nullptr || p.dtable == nullptr) return;
    for (int b = threadIdx.x; b < p.n_buckets; b += 64 * WAVES) p.slots[slot * p.n_buckets + b] = 0.f;
}

// All threads of one workgroup of the pass over the keys: the slots of a head, into its column of the table's gradient.
// `scratch`: 64 WAVES floats, free on return.
template <int WAVES>
__device__ __forceinline__ void table_grad_reduce(const BwdParams& p, int h, float* scratch) {
    const int tid = threadIdx.x, shift = p.n_buckets <= 32 ? 5 : 6, b = tid & ((1 << shift) - 1), parts = 64 * WAVES >> shift;
    const float* const from = p.slots + (int64_t)h * p.slots_per_head * p.n_buckets + b;
    float s = 0.f;
    if (b < p.n_buckets) {
#pragma unroll 8
        for (int x = tid >> shift; x < p.slots_per_head; x += parts) s += from[(int64_t)x * p.n_buckets];
    }
    scratch[tid] = s;
    __syncthreads();
    if (tid < p.n_buckets) {
        for (int x = 1; x < parts; ++x) s += scratch[tid + (x << shift)];
        p.dtable[(int64_t)tid * p.H + h] = s;
    }
    __syncthreads();
}

}  // namespace t5a
