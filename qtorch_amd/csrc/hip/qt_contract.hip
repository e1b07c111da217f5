// Pairwise contraction kernels of libqtorch_hip.so (gfx950).
//
// C[c] = sum_s A[a(c,s)] * B[b(c,s)] (Network::ContractIndices, reference
// src/Network.h:876-971), on the bit-level description qt::BitMap.  Three regimes:
//
//   k_direct        : one lane per output element, the summed index in the inner
//                     loop in the reference's order (last pair fastest).  In the
//                     plain complex128 form floating-point contraction is off, so
//                     results are bit-identical to the reference's loop.  Covers
//                     every shape; chosen for small summed extents (memory-bound).
//   k_skinny        : at most 5 free bits on one side of C: one lane per element of
//                     the large side holds all outputs of the small side, summed in
//                     k_direct's order (bit-identical to it); the large operand is
//                     read once instead of once per small-side output.
//   k_reduce_*      : small outputs with a large summed extent (e.g. a scalar from
//                     two big tensors): the summed index is split over workgroups,
//                     wavefront/LDS reductions, then an ordered second pass.
//   k_permute +     : large GEMM-shaped steps: operands are rewritten by the
//   k_gemm_c128       LDS-staged bit-permute kernel into A'[s][m], B'[s][n], then a
//                     complex FP64 GEMM on MFMA (v_mfma_f64_16x16x4f64) writes
//                     C[m + M n], which is already the reference's C layout
//                     (A's free axes low, B's high: src/Network.h:739-769).
#include <algorithm>
#include <cmath>
#include <cstring>

#include "qt_internal.h"
#include "qt_mac.h"

namespace qt {

namespace {

// Eight bit positions of a BitMap array at a time: one scalar load, where a loop over the
// bytes is a chain of vector loads (the plan is a kernel argument).
__device__ __forceinline__ uint64_t eight_positions(const uint8_t* pos, int w) {
    return reinterpret_cast<const uint64_t*>(pos)[w];
}

// offsets of the summed bits of s in A and B
__device__ __forceinline__ void s_offsets(const BitMap& m, int64_t s, int64_t& ga, int64_t& gb) {
    ga = 0;
    gb = 0;
    for (int w = 0; 8 * w < m.nbits_s; ++w) {
        const uint64_t pa = eight_positions(m.s_a, w), pb = eight_positions(m.s_b, w);
#pragma unroll
        for (int b = 0; b < 8; ++b)
            if (8 * w + b < m.nbits_s && ((s >> (8 * w + b)) & 1)) {
                ga += int64_t(1) << ((pa >> (8 * b)) & 0xff);
                gb += int64_t(1) << ((pb >> (8 * b)) & 0xff);
            }
    }
}

// offsets in A and B of the output bits lo to hi - 1 of c
__device__ __forceinline__ void c_offsets(const BitMap& m, int64_t c, int lo, int hi, int64_t& oa,
                                          int64_t& ob) {
    oa = 0;
    ob = 0;
    for (int w = lo >> 3; 8 * w < hi; ++w) {
        const uint64_t p = eight_positions(m.c_src, w);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const int i = 8 * w + b;
            if (i >= lo && i < hi && ((c >> i) & 1)) {
                const int src = int((p >> (8 * b)) & 0xff);
                if (src < 64) oa += int64_t(1) << src;
                else ob += int64_t(1) << (src - 64);
            }
        }
    }
}

// The n summed terms of one output in order (n a power of two), 8 operand pairs in flight.
// ga, gb: the terms' operand offsets (LDS).
template <class V, int MODE>
__device__ __forceinline__ void sum_terms(Acc<V, MODE>& acc, const V* __restrict__ A, const V* __restrict__ B,
                                          const int64_t* ga, const int64_t* gb, int n) {
    constexpr int U = 8;
    int j = 0;
    for (; j + U <= n; j += U) {
        V x[U], y[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            x[u] = A[ga[j + u]];
            y[u] = B[gb[j + u]];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) mac<V, MODE>(acc, x[u], y[u]);
    }
    if (n == 4) {
        V x[4], y[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            x[u] = A[ga[u]];
            y[u] = B[gb[u]];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) mac<V, MODE>(acc, x[u], y[u]);
        return;
    }
    for (; j < n; ++j) mac<V, MODE>(acc, A[ga[j]], B[gb[j]]);
}

// Most of a network's steps: a few thousand outputs over 4 to 64 terms, which a launch and
// the latency of the operand reads bound.  1,024 complex128 outputs over 16
// terms: 5.15 us, 5.63 with one term at a time and the plan read byte by byte; the 680
// steps of a 12-vertex energy 2.99 us on average, 3.41 before.
template <class V, int MODE>
__global__ __launch_bounds__(kThreads) void k_direct(const V* __restrict__ A, const V* __restrict__ B,
                                                     V* __restrict__ C, BitMap m, int64_t nC) {
    __shared__ int64_t low_a[kThreads], low_b[kThreads];
    __shared__ int64_t ga[kThreads], gb[kThreads];
    const int tid = threadIdx.x;
    const int lo = m.nbits_c < 8 ? m.nbits_c : 8;
    {
        int64_t oa, ob;
        c_offsets(m, tid, 0, lo, oa, ob);
        low_a[tid] = oa;
        low_b[tid] = ob;
    }
    const int64_t nS = int64_t(1) << m.nbits_s;
    const bool one_chunk = nS <= kThreads;
    if (one_chunk) {
        if (tid < nS) {
            int64_t a, b;
            s_offsets(m, tid, a, b);
            ga[tid] = a;
            gb[tid] = b;
        }
    }
    __syncthreads();
    const int64_t stride = int64_t(gridDim.x) * kThreads;
    for (int64_t base = int64_t(blockIdx.x) * kThreads; base < nC; base += stride) {
        int64_t ha, hb;
        c_offsets(m, base, lo, m.nbits_c, ha, hb);  // uniform across the workgroup
        const int64_t c = base + tid;
        const int64_t oa = ha + low_a[tid], ob = hb + low_b[tid];
        Acc<V, MODE> acc;
        if (one_chunk) {
            if (c < nC) sum_terms<V, MODE>(acc, A + oa, B + ob, ga, gb, int(nS));
        } else {
            for (int64_t s0 = 0; s0 < nS; s0 += kThreads) {
                __syncthreads();
                {
                    int64_t a, b;
                    s_offsets(m, s0 + tid, a, b);
                    ga[tid] = a;
                    gb[tid] = b;
                }
                __syncthreads();
                if (c < nC) sum_terms<V, MODE>(acc, A + oa, B + ob, ga, gb, kThreads);
            }
        }
        if (c < nC) C[c] = finish<V, MODE>(acc);
    }
}

// Steps with at most 5 free bits on one side of C (a gate, or a thin tensor, against a
// large tensor; C = [A's free bits low | B's free bits high]).  One lane per element
// of the large side's part of C holds all 2^NB outputs of the small side, so the large
// operand is read once (k_direct reads it once per small-side output); the small
// operand's elements for a chunk of summed indices are staged in LDS and read there
// by every lane at once.  Each output is summed in k_direct's order with the same
// arithmetic: bit-identical to k_direct.
// SMALL_B: B is the small side, output o of lane t is C[t + (o << lo_bits)];
// otherwise A is (lo_bits == NB), output o of lane t is C[o + (t << NB)].
template <class V, int MODE, int NB, bool SMALL_B>
__global__ __launch_bounds__(kThreads) void k_skinny(const V* __restrict__ A, const V* __restrict__ B,
                                                     V* __restrict__ C, BitMap m, int lo_bits, int64_t n_big) {
    constexpr int NO = 1 << NB;
    constexpr int SC = NB >= 5 ? 32 : 64;  // summed indices per staged chunk (<= 16 KB complex128)
    constexpr int LU = sizeof(V) == 16 && NB >= 5 ? 4 : 8;  // loads in flight (registers: 175 at most)
    __shared__ int64_t g_big[SC];          // the large operand's offset of each summed index
    __shared__ V ys[SC][NO];               // the small operand's elements
    __shared__ int64_t small_off[NO];
    const int tid = threadIdx.x;
    if (tid < NO) {
        int64_t oa, ob;
        if constexpr (SMALL_B) {
            c_offsets(m, int64_t(tid) << lo_bits, lo_bits, m.nbits_c, oa, ob);
            small_off[tid] = ob;
        } else {
            c_offsets(m, tid, 0, NB, oa, ob);
            small_off[tid] = oa;
        }
    }
    const int64_t nS = int64_t(1) << m.nbits_s;
    const int64_t stride = int64_t(gridDim.x) * kThreads;
    for (int64_t base = int64_t(blockIdx.x) * kThreads; base < n_big; base += stride) {
        const int64_t t = base + tid;
        int64_t big_off;
        {
            int64_t oa, ob;
            if constexpr (SMALL_B) {
                c_offsets(m, t, 0, lo_bits, oa, ob);
                big_off = oa;
            } else {
                c_offsets(m, t << NB, NB, m.nbits_c, oa, ob);
                big_off = ob;
            }
        }
        Acc<V, MODE> acc[NO];
        for (int64_t s0 = 0; s0 < nS; s0 += SC) {
            const int n_s = int(nS - s0 < SC ? nS - s0 : SC);
            __syncthreads();  // small_off is written; the previous chunk's reads are done
            for (int e = tid; e < n_s * NO; e += kThreads) {
                const int j = e / NO, o = e % NO;
                int64_t a, b;
                s_offsets(m, s0 + j, a, b);
                if (o == 0) g_big[j] = SMALL_B ? a : b;
                ys[j][o] = SMALL_B ? B[small_off[o] + b] : A[small_off[o] + a];
            }
            __syncthreads();
            if (t < n_big)
                // LU loads of the large operand in flight before their products (one at a
                // time left the kernel waiting on each load: 14-20 % slower on 28-bit
                // slices); the products keep j's order
                for (int j0 = 0; j0 < n_s; j0 += LU) {
                    V x[LU];
#pragma unroll
                    for (int u = 0; u < LU; ++u)
                        if (j0 + u < n_s) x[u] = SMALL_B ? A[big_off + g_big[j0 + u]] : B[big_off + g_big[j0 + u]];
#pragma unroll
                    for (int u = 0; u < LU; ++u)
                        if (j0 + u < n_s)
#pragma unroll
                            for (int o = 0; o < NO; ++o) {
                                if constexpr (SMALL_B) mac<V, MODE>(acc[o], x[u], ys[j0 + u][o]);
                                else mac<V, MODE>(acc[o], ys[j0 + u][o], x[u]);
                            }
                }
        }
        if (t < n_big)
#pragma unroll
            for (int o = 0; o < NO; ++o) {
                const int64_t idx = SMALL_B ? t + (int64_t(o) << lo_bits) : int64_t(o) + (t << NB);
                C[idx] = finish<V, MODE>(acc[o]);
            }
    }
}

// k_skinny's steps when the large side's free bits keep their order in C (a gate on
// a large tensor, as in a circuit sweep) and at most 4 bits are summed: lane t's
// element of the large operand X sits at t with zero bits inserted at X's summed
// positions (a few shifts instead of a walk over every bit of C), the small operand's
// elements are uniform (scalar loads from the kernel's arguments' offsets), and each
// lane issues its 2^NS loads of X before any arithmetic.  Same summation order and
// arithmetic as k_skinny: bit-identical to it.
struct ThinArgs {
    int64_t n_big;
    int32_t lo_bits;        // small B: output o of lane t is C[t + (o << lo_bits)]
    int32_t n_ins;          // X's summed positions, ascending
    int32_t ins_pos[4];
    int64_t g_big[16];      // X offset of summed index j (k_direct's digit order)
    int32_t g_small[16];    // small operand offset of summed index j
    int32_t small_off[16];  // small operand offset of its free part o
};

template <class V, int MODE, int NS, int NB, bool SMALL_B>
__global__ __launch_bounds__(kThreads) void k_thin(const V* __restrict__ X, const V* __restrict__ G,
                                                   V* __restrict__ C, ThinArgs r) {
    constexpr int NJ = 1 << NS, NO = 1 << NB;
    const int64_t stride = int64_t(gridDim.x) * kThreads;
    for (int64_t t = int64_t(blockIdx.x) * kThreads + threadIdx.x; t < r.n_big; t += stride) {
        int64_t x = t;
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const int p = r.ins_pos[i];
            x = ((x >> p) << (p + 1)) | (x & ((int64_t(1) << p) - 1));
        }
        V xs[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) xs[j] = X[x + r.g_big[j]];
        Acc<V, MODE> acc[NO];
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int o = 0; o < NO; ++o) {
                const V g = G[r.small_off[o] + r.g_small[j]];
                if constexpr (SMALL_B) mac<V, MODE>(acc[o], xs[j], g);
                else mac<V, MODE>(acc[o], g, xs[j]);
            }
#pragma unroll
        for (int o = 0; o < NO; ++o) {
            const int64_t idx = SMALL_B ? t + (int64_t(o) << r.lo_bits) : int64_t(o) + (t << NB);
            C[idx] = finish<V, MODE>(acc[o]);
        }
    }
}

// Long sums into few outputs (see reduce_shape): the summed index is split over lanes,
// steps and workgroups, the outputs over row groups.
constexpr int64_t kReduceMaxBlocks = int64_t(1) << 15;

template <class V>
__device__ __forceinline__ V shfl_xor_v(V v, int d) {
    V r;
    r.x = __shfl_xor(v.x, d, 64);
    r.y = __shfl_xor(v.y, d, 64);
    return r;
}

// Rows of an operand: its elements that share one value of its free bits.  A workgroup
// takes one group of GA rows of A and GB rows of B (blockIdx.y) and accumulates the
// GA x GB outputs they form, so an operand element is read once per group of the other
// side's rows.  The summed index s splits into the lane (bits 0-7), the workgroup (the
// next log2(gridDim.x) bits) and the step (the bits above).  The host orders the summed
// bits (order_summed_bits): the lanes of a wave cover the lowest summed bits of A and of
// B in turn, so that both operands are read in whole 64-byte pieces however their axes
// lie, and workgroups that run together read neighbouring runs.  Every output of a call is
// summed in the same fixed order: each lane over its steps in order, then the lanes of a
// wave pairwise (lane bits 5 to 0), the waves in order, the workgroups in order.  How many
// steps a workgroup takes depends on the number of row groups (run_reduce), so the order
// differs between shapes, and from the one-output-per-lane kernels'.
// Bound by HBM.  A step of two complex64 operands (2^25 and 2^24 elements, shuffled axes,
// 8 x 4 outputs, 2^22 summed indices: 403 MB), read-back included: 119 us, 586 us with
// the lanes on the pairs' own bit order and two passes of 4 x 4 outputs.
struct RowSet {
    int64_t oa[32], ob[32];        // offsets of a group's rows of A and of B
    int32_t c[32];                 // output offset of row pair (i, j) at c[i * GB + j]
    int32_t n_ga, n_gb;            // group bits of A and of B (the group index is A's low, B's high)
    int32_t ga_pos[24], ga_c[24];  // operand and output bit of each group bit of A
    int32_t gb_pos[24], gb_c[24];
};

template <class V, int MODE, int GA, int GB>
__global__ __launch_bounds__(kThreads) void k_reduce_rows(const V* __restrict__ A, const V* __restrict__ B,
                                                          V* __restrict__ partials, BitMap m, int step_bits,
                                                          RowSet r) {
    constexpr int Q = GA * GB;
    __shared__ V wsum[Q][kThreads / 64];
    // offsets of the step bits 0-5 and 6-11: plan bytes read inside the step loop
    // would be vector loads whose waits also wait for every operand load in flight
    __shared__ int64_t t_lo[2][64], t_hi[2][64];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int first_step_bit = m.nbits_s - step_bits;  // 8 + log2(gridDim.x)
    int64_t la = 0, lb = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j)
        if ((tid >> j) & 1) {
            la += int64_t(1) << m.s_a[j];
            lb += int64_t(1) << m.s_b[j];
        }
    if (tid < 128) {
        const int x = tid & 63, first = first_step_bit + (tid < 64 ? 0 : 6);
        int64_t oa = 0, ob = 0;
        for (int k = 0; k < 6; ++k)
            if (((x >> k) & 1) && first + k < m.nbits_s) {
                oa += int64_t(1) << m.s_a[first + k];
                ob += int64_t(1) << m.s_b[first + k];
            }
        if (tid < 64) {
            t_lo[0][x] = oa;
            t_lo[1][x] = ob;
        } else {
            t_hi[0][x] = oa;
            t_hi[1][x] = ob;
        }
    }
    int64_t base_a = la, base_b = lb;  // lane, workgroup and row-group bits
    for (int j = 8; j < first_step_bit; ++j)
        if ((blockIdx.x >> (j - 8)) & 1) {
            base_a += int64_t(1) << m.s_a[j];
            base_b += int64_t(1) << m.s_b[j];
        }
    int64_t c0 = 0;
    for (int i = 0; i < r.n_ga; ++i)
        if ((blockIdx.y >> i) & 1) {
            base_a += int64_t(1) << r.ga_pos[i];
            c0 += int64_t(1) << r.ga_c[i];
        }
    for (int i = 0; i < r.n_gb; ++i)
        if ((blockIdx.y >> (r.n_ga + i)) & 1) {
            base_b += int64_t(1) << r.gb_pos[i];
            c0 += int64_t(1) << r.gb_c[i];
        }
    __syncthreads();
    Acc<V, MODE> acc[GA][GB];
    // U steps per iteration, all loads issued before the first multiply.  Measured on
    // 2^24 summed indices: 0.19 ms; with the U loads of an iteration on neighbouring
    // runs instead of U steps apart, 0.60 ms
    constexpr int U0 = GA + GB >= 16 ? 1 : 16 / (GA + GB);
    constexpr int U = U0 >= 8 ? 8 : U0 >= 4 ? 4 : U0 >= 2 ? 2 : 1;
    const int steps = 1 << step_bits;
    for (int k0 = 0; k0 < steps; k0 += U) {
        V a[U][GA], b[U][GB];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u;
            if (u > 0 && k >= steps) break;  // fewer steps than U
            const int64_t ha = base_a + t_lo[0][k & 63] + t_hi[0][k >> 6];
            const int64_t hb = base_b + t_lo[1][k & 63] + t_hi[1][k >> 6];
#pragma unroll
            for (int i = 0; i < GA; ++i) a[u][i] = A[r.oa[i] + ha];
#pragma unroll
            for (int j = 0; j < GB; ++j) b[u][j] = B[r.ob[j] + hb];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u > 0 && k0 + u >= steps) break;
#pragma unroll
            for (int i = 0; i < GA; ++i)
#pragma unroll
                for (int j = 0; j < GB; ++j) mac<V, MODE>(acc[i][j], a[u][i], b[u][j]);
        }
    }
    // lanes pairwise at distances 32, 16, ..., 1.  While a lane holds more than one output
    // it keeps the half that its lane bit names and hands the other half over; after
    // log2(Q) distances it holds one output, whose index is its highest lane bits
    V v[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) v[q] = finish<V, MODE>(acc[q / GB][q % GB]);
    int q_own = 0;
#pragma unroll
    for (int l = 5; l >= 0; --l) {
        const int d = 1 << l, done = 1 << (5 - l);  // outputs per lane: Q / done
        if (Q / done > 1) {
            const int half = Q / done / 2;
            const bool up = (lane & d) != 0;
#pragma unroll
            for (int q = 0; q < half; ++q) {
                const V keep = up ? v[q + half] : v[q], give = up ? v[q] : v[q + half];
                const V got = shfl_xor_v(give, d);
                v[q].x = keep.x + got.x;
                v[q].y = keep.y + got.y;
            }
            if (up) q_own += half;
        } else {
            const V got = shfl_xor_v(v[0], d);
            v[0].x += got.x;
            v[0].y += got.y;
        }
    }
    if ((lane & (64 / Q - 1)) == 0) wsum[q_own][wave] = v[0];
    __syncthreads();
    if (tid < Q) {
        V t = wsum[tid][0];
        for (int w = 1; w < kThreads / 64; ++w) {
            t.x += wsum[tid][w].x;
            t.y += wsum[tid][w].y;
        }
        // one workgroup per output group: the result itself; else partials[c][workgroup]
        partials[(c0 + r.c[tid]) * gridDim.x + blockIdx.x] = t;
    }
}

template <class V>
__global__ __launch_bounds__(kThreads) void k_reduce_final(const V* __restrict__ partials, V* __restrict__ C,
                                                           int64_t nblocks) {
    // one workgroup per output: strided partial sums, then a fixed-shape tree (the
    // order does not depend on timing, so the result is reproducible)
    __shared__ V part[kThreads];
    const int64_t c = blockIdx.x;
    V t;
    t.x = 0;
    t.y = 0;
    for (int64_t b = threadIdx.x; b < nblocks; b += kThreads) {
        const V p = partials[c * nblocks + b];
        t.x += p.x;
        t.y += p.y;
    }
    part[threadIdx.x] = t;
    __syncthreads();
    for (int d = kThreads / 2; d >= 1; d >>= 1) {
        if (int(threadIdx.x) < d) {
            part[threadIdx.x].x += part[threadIdx.x + d].x;
            part[threadIdx.x].y += part[threadIdx.x + d].y;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) C[c] = part[0];
}

__device__ __forceinline__ uint16_t bf16_bits(float x) {  // round to nearest even
    return uint16_t(__float_as_uint(bf16_round(x)) >> 16);
}

// LDS-staged bit permutation (see PermPlan).  Reads walk the input-low bits
// contiguously, writes walk the output-low bits contiguously.
// Tile element t sits at slot t with its low 6 bits xor-ed with its row t / 64: a read
// that walks the tile 64 elements at a time (an input-low bit moved to an output-high
// position) hits a different bank with every lane, and the tile stays 2^tbits slots.
// P = 1 (complex64): each lane moves two elements that are neighbours on the read side
// (input bit 0) as one 16-byte load, and two that are neighbours on the write side
// (output bit 0) as one 16-byte store; 8-byte accesses measured well below the rate of
// 16-byte ones.
__device__ __forceinline__ int tile_slot(int t) { return t ^ ((t >> 6) & 63); }

// SPLIT (complex64, P = 1): out is four bf16 planes of 2^nbits elements (re hi, re lo, im hi,
// im lo; x = hi + lo, both rounded to nearest), a pair of neighbours one 4-byte store each.
template <class V, int P, bool SPLIT>
__global__ __launch_bounds__(kThreads) void k_permute(const V* __restrict__ in, V* __restrict__ out,
                                                      PermPlan p) {
    extern __shared__ unsigned char smem_raw[];
    V* tile = reinterpret_cast<V*>(smem_raw);
    const int64_t rb = int64_t(blockIdx.x) + int64_t(blockIdx.y) * gridDim.x;
    int64_t base_in = 0, base_out = 0;
    for (int i = 0; i < p.n_rest; ++i)
        if ((rb >> i) & 1) {
            base_in += int64_t(1) << p.rest_in[i];
            base_out += int64_t(1) << p.rest_out[i];
        }
    const int tbits = p.tl + p.n_extra_in;
    const int n = 1 << tbits;
    const int tid = threadIdx.x;
    // element e = (tid << P) + (q << (8 + P)): the offsets split into the thread's part
    // (tile bits P to P + 7, computed once) and the step's part (bits 8 + P and up,
    // uniform); with P = 1 bit 0 selects the pair's second element
    auto in_bit = [&](int b) -> int64_t { return b < p.tl ? int64_t(1) << b : int64_t(1) << p.extra_in_pos[b - p.tl]; };
    auto out_bit = [&](int b) -> int64_t { return b < p.tl ? int64_t(1) << b : int64_t(1) << p.extra_out_pos[b - p.tl]; };
    auto tile_bit = [&](int b) -> int { return b < p.tl ? p.lowout_tile[b] : p.extra_out_tile[b - p.tl]; };
    constexpr int hi = 8 + P;
    const int lo_bits = tbits < hi ? tbits : hi;
    int64_t in_t = base_in, out_t = base_out;
    int slot_t = 0;
    for (int b = P; b < lo_bits; ++b)
        if ((tid >> (b - P)) & 1) {
            in_t += in_bit(b);
            out_t += out_bit(b);
            slot_t |= 1 << tile_bit(b);
        }
    constexpr int per = kThreads << P;
    const int steps = n > per ? n / per : 1;
    // the step bits' offsets, read from the plan before the first data load: a plan
    // byte read inside the step loops is a vector load whose wait also waits for every
    // element load in flight
    constexpr int kStepBits = 4;  // tiles of at most 2^12 elements
    int64_t step_in[kStepBits], step_out[kStepBits];
    int step_tile[kStepBits];
#pragma unroll
    for (int k = 0; k < kStepBits; ++k) {
        const bool on = hi + k < tbits;
        step_in[k] = on ? in_bit(hi + k) : 0;
        step_out[k] = on ? out_bit(hi + k) : 0;
        step_tile[k] = on ? 1 << tile_bit(hi + k) : 0;
    }
    const int pair_bit = P == 1 ? 1 << tile_bit(0) : 0;
    if ((tid << P) < n) {
        for (int q = 0; q < steps; ++q) {
            int64_t off = in_t;
#pragma unroll
            for (int k = 0; k < kStepBits; ++k)
                if ((q >> k) & 1) off += step_in[k];
            const int t = (tid << P) + (q << hi);
            if constexpr (P == 1) {
                const float4 v = *reinterpret_cast<const float4*>(in + off);
                tile[tile_slot(t)] = make_float2(v.x, v.y);
                tile[tile_slot(t + 1)] = make_float2(v.z, v.w);
            } else {
                tile[tile_slot(t)] = in[off];
            }
        }
    }
    __syncthreads();
    if ((tid << P) < n) {
        for (int q = 0; q < steps; ++q) {
            int64_t off = out_t;
            int t = slot_t;
#pragma unroll
            for (int k = 0; k < kStepBits; ++k)
                if ((q >> k) & 1) {
                    off += step_out[k];
                    t |= step_tile[k];
                }
            if constexpr (P == 1) {
                const V a = tile[tile_slot(t)], b2 = tile[tile_slot(t | pair_bit)];
                if constexpr (SPLIT) {
                    uint32_t* const o = reinterpret_cast<uint32_t*>(out) + (off >> 1);
                    const int64_t plane = int64_t(1) << (p.nbits - 1);
                    auto two = [](float x, float y) { return uint32_t(bf16_bits(x)) | uint32_t(bf16_bits(y)) << 16; };
                    o[0] = two(a.x, b2.x);
                    o[plane] = two(a.x - bf16_round(a.x), b2.x - bf16_round(b2.x));
                    o[2 * plane] = two(a.y, b2.y);
                    o[3 * plane] = two(a.y - bf16_round(a.y), b2.y - bf16_round(b2.y));
                } else {
                    *reinterpret_cast<float4*>(out + off) = make_float4(a.x, a.y, b2.x, b2.y);
                }
            } else {
                out[off] = tile[tile_slot(t)];
            }
        }
    }
}

// Output tile of a workgroup (tile counts are powers of two).  Workgroups go to the eight
// XCDs in turn, each with its own L2: XCD x takes the x-th eighth of the tiles, in columns
// of up to 8 tiles of m, so that the 32 to 64 tiles it runs at once share 8 panels of A'
// and 4 to 8 of B' instead of one of B' and as many of A' as there are tiles.
__device__ __forceinline__ void gemm_tile(int64_t id, int64_t tiles_m, int64_t tiles_n, int64_t& tm, int64_t& tn) {
    const int64_t total = tiles_m * tiles_n;
    if (total >= 64) id = (id & 7) * (total >> 3) + (id >> 3);
    const int64_t gm = tiles_m < 8 ? tiles_m : 8;
    const int64_t per = gm * tiles_n, g = id / per, r = id % per;
    tm = g * gm + r % gm;
    tn = r / gm;
}

// Complex FP64 GEMM on MFMA: C[m + M n] = sum_s A'[s][m] * B'[s][n].
// 64x64 output tile per workgroup, four waves of 32x32; each 16x16 block of a wave
// takes four real v_mfma_f64_16x16x4f64 per k-step of 4 (re*re, -im*im, re*im, im*re).
// The MFMA row operand carries B' (rows = n) and the column operand A' (cols = m), so
// the lanes of one accumulator row hold 16 consecutive m and store contiguously.
constexpr int GM = 64, GN = 64, GK = 16;
typedef double d4_t __attribute__((ext_vector_type(4)));
typedef double d2_t __attribute__((ext_vector_type(2)));

__global__ __launch_bounds__(kThreads, 2) void k_gemm_c128(const double2* __restrict__ Ap,
                                                        const double2* __restrict__ Bp,
                                                        double2* __restrict__ C, int64_t M,
                                                        int64_t N, int64_t K) {
    __shared__ d2_t sa[2][GK][GM], sb[2][GK][GN];  // two k-tiles: one barrier per k-tile
    // split K: workgroups with blockIdx.z = z take summed rows [z K, (z + 1) K) and write
    // their own M x N partial product at C + z M N
    Ap += int64_t(blockIdx.z) * K * M;
    Bp += int64_t(blockIdx.z) * K * N;
    C += int64_t(blockIdx.z) * M * N;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave & 1, wn = wave >> 1;
    const int64_t tiles_m = M / GM;
    const int64_t tile = int64_t(blockIdx.x) + int64_t(blockIdx.y) * gridDim.x;
    if (tile >= tiles_m * (N / GN)) return;
    int64_t tm, tn;
    gemm_tile(tile, tiles_m, N / GN, tm, tn);
    const int64_t m0 = tm * GM, n0 = tn * GN;
    d4_t acc_re[2][2], acc_im[2][2];
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j) {
            acc_re[i][j] = d4_t{0, 0, 0, 0};
            acc_im[i][j] = d4_t{0, 0, 0, 0};
        }
    const int li = lane & 15, lk = lane >> 4;
    // each thread stages kPer elements of A' and of B' per k-tile: rows (tid / 64) + 4 q; the
    // next k-tile is in flight while the current one is multiplied from LDS.  A last
    // k-tile beyond K (K = 8) is filled with zeros, which add nothing.
    constexpr int kPer = GK * GM / kThreads;
    static_assert(GM == 64 && GN == 64 && kPer * kThreads == GK * GM, "tile staging");
    d2_t ra[kPer], rb[kPer];
    const d2_t* pa = reinterpret_cast<const d2_t*>(Ap) + int64_t(wave) * M + m0 + lane;
    const d2_t* pb = reinterpret_cast<const d2_t*>(Bp) + int64_t(wave) * N + n0 + lane;
    auto fetch = [&](int64_t k0) {
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            const bool in_k = k0 + wave + 4 * q < K;
            ra[q] = in_k ? pa[4 * q * M] : d2_t{0.0, 0.0};
            rb[q] = in_k ? pb[4 * q * N] : d2_t{0.0, 0.0};
        }
        pa += GK * M;
        pb += GK * N;
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            sa[buf][wave + 4 * q][lane] = ra[q];
            sb[buf][wave + 4 * q][lane] = rb[q];
        }
    };
    fetch(0);
    stage(0);
    __syncthreads();
    int buf = 0;
    for (int64_t k0 = 0; k0 < K; k0 += GK, buf ^= 1) {
        const bool more = k0 + GK < K;
        if (more) fetch(k0 + GK);
#pragma unroll
        for (int kk = 0; kk < GK; kk += 4) {
            const int kl = kk + lk;
            double are[2], aim[2];
#pragma unroll
            for (int bm = 0; bm < 2; ++bm) {
                const d2_t v = sa[buf][kl][wm * 32 + bm * 16 + li];
                are[bm] = v.x;
                aim[bm] = v.y;
            }
            double bre[2], bim[2];
#pragma unroll
            for (int bn = 0; bn < 2; ++bn) {
                const d2_t v = sb[buf][kl][wn * 32 + bn * 16 + li];
                bre[bn] = v.x;
                bim[bn] = v.y;
            }
            // the four products of a block go to two accumulators; issuing them in
            // four rounds over the blocks keeps dependent MFMAs apart
#pragma unroll
            for (int bn = 0; bn < 2; ++bn)
#pragma unroll
                for (int bm = 0; bm < 2; ++bm)
                    acc_re[bn][bm] = __builtin_amdgcn_mfma_f64_16x16x4f64(bre[bn], are[bm], acc_re[bn][bm], 0, 0, 0);
#pragma unroll
            for (int bn = 0; bn < 2; ++bn)
#pragma unroll
                for (int bm = 0; bm < 2; ++bm)
                    acc_im[bn][bm] = __builtin_amdgcn_mfma_f64_16x16x4f64(bim[bn], are[bm], acc_im[bn][bm], 0, 0, 0);
#pragma unroll
            for (int bn = 0; bn < 2; ++bn)
#pragma unroll
                for (int bm = 0; bm < 2; ++bm)
                    acc_re[bn][bm] = __builtin_amdgcn_mfma_f64_16x16x4f64(-bim[bn], aim[bm], acc_re[bn][bm], 0, 0, 0);
#pragma unroll
            for (int bn = 0; bn < 2; ++bn)
#pragma unroll
                for (int bm = 0; bm < 2; ++bm)
                    acc_im[bn][bm] = __builtin_amdgcn_mfma_f64_16x16x4f64(bre[bn], aim[bm], acc_im[bn][bm], 0, 0, 0);
        }
        if (more) stage(buf ^ 1);  // read last in the k-tile before, behind its barrier
        __syncthreads();
    }
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
        for (int bm = 0; bm < 2; ++bm)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // f64 16x16x4 accumulator: item r of lane l is row (l / 16) + 4 r, column l % 16
                const int64_t n = n0 + wn * 32 + bn * 16 + lk + 4 * r;
                const int64_t mm = m0 + wm * 32 + bm * 16 + li;
                C[mm + M * n] = double2{acc_re[bn][bm][r], acc_im[bn][bm][r]};
            }
}

// Complex64 GEMM on MFMA, C[m + M n] = sum_s A'[s][m] * B'[s][n], in the three
// complex64 forms.  64x64 output tile per workgroup, four waves of 32x32, k-tiles
// of 32.  4M and 3M use v_mfma_f32_16x16x4f32 (four / three real products per
// complex product); bf16x3 splits every FP32 operand into bf16 hi + lo when staging
// it in LDS and takes hi*hi + hi*lo + lo*hi on v_mfma_f32_16x16x32_bf16, all with
// FP32 accumulation.  f32 16x16 accumulator layout: item r of lane l is row
// 4 (l / 16) + r, column l % 16; rows are n (the B' operand), columns m (A').
constexpr int HK = 32;
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));

template <int MODE>
__global__ __launch_bounds__(kThreads) void k_gemm_c64(const float2* __restrict__ Ap, const float2* __restrict__ Bp,
                                                       float2* __restrict__ C, int64_t M, int64_t N, int64_t K) {
    // f32 forms: [k][row] planes of re / im; bf16x3: [row][k] planes of re_hi, re_lo,
    // im_hi, im_lo (k contiguous: one 16-byte load is a lane's 8 operands)
    constexpr int kPlaneF = HK * (GM + 1);
    constexpr int kRowB = HK + 8;
    constexpr int kPlaneB = GM * kRowB;
    __shared__ __align__(16) unsigned char smem[MODE == MODE_BF16X3 ? 2 * 4 * kPlaneB * 2 : 2 * 2 * kPlaneF * 4];
    // split K: workgroups with blockIdx.z = z take summed rows [z K, (z + 1) K) and write
    // their own M x N partial product at C + z M N
    Ap += int64_t(blockIdx.z) * K * M;
    Bp += int64_t(blockIdx.z) * K * N;
    C += int64_t(blockIdx.z) * M * N;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave & 1, wn = wave >> 1;
    const int li = lane & 15, lk = lane >> 4;
    const int64_t tiles_m = M / GM;
    const int64_t tile = int64_t(blockIdx.x) + int64_t(blockIdx.y) * gridDim.x;
    if (tile >= tiles_m * (N / GN)) return;
    const int64_t m0 = (tile % tiles_m) * GM, n0 = (tile / tiles_m) * GN;
    f4_t acc0[2][2], acc1[2][2], acc2[2][2];  // 4M / bf16x3: re, im; 3M: P1, P2, P3
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j) acc0[i][j] = acc1[i][j] = acc2[i][j] = f4_t{0, 0, 0, 0};
    for (int64_t k0 = 0; k0 < K; k0 += HK) {
        if constexpr (MODE == MODE_BF16X3) {
            uint16_t* sa = reinterpret_cast<uint16_t*>(smem);  // 4 planes of A', then 4 of B'
            uint16_t* sb = sa + 4 * kPlaneB;
            for (int e = tid; e < HK * GM; e += kThreads) {
                const int kk = e / GM, rr = e % GM;
                const bool in_k = k0 + kk < K;  // a last k-tile beyond K is zero-filled
                const float2 va = in_k ? Ap[(k0 + kk) * M + m0 + rr] : float2{0.0f, 0.0f};
                const float2 vb = in_k ? Bp[(k0 + kk) * N + n0 + rr] : float2{0.0f, 0.0f};
                const int o = rr * kRowB + kk;
                const float arh = bf16_round(va.x), aih = bf16_round(va.y);
                const float brh = bf16_round(vb.x), bih = bf16_round(vb.y);
                sa[o] = bf16_bits(arh);
                sa[kPlaneB + o] = bf16_bits(va.x - arh);
                sa[2 * kPlaneB + o] = bf16_bits(aih);
                sa[3 * kPlaneB + o] = bf16_bits(va.y - aih);
                sb[o] = bf16_bits(brh);
                sb[kPlaneB + o] = bf16_bits(vb.x - brh);
                sb[2 * kPlaneB + o] = bf16_bits(bih);
                sb[3 * kPlaneB + o] = bf16_bits(vb.y - bih);
            }
            __syncthreads();
            auto ld = [&](const uint16_t* plane, int row) {
                return *reinterpret_cast<const bf8_t*>(plane + row * kRowB + 8 * lk);
            };
            auto neg = [](bf8_t v) {
                uint4 u = *reinterpret_cast<uint4*>(&v);
                u.x ^= 0x80008000u;
                u.y ^= 0x80008000u;
                u.z ^= 0x80008000u;
                u.w ^= 0x80008000u;
                return *reinterpret_cast<bf8_t*>(&u);
            };
            bf8_t a[2][4];
#pragma unroll
            for (int bm = 0; bm < 2; ++bm)
#pragma unroll
                for (int q = 0; q < 4; ++q) a[bm][q] = ld(sa + q * kPlaneB, wm * 32 + bm * 16 + li);
            bf8_t b[2][6];  // per bn: re_hi, re_lo, im_hi, im_lo, -im_hi, -im_lo
#pragma unroll
            for (int bn = 0; bn < 2; ++bn) {
#pragma unroll
                for (int q = 0; q < 4; ++q) b[bn][q] = ld(sb + q * kPlaneB, wn * 32 + bn * 16 + li);
                b[bn][4] = neg(b[bn][2]);
                b[bn][5] = neg(b[bn][3]);
            }
            // re += br ar - bi ai; im += bi ar + br ai, each product hi*hi + hi*lo + lo*hi;
            // every round touches each of the eight accumulators once, so no MFMA waits
            // for the one before it.  (B operand index, A operand index) per round:
            constexpr int kRe[6][2] = {{0, 0}, {0, 1}, {1, 0}, {4, 2}, {4, 3}, {5, 2}};
            constexpr int kIm[6][2] = {{2, 0}, {2, 1}, {3, 0}, {0, 2}, {0, 3}, {1, 2}};
#pragma unroll
            for (int t = 0; t < 6; ++t)
#pragma unroll
                for (int bn = 0; bn < 2; ++bn)
#pragma unroll
                    for (int bm = 0; bm < 2; ++bm) {
                        acc0[bn][bm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[bn][kRe[t][0]], a[bm][kRe[t][1]],
                                                                               acc0[bn][bm], 0, 0, 0);
                        acc1[bn][bm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[bn][kIm[t][0]], a[bm][kIm[t][1]],
                                                                               acc1[bn][bm], 0, 0, 0);
                    }
        } else {
            float* sa = reinterpret_cast<float*>(smem);  // re plane, im plane of A', then of B'
            float* sb = sa + 2 * kPlaneF;
            for (int e = tid; e < HK * GM; e += kThreads) {
                const int kk = e / GM, rr = e % GM;
                const bool in_k = k0 + kk < K;  // a last k-tile beyond K is zero-filled
                const float2 va = in_k ? Ap[(k0 + kk) * M + m0 + rr] : float2{0.0f, 0.0f};
                const float2 vb = in_k ? Bp[(k0 + kk) * N + n0 + rr] : float2{0.0f, 0.0f};
                const int o = kk * (GM + 1) + rr;
                sa[o] = va.x;
                sa[kPlaneF + o] = va.y;
                sb[o] = vb.x;
                sb[kPlaneF + o] = vb.y;
            }
            __syncthreads();
#pragma unroll
            for (int kk = 0; kk < HK; kk += 4) {
                const int o = (kk + lk) * (GM + 1);
                float are[2], aim[2];
#pragma unroll
                for (int bm = 0; bm < 2; ++bm) {
                    are[bm] = sa[o + wm * 32 + bm * 16 + li];
                    aim[bm] = sa[kPlaneF + o + wm * 32 + bm * 16 + li];
                }
                float bre[2], bim[2];
#pragma unroll
                for (int bn = 0; bn < 2; ++bn) {
                    bre[bn] = sb[o + wn * 32 + bn * 16 + li];
                    bim[bn] = sb[kPlaneF + o + wn * 32 + bn * 16 + li];
                }
                // rounds over the four blocks (dependent MFMAs four apart)
                if constexpr (MODE == MODE_3M) {
#pragma unroll
                    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
                        for (int bm = 0; bm < 2; ++bm) {
                            acc0[bn][bm] = __builtin_amdgcn_mfma_f32_16x16x4f32(bre[bn], are[bm], acc0[bn][bm], 0, 0, 0);
                            acc1[bn][bm] = __builtin_amdgcn_mfma_f32_16x16x4f32(bim[bn], aim[bm], acc1[bn][bm], 0, 0, 0);
                            acc2[bn][bm] = __builtin_amdgcn_mfma_f32_16x16x4f32(bre[bn] + bim[bn], are[bm] + aim[bm],
                                                                               acc2[bn][bm], 0, 0, 0);
                        }
                } else {
#pragma unroll
                    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
                        for (int bm = 0; bm < 2; ++bm) {
                            acc0[bn][bm] = __builtin_amdgcn_mfma_f32_16x16x4f32(bre[bn], are[bm], acc0[bn][bm], 0, 0, 0);
                            acc1[bn][bm] = __builtin_amdgcn_mfma_f32_16x16x4f32(bim[bn], are[bm], acc1[bn][bm], 0, 0, 0);
                        }
#pragma unroll
                    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
                        for (int bm = 0; bm < 2; ++bm) {
                            acc0[bn][bm] = __builtin_amdgcn_mfma_f32_16x16x4f32(-bim[bn], aim[bm], acc0[bn][bm], 0, 0, 0);
                            acc1[bn][bm] = __builtin_amdgcn_mfma_f32_16x16x4f32(bre[bn], aim[bm], acc1[bn][bm], 0, 0, 0);
                        }
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int bn = 0; bn < 2; ++bn)
#pragma unroll
        for (int bm = 0; bm < 2; ++bm)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t n = n0 + wn * 32 + bn * 16 + 4 * lk + r;
                const int64_t mm = m0 + wm * 32 + bm * 16 + li;
                float2 v;
                if constexpr (MODE == MODE_3M) {
                    v.x = acc0[bn][bm][r] - acc1[bn][bm][r];
                    v.y = acc2[bn][bm][r] - acc0[bn][bm][r] - acc1[bn][bm][r];
                } else {
                    v.x = acc0[bn][bm][r];
                    v.y = acc1[bn][bm][r];
                }
                C[mm + M * n] = v;
            }
}

__global__ void k_fill_zero(uint4* p, int64_t n16) {
    const int64_t stride = int64_t(gridDim.x) * blockDim.x;
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n16; i += stride)
        p[i] = uint4{0, 0, 0, 0};
}

inline unsigned grid_for(int64_t items, int64_t per_block, unsigned cap) {
    int64_t g = (items + per_block - 1) / per_block;
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return unsigned(g);
}

template <class V, int MODE>
qt_status run_direct(Ctx* c, const V* A, const V* B, V* C, const BitMap& m) {
    const int64_t nC = int64_t(1) << m.nbits_c;
    const unsigned grid = grid_for(nC, kThreads, 16384);
    hipLaunchKernelGGL((k_direct<V, MODE>), dim3(grid), dim3(kThreads), 0, c->stream, A, B, C, m, nC);
    return check_hip(c, hipGetLastError(), "k_direct");
}

template <class V, int MODE, int NB>
qt_status launch_skinny(Ctx* c, const V* A, const V* B, V* C, const BitMap& m, int mbits, bool small_b) {
    const int64_t n_big = int64_t(1) << (m.nbits_c - NB);
    const unsigned grid = grid_for(n_big, kThreads, 16384);
    if (small_b)
        hipLaunchKernelGGL((k_skinny<V, MODE, NB, true>), dim3(grid), dim3(kThreads), 0, c->stream, A, B, C, m,
                           mbits, n_big);
    else
        hipLaunchKernelGGL((k_skinny<V, MODE, NB, false>), dim3(grid), dim3(kThreads), 0, c->stream, A, B, C, m,
                           mbits, n_big);
    return check_hip(c, hipGetLastError(), "k_skinny");
}

template <class V, int MODE, int NS, int NB>
qt_status launch_thin_nb(Ctx* c, const V* X, const V* G, V* C, const ThinArgs& r, bool small_b) {
    // one element per lane, no grid-stride reuse: on MI355X streaming kernels reach
    // their highest HBM rates with a workgroup per 256 elements (a capped grid looping
    // over the tensor measured 10-30 % slower, two adjacent elements per lane 5-8 %)
    const unsigned grid = grid_for(r.n_big, kThreads, 1u << 30);
    if (small_b)
        hipLaunchKernelGGL((k_thin<V, MODE, NS, NB, true>), dim3(grid), dim3(kThreads), 0, c->stream, X, G, C, r);
    else
        hipLaunchKernelGGL((k_thin<V, MODE, NS, NB, false>), dim3(grid), dim3(kThreads), 0, c->stream, X, G, C, r);
    return check_hip(c, hipGetLastError(), "k_thin");
}

template <class V, int MODE, int NS>
qt_status launch_thin_ns(Ctx* c, const V* X, const V* G, V* C, const ThinArgs& r, int nb, bool small_b) {
    switch (nb) {
        case 0: return launch_thin_nb<V, MODE, NS, 0>(c, X, G, C, r, small_b);
        case 1: return launch_thin_nb<V, MODE, NS, 1>(c, X, G, C, r, small_b);
        case 2: return launch_thin_nb<V, MODE, NS, 2>(c, X, G, C, r, small_b);
        case 3: return launch_thin_nb<V, MODE, NS, 3>(c, X, G, C, r, small_b);
        default: return launch_thin_nb<V, MODE, NS, 4>(c, X, G, C, r, small_b);
    }
}

// k_thin when it applies (1-4 summed bits, at most 4 bits on the small side, the
// large side's free bits in their own order in C); false otherwise.
template <class V, int MODE>
bool try_thin(Ctx* c, const V* A, const V* B, V* C, const BitMap& m, int mbits, bool small_b, qt_status* st) {
    const int nb = small_b ? m.nbits_c - mbits : mbits;
    const int ns = m.nbits_s;
    if (ns < 1 || ns > 4 || nb > 4) return false;
    // the large side's C bits, in C order, must be its free bits in increasing order
    const int lo = small_b ? 0 : nb, hi = small_b ? mbits : m.nbits_c;
    int prev = -1;
    for (int i = lo; i < hi; ++i) {
        const int src = small_b ? m.c_src[i] : m.c_src[i] - 64;
        if (src <= prev) return false;
        prev = src;
    }
    ThinArgs r;
    std::memset(&r, 0, sizeof r);
    r.n_big = int64_t(1) << (hi - lo);
    r.lo_bits = mbits;
    int pos[4];
    for (int d = 0; d < ns; ++d) pos[d] = small_b ? m.s_a[d] : m.s_b[d];
    std::sort(pos, pos + ns);
    r.n_ins = ns;
    for (int d = 0; d < ns; ++d) r.ins_pos[d] = pos[d];
    for (int j = 0; j < (1 << ns); ++j) {
        int64_t gb = 0, gs = 0;
        for (int d = 0; d < ns; ++d)
            if ((j >> d) & 1) {
                gb += int64_t(1) << (small_b ? m.s_a[d] : m.s_b[d]);
                gs += int64_t(1) << (small_b ? m.s_b[d] : m.s_a[d]);
            }
        r.g_big[j] = gb;
        r.g_small[j] = int32_t(gs);
    }
    for (int o = 0; o < (1 << nb); ++o) {
        int64_t off = 0;
        for (int i = 0; i < nb; ++i)
            if ((o >> i) & 1) {
                const int src = small_b ? m.c_src[mbits + i] - 64 : m.c_src[i];
                off += int64_t(1) << src;
            }
        r.small_off[o] = int32_t(off);
    }
    const V* X = small_b ? A : B;
    const V* G = small_b ? B : A;
    switch (ns) {
        case 1: *st = launch_thin_ns<V, MODE, 1>(c, X, G, C, r, nb, small_b); break;
        case 2: *st = launch_thin_ns<V, MODE, 2>(c, X, G, C, r, nb, small_b); break;
        case 3: *st = launch_thin_ns<V, MODE, 3>(c, X, G, C, r, nb, small_b); break;
        default: *st = launch_thin_ns<V, MODE, 4>(c, X, G, C, r, nb, small_b); break;
    }
    return true;
}

// C = [A part (mbits) | B part]; the side with at most 5 bits is the small one
template <class V, int MODE>
qt_status run_skinny(Ctx* c, const V* A, const V* B, V* C, const BitMap& m, int mbits) {
    const int nbits_n = m.nbits_c - mbits;
    const bool small_b = nbits_n <= 5;
    qt_status st = QT_OK;
    if (try_thin<V, MODE>(c, A, B, C, m, mbits, small_b, &st)) return st;
    switch (small_b ? nbits_n : mbits) {
        case 0: return launch_skinny<V, MODE, 0>(c, A, B, C, m, mbits, small_b);
        case 1: return launch_skinny<V, MODE, 1>(c, A, B, C, m, mbits, small_b);
        case 2: return launch_skinny<V, MODE, 2>(c, A, B, C, m, mbits, small_b);
        case 3: return launch_skinny<V, MODE, 3>(c, A, B, C, m, mbits, small_b);
        case 4: return launch_skinny<V, MODE, 4>(c, A, B, C, m, mbits, small_b);
        default: return launch_skinny<V, MODE, 5>(c, A, B, C, m, mbits, small_b);
    }
}

template <class V, int MODE, int GA, int GB>
qt_status launch_rows(Ctx* c, dim3 grid, const V* A, const V* B, V* part, const BitMap& m, int step_bits,
                      const RowSet& r) {
    hipLaunchKernelGGL((k_reduce_rows<V, MODE, GA, GB>), grid, dim3(kThreads), 0, c->stream, A, B, part, m, step_bits,
                       r);
    return check_hip(c, hipGetLastError(), "k_reduce_rows");
}

template <class V, int MODE>
qt_status launch_reduce_rows(Ctx* c, int ga, int gb, dim3 grid, const V* A, const V* B, V* part, const BitMap& m,
                             int step_bits, const RowSet& r) {
#define QT_ROWS(GA, GB) \
    case GA * 64 + GB: return launch_rows<V, MODE, GA, GB>(c, grid, A, B, part, m, step_bits, r)
    switch (ga * 64 + gb) {
        QT_ROWS(1, 1); QT_ROWS(1, 2); QT_ROWS(1, 4); QT_ROWS(1, 8); QT_ROWS(1, 16);
        QT_ROWS(2, 1); QT_ROWS(2, 2); QT_ROWS(2, 4); QT_ROWS(2, 8);
        QT_ROWS(4, 1); QT_ROWS(4, 2); QT_ROWS(4, 4);
        QT_ROWS(8, 1); QT_ROWS(8, 2);
        QT_ROWS(16, 1);
        default: break;
    }
    if constexpr (sizeof(V) == 8) {
        switch (ga * 64 + gb) {
            QT_ROWS(1, 32); QT_ROWS(2, 16); QT_ROWS(4, 8); QT_ROWS(8, 4); QT_ROWS(16, 2); QT_ROWS(32, 1);
            default: break;
        }
    }
#undef QT_ROWS
    return set_error(c, QT_UNSUPPORTED, "split reduction: unsupported row grouping");
}

// The summed bits in the order k_reduce_rows takes them: the lowest position in A not yet
// taken, then the lowest in B, and so on (bits 0-5 are a wave's lanes: three bits of each
// operand are 64 bytes of complex64, 128 of complex128).
void order_summed_bits(BitMap& m) {
    const int n = m.nbits_s;
    int by_a[64], by_b[64];
    for (int j = 0; j < n; ++j) by_a[j] = by_b[j] = j;
    std::sort(by_a, by_a + n, [&](int x, int y) { return m.s_a[x] < m.s_a[y]; });
    std::sort(by_b, by_b + n, [&](int x, int y) { return m.s_b[x] < m.s_b[y]; });
    bool taken[64] = {false};
    uint8_t sa[64], sb[64];
    for (int k = 0, ia = 0, ib = 0; k < n; ++k) {
        const int* by = (k & 1) == 0 ? by_a : by_b;
        int& i = (k & 1) == 0 ? ia : ib;
        while (taken[by[i]]) ++i;
        const int j = by[i];
        taken[j] = true;
        sa[k] = m.s_a[j];
        sb[k] = m.s_b[j];
    }
    std::memcpy(m.s_a, sa, size_t(n));
    std::memcpy(m.s_b, sb, size_t(n));
}

// *no_room: nothing was queued, the partial sums found no device memory.
template <class V, int MODE>
qt_status run_reduce(Ctx* c, const V* A, const V* B, V* C, const BitMap& m0, const Workspace* ws, bool* no_room) {
    BitMap m = m0;
    order_summed_bits(m);
    const int64_t nC = int64_t(1) << m.nbits_c;
    const int64_t nS = int64_t(1) << m.nbits_s;
    // free bits of each side, lowest operand position first: a group's rows are the
    // lowest ones, neighbours in memory
    struct Bit {
        int pos, c;
    };
    Bit fa[64], fb[64];
    int ka = 0, kb = 0;
    for (int i = 0; i < m.nbits_c; ++i) {
        if (m.c_src[i] < 64) fa[ka++] = Bit{m.c_src[i], i};
        else fb[kb++] = Bit{m.c_src[i] - 64, i};
    }
    auto lower = [](const Bit& x, const Bit& y) { return x.pos < y.pos; };
    std::sort(fa, fa + ka, lower);
    std::sort(fb, fb + kb, lower);
    // rows per group: A is read 2^(kb - gb) times, B 2^(ka - ga) times; the accumulators
    // of 2^5 outputs (complex64) or 2^4 fit the registers at two waves per SIMD and more
    const int out_bits = sizeof(V) == 8 ? 5 : 4;
    int ga = 0, gb = 0;
    double least = -1;
    for (int x = 0; x <= ka && x <= out_bits; ++x) {
        const int y = kb < out_bits - x ? kb : out_bits - x;
        const double cost = std::ldexp(1.0, ka + kb - y) + std::ldexp(1.0, kb + ka - x);
        if (least < 0 || cost < least) {
            least = cost;
            ga = x;
            gb = y;
        }
    }
    const int64_t groups = int64_t(1) << (ka - ga + kb - gb);
    // 16 steps of 256 summed indices per workgroup: fewer where that leaves the chip with
    // less than two workgroups per CU (but not where it saves the second pass), more only
    // beyond 2^15 workgroups, and at most 2^12 (the kernel's offset tables)
    int step_bits = m.nbits_s - 8 < 4 ? m.nbits_s - 8 : 4;
    while (step_bits > 0 && groups * ((nS >> 8) >> step_bits) < 512 && !(groups >= 128 && (nS >> 8) >> step_bits == 1))
        --step_bits;
    while ((nS >> 8) >> step_bits > kReduceMaxBlocks && step_bits < 12) ++step_bits;
    // partial sums of at most 32 MiB
    while (((nS >> 8) >> step_bits) * nC * int64_t(sizeof(V)) > (int64_t(32) << 20) && (nS >> 8) >> step_bits > 1 &&
           step_bits < 12)
        ++step_bits;
    const int64_t nblocks = (nS >> 8) >> step_bits;
    V* part = C;
    if (nblocks > 1) {
        const size_t need = size_t(nblocks * nC) * sizeof(V);
        if (ws) {
            if (need > ws->bytes)
                return set_error(c, QT_INVALID_INPUT, "split reduction: partial sums exceed the workspace");
            part = reinterpret_cast<V*>(ws->base);
        } else {
            if (c->partials_bytes < need) {
                if (c->partials) {
                    (void)hipStreamSynchronize(c->stream);
                    (void)hipFree(c->partials);
                    c->partials = nullptr;
                    c->partials_bytes = 0;
                }
                if (hipMalloc(&c->partials, need) != hipSuccess) {
                    (void)hipGetLastError();
                    c->partials = nullptr;
                    *no_room = true;
                    return QT_OOM;
                }
                c->partials_bytes = need;
            }
            part = static_cast<V*>(c->partials);
        }
    }
    RowSet r;
    std::memset(&r, 0, sizeof r);
    const int na = 1 << ga, nb = 1 << gb;
    for (int x = 0; x < na; ++x)
        for (int k = 0; k < ga; ++k)
            if ((x >> k) & 1) r.oa[x] += int64_t(1) << fa[k].pos;
    for (int y = 0; y < nb; ++y)
        for (int k = 0; k < gb; ++k)
            if ((y >> k) & 1) r.ob[y] += int64_t(1) << fb[k].pos;
    for (int x = 0; x < na; ++x)
        for (int y = 0; y < nb; ++y) {
            int32_t o = 0;
            for (int k = 0; k < ga; ++k)
                if ((x >> k) & 1) o += 1 << fa[k].c;
            for (int k = 0; k < gb; ++k)
                if ((y >> k) & 1) o += 1 << fb[k].c;
            r.c[x * nb + y] = o;
        }
    for (int k = ga; k < ka; ++k, ++r.n_ga) {
        r.ga_pos[r.n_ga] = fa[k].pos;
        r.ga_c[r.n_ga] = fa[k].c;
    }
    for (int k = gb; k < kb; ++k, ++r.n_gb) {
        r.gb_pos[r.n_gb] = fb[k].pos;
        r.gb_c[r.n_gb] = fb[k].c;
    }
    qt_status s = launch_reduce_rows<V, MODE>(c, na, nb, dim3(unsigned(nblocks), unsigned(groups)), A, B, part, m,
                                              step_bits, r);
    if (s != QT_OK || nblocks == 1) return s;
    hipLaunchKernelGGL((k_reduce_final<V>), dim3(unsigned(nC)), dim3(kThreads), 0, c->stream, part, C, nblocks);
    return check_hip(c, hipGetLastError(), "k_reduce_final");
}

template <class V>
qt_status run_permute(Ctx* c, const V* in, V* out, const PermPlan& p) {
    const int64_t blocks = int64_t(1) << p.n_rest;
    const unsigned gx = unsigned(blocks < 65536 ? blocks : 65536);
    const unsigned gy = unsigned((blocks + gx - 1) / gx);
    const size_t lds = (size_t(1) << (p.tl + p.n_extra_in)) * sizeof(V);
    // element pairs need input and output bit 0 inside the tile (tl >= 1) and 16-byte
    // aligned buffers
    const bool pairs = p.tl >= 1 && (reinterpret_cast<uintptr_t>(in) & 15) == 0 &&
                       (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    if constexpr (sizeof(V) == 8) {
        if (pairs) {
            hipLaunchKernelGGL((k_permute<V, 1, false>), dim3(gx, gy), dim3(kThreads), lds, c->stream, in, out, p);
            return check_hip(c, hipGetLastError(), "k_permute");
        }
    }
    hipLaunchKernelGGL((k_permute<V, 0, false>), dim3(gx, gy), dim3(kThreads), lds, c->stream, in, out, p);
    return check_hip(c, hipGetLastError(), "k_permute");
}

// in -> four bf16 planes in `out` (2^nbits elements of 8 bytes in all)
qt_status run_permute_split(Ctx* c, const float2* in, void* out, const PermPlan& p) {
    const int64_t blocks = int64_t(1) << p.n_rest;
    const unsigned gx = unsigned(blocks < 65536 ? blocks : 65536);
    const unsigned gy = unsigned((blocks + gx - 1) / gx);
    const size_t lds = (size_t(1) << (p.tl + p.n_extra_in)) * sizeof(float2);
    hipLaunchKernelGGL((k_permute<float2, 1, true>), dim3(gx, gy), dim3(kThreads), lds, c->stream, in,
                       static_cast<float2*>(out), p);
    return check_hip(c, hipGetLastError(), "k_permute (split)");
}

bool is_identity(const int* src, int n) {
    for (int i = 0; i < n; ++i)
        if (src[i] != i) return false;
    return true;
}

}  // namespace

PermPlan make_perm_plan(int nbits, const int* src, int tile_bits_max) {
    PermPlan p;
    std::memset(&p, 0, sizeof p);
    p.nbits = nbits;
    // tile of 2^tbits elements, tbits = tl + (output-low bits that come from outside the
    // input-low ones): the largest tl whose tile has at most 2^tile_bits_max elements
    // and leaves at least 2^10 tiles (tbits never falls with tl).  Measured on 2^22- to
    // 2^28-element operands: the largest tiles (2^12 elements) move the most bytes per
    // second (2^28 complex64 elements, low and high 14 bits exchanged: 1.14 ms with
    // 2^12-element tiles, 2.12 ms with 2^10), and tiles under 2^8 leave most of a
    // workgroup's lanes idle (a permutation that keeps its low 6 bits in place ran at
    // 0.3 TB/s with tiles of 2^6)
    auto tbits_for = [&](int t) {
        int n = t;
        for (int j = 0; j < t; ++j) n += src[j] >= t ? 1 : 0;
        return n;
    };
    int cap = nbits - 10 < tile_bits_max ? nbits - 10 : tile_bits_max;
    if (cap < 6) cap = 6;
    int tl = 1;
    while (tl < nbits && tbits_for(tl + 1) <= cap) ++tl;
    if (tl > nbits) tl = nbits;
    p.tl = tl;
    int inv[64];
    for (int j = 0; j < nbits; ++j) inv[src[j]] = j;
    int tile_of_input[64];
    for (int i = 0; i < 64; ++i) tile_of_input[i] = -1;
    for (int i = 0; i < tl; ++i) tile_of_input[i] = i;
    for (int j = 0; j < tl; ++j) {
        const int s = src[j];
        if (s >= tl) {
            p.extra_in_pos[p.n_extra_in] = uint8_t(s);
            p.extra_in_out[p.n_extra_in] = uint8_t(j);
            tile_of_input[s] = tl + p.n_extra_in;
            ++p.n_extra_in;
        }
    }
    for (int i = 0; i < tl; ++i) p.lowin_out[i] = uint8_t(inv[i]);
    for (int j = 0; j < tl; ++j) p.lowout_tile[j] = uint8_t(tile_of_input[src[j]]);
    for (int i = 0; i < tl; ++i)
        if (inv[i] >= tl) {
            p.extra_out_pos[p.n_extra_out] = uint8_t(inv[i]);
            p.extra_out_tile[p.n_extra_out] = uint8_t(i);
            ++p.n_extra_out;
        }
    for (int i = 0; i < nbits; ++i)
        if (tile_of_input[i] < 0) {
            p.rest_in[p.n_rest] = uint8_t(i);
            p.rest_out[p.n_rest] = uint8_t(inv[i]);
            ++p.n_rest;
        }
    return p;
}

qt_status permute(Ctx* c, const void* in, void* out, int dtype, const PermPlan& p) {
    if (dtype == QT_DTYPE_C128)
        return run_permute<double2>(c, static_cast<const double2*>(in), static_cast<double2*>(out), p);
    return run_permute<float2>(c, static_cast<const float2*>(in), static_cast<float2*>(out), p);
}

namespace {

// Large complex64 GEMMs in the 4M / 3M forms: 128x128 output tile per workgroup,
// four waves of 64x64 (4x4 blocks of v_mfma_f32_16x16x4f32), k-tiles of 16; the next
// k-tile is staged in a second LDS buffer while the current one is multiplied.
// LDS rows are 144 complex values apart (288 words: half of the 64 banks beyond whole
// turns), so the two k-rows that half a wave reads at once sit in different halves.
constexpr int BT = 128, BK = 16, BROW = BT + 16;
constexpr int64_t kSplitRows = 256;

// C = the sum of S partial products part[z] (z in order), one complex128 per lane
__global__ __launch_bounds__(kThreads) void k_sum_splits_c128(const double2* __restrict__ part,
                                                              double2* __restrict__ C, int64_t n, int S) {
    const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= n) return;
    double2 a = part[i];
    for (int z = 1; z < S; ++z) {
        const double2 b = part[int64_t(z) * n + i];
        a.x += b.x;
        a.y += b.y;
    }
    C[i] = a;
}

// C = the sum of S partial products part[z] (z in order), two complex64 per lane
__global__ __launch_bounds__(kThreads) void k_sum_splits(const float4* __restrict__ part, float4* __restrict__ C,
                                                         int64_t n4, int S) {
    const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= n4) return;
    float4 a = part[i];
    for (int z = 1; z < S; ++z) {
        const float4 b = part[int64_t(z) * n4 + i];
        a.x += b.x;
        a.y += b.y;
        a.z += b.z;
        a.w += b.w;
    }
    C[i] = a;
}

// Two workgroups a CU (4M: 128 accumulation registers of 256) cover each other's barriers
// and LDS latency; 3M's 192 leave room for one.
template <int MODE>
__global__ __launch_bounds__(kThreads, MODE == MODE_3M ? 1 : 2) void k_gemm_c64_big(
    const float2* __restrict__ Ap, const float2* __restrict__ Bp, float2* __restrict__ C, int64_t M, int64_t N,
    int64_t K) {
    __shared__ float2 sa[2][BK * BROW], sb[2][BK * BROW];  // [buffer][k][row]
    // split K: workgroups with blockIdx.z = z take summed rows [z K, (z + 1) K) and write
    // their own M x N partial product at C + z M N
    Ap += int64_t(blockIdx.z) * K * M;
    Bp += int64_t(blockIdx.z) * K * N;
    C += int64_t(blockIdx.z) * M * N;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave & 1, wn = wave >> 1;
    const int li = lane & 15, lk = lane >> 4;
    const int64_t tiles_m = M / BT;
    const int64_t tile = int64_t(blockIdx.x) + int64_t(blockIdx.y) * gridDim.x;
    if (tile >= tiles_m * (N / BT)) return;
    int64_t tm, tn;
    gemm_tile(tile, tiles_m, N / BT, tm, tn);
    const int64_t m0 = tm * BT, n0 = tn * BT;
    constexpr int NA = MODE == MODE_3M ? 3 : 2;
    f4_t acc[NA][4][4];
#pragma unroll
    for (int q = 0; q < NA; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[q][i][j] = f4_t{0, 0, 0, 0};
    // each thread moves 8 elements of A' and 8 of B' per k-tile, two neighbours per load:
    // rows (tid / 64) + 4 q, elements 2 (tid % 64) and the next
    f4_t ra[4], rb[4];
    const float2* pa = Ap + int64_t(tid >> 6) * M + m0 + 2 * (tid & 63);
    const float2* pb = Bp + int64_t(tid >> 6) * N + n0 + 2 * (tid & 63);
    auto fetch = [&]() {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            ra[q] = *reinterpret_cast<const f4_t*>(pa + 4 * q * M);
            rb[q] = *reinterpret_cast<const f4_t*>(pb + 4 * q * N);
        }
        pa += BK * M;
        pb += BK * N;
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int o = ((tid >> 6) + 4 * q) * BROW + 2 * (tid & 63);
            *reinterpret_cast<f4_t*>(&sa[buf][o]) = ra[q];
            *reinterpret_cast<f4_t*>(&sb[buf][o]) = rb[q];
        }
    };
    fetch();
    stage(0);
    __syncthreads();
    int buf = 0;
    for (int64_t k0 = 0; k0 < K; k0 += BK, buf ^= 1) {
        const bool more = k0 + BK < K;
        if (more) fetch();
#pragma unroll
        for (int kk = 0; kk < BK; kk += 4) {
            const int o = (kk + lk) * BROW;
            float ar[4], ai[4], br[4], bi[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float2 va = sa[buf][o + wm * 64 + i * 16 + li], vb = sb[buf][o + wn * 64 + i * 16 + li];
                ar[i] = va.x;
                ai[i] = va.y;
                br[i] = vb.x;
                bi[i] = vb.y;
            }
            // one round of MFMAs over all 16 blocks per product, so that no MFMA waits
            // for the one just before it
            if constexpr (MODE == MODE_3M) {
                float sr[4], si[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    sr[i] = br[i] + bi[i];
                    si[i] = ar[i] + ai[i];
                }
#pragma unroll
                for (int bn = 0; bn < 4; ++bn)
#pragma unroll
                    for (int bm = 0; bm < 4; ++bm)
                        acc[0][bn][bm] = __builtin_amdgcn_mfma_f32_16x16x4f32(br[bn], ar[bm], acc[0][bn][bm], 0, 0, 0);
#pragma unroll
                for (int bn = 0; bn < 4; ++bn)
#pragma unroll
                    for (int bm = 0; bm < 4; ++bm)
                        acc[1][bn][bm] = __builtin_amdgcn_mfma_f32_16x16x4f32(bi[bn], ai[bm], acc[1][bn][bm], 0, 0, 0);
#pragma unroll
                for (int bn = 0; bn < 4; ++bn)
#pragma unroll
                    for (int bm = 0; bm < 4; ++bm)
                        acc[2][bn][bm] = __builtin_amdgcn_mfma_f32_16x16x4f32(sr[bn], si[bm], acc[2][bn][bm], 0, 0, 0);
            } else {
#pragma unroll
                for (int bn = 0; bn < 4; ++bn)
#pragma unroll
                    for (int bm = 0; bm < 4; ++bm)
                        acc[0][bn][bm] = __builtin_amdgcn_mfma_f32_16x16x4f32(br[bn], ar[bm], acc[0][bn][bm], 0, 0, 0);
#pragma unroll
                for (int bn = 0; bn < 4; ++bn)
#pragma unroll
                    for (int bm = 0; bm < 4; ++bm)
                        acc[1][bn][bm] = __builtin_amdgcn_mfma_f32_16x16x4f32(bi[bn], ar[bm], acc[1][bn][bm], 0, 0, 0);
#pragma unroll
                for (int bn = 0; bn < 4; ++bn)
#pragma unroll
                    for (int bm = 0; bm < 4; ++bm)
                        acc[0][bn][bm] = __builtin_amdgcn_mfma_f32_16x16x4f32(-bi[bn], ai[bm], acc[0][bn][bm], 0, 0, 0);
#pragma unroll
                for (int bn = 0; bn < 4; ++bn)
#pragma unroll
                    for (int bm = 0; bm < 4; ++bm)
                        acc[1][bn][bm] = __builtin_amdgcn_mfma_f32_16x16x4f32(br[bn], ai[bm], acc[1][bn][bm], 0, 0, 0);
            }
        }
        if (more) stage(buf ^ 1);  // read last in the k-tile before, behind its barrier
        __syncthreads();
    }
#pragma unroll
    for (int bn = 0; bn < 4; ++bn)
#pragma unroll
        for (int bm = 0; bm < 4; ++bm)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t n = n0 + wn * 64 + bn * 16 + 4 * lk + r;
                const int64_t mm = m0 + wm * 64 + bm * 16 + li;
                float2 v;
                if constexpr (MODE == MODE_3M) {
                    v.x = acc[0][bn][bm][r] - acc[1][bn][bm][r];
                    v.y = acc[2][bn][bm][r] - acc[0][bn][bm][r] - acc[1][bn][bm][r];
                } else {
                    v.x = acc[0][bn][bm][r];
                    v.y = acc[1][bn][bm][r];
                }
                C[mm + M * n] = v;
            }
}

// Large bf16x3 GEMMs: the permutes write the operands as bf16 planes in the order that an
// MFMA lane reads, plane[k / 8][row][k % 8], so a k-tile goes to LDS and from LDS to the
// matrix cores in 16-byte pieces without any conversion (k_gemm_c64 splits every element
// again for each tile that reads it, in 2-byte LDS writes: 235 million bank-conflict cycles
// on the product below).  128 x 128 outputs, four waves of 64 x 64, k-tiles of 32 in two LDS
// buffers; same products in the same order as k_gemm_c64.
constexpr int kPlaneTile = 4 * BT;  // 16-byte pieces of one plane of a k-tile: [k / 8][row]

__global__ __launch_bounds__(kThreads, 1) void k_gemm_bf16x3(const uint4* __restrict__ Ap, const uint4* __restrict__ Bp,
                                                             float2* __restrict__ C, int64_t M, int64_t N, int64_t K,
                                                             int64_t k_all) {
    __shared__ uint4 lds[2][2][4 * kPlaneTile];  // [buffer][operand][plane][k / 8][row]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave & 1, wn = wave >> 1;
    const int li = lane & 15, lk = lane >> 4;
    const int64_t tiles_m = M / BT;
    const int64_t tile = int64_t(blockIdx.x) + int64_t(blockIdx.y) * gridDim.x;
    if (tile >= tiles_m * (N / BT)) return;
    int64_t tm, tn;
    gemm_tile(tile, tiles_m, N / BT, tm, tn);
    const int64_t m0 = tm * BT, n0 = tn * BT;
    // split K: workgroups with blockIdx.z = z take summed rows [z K, (z + 1) K) and write
    // their own M x N partial product at C + z M N
    const int64_t k8_0 = int64_t(blockIdx.z) * (K / 8);
    C += int64_t(blockIdx.z) * M * N;
    f4_t acc_re[4][4], acc_im[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc_re[i][j] = acc_im[i][j] = f4_t{0, 0, 0, 0};
    // a thread moves piece tid + 256 q of each plane: k / 8 = tid / 128 + 2 q, row tid % 128
    typedef uint32_t u4_t __attribute__((ext_vector_type(4)));
    u4_t ra[4][2], rb[4][2];
    const u4_t* pa = reinterpret_cast<const u4_t*>(Ap) + (k8_0 + (tid >> 7)) * M + m0 + (tid & 127);
    const u4_t* pb = reinterpret_cast<const u4_t*>(Bp) + (k8_0 + (tid >> 7)) * N + n0 + (tid & 127);
    const int64_t plane_a = k_all / 8 * M, plane_b = k_all / 8 * N;
    auto fetch = [&]() {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                ra[q][h] = pa[q * plane_a + 2 * h * M];
                rb[q][h] = pb[q * plane_b + 2 * h * N];
            }
        pa += 4 * M;
        pb += 4 * N;
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                *reinterpret_cast<u4_t*>(&lds[buf][0][q * kPlaneTile + tid + kThreads * h]) = ra[q][h];
                *reinterpret_cast<u4_t*>(&lds[buf][1][q * kPlaneTile + tid + kThreads * h]) = rb[q][h];
            }
    };
    auto frag = [&](int buf, int op, int q, int row) {
        return *reinterpret_cast<const bf8_t*>(&lds[buf][op][q * kPlaneTile + lk * BT + row]);
    };
    auto neg = [](bf8_t v) {
        u4_t u = *reinterpret_cast<u4_t*>(&v);
        u ^= 0x80008000u;
        return *reinterpret_cast<bf8_t*>(&u);
    };
    fetch();
    stage(0);
    __syncthreads();
    int buf = 0;
    for (int64_t k0 = 0; k0 < K; k0 += HK, buf ^= 1) {
        const bool more = k0 + HK < K;
        if (more) fetch();
        bf8_t a[4][4];
#pragma unroll
        for (int bm = 0; bm < 4; ++bm)
#pragma unroll
            for (int q = 0; q < 4; ++q) a[bm][q] = frag(buf, 0, q, wm * 64 + bm * 16 + li);
        // re += br ar - bi ai; im += bi ar + br ai, each product hi*hi + hi*lo + lo*hi: (B
        // operand, A operand) per round, 4 and 5 being -im hi and -im lo
        constexpr int kRe[6][2] = {{0, 0}, {0, 1}, {1, 0}, {4, 2}, {4, 3}, {5, 2}};
        constexpr int kIm[6][2] = {{2, 0}, {2, 1}, {3, 0}, {0, 2}, {0, 3}, {1, 2}};
#pragma unroll
        for (int bn = 0; bn < 4; ++bn) {
            bf8_t b[6];
#pragma unroll
            for (int q = 0; q < 4; ++q) b[q] = frag(buf, 1, q, wn * 64 + bn * 16 + li);
            b[4] = neg(b[2]);
            b[5] = neg(b[3]);
#pragma unroll
            for (int t = 0; t < 6; ++t)
#pragma unroll
                for (int bm = 0; bm < 4; ++bm) {
                    acc_re[bn][bm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[kRe[t][0]], a[bm][kRe[t][1]],
                                                                             acc_re[bn][bm], 0, 0, 0);
                    acc_im[bn][bm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[kIm[t][0]], a[bm][kIm[t][1]],
                                                                             acc_im[bn][bm], 0, 0, 0);
                }
        }
        if (more) stage(buf ^ 1);  // read last in the k-tile before, behind its barrier
        __syncthreads();
    }
#pragma unroll
    for (int bn = 0; bn < 4; ++bn)
#pragma unroll
        for (int bm = 0; bm < 4; ++bm)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t n = n0 + wn * 64 + bn * 16 + 4 * lk + r;
                C[m0 + wm * 64 + bm * 16 + li + M * n] = float2{acc_re[bn][bm][r], acc_im[bn][bm][r]};
            }
}

// Largest |re|, |im| of a complex64 tensor in two launches and no atomics: each
// workgroup of k_absmax_c64 writes the maximum of its grid-stride share to parts[];
// every workgroup of k_rescale_c64 reduces the (at most kAbsParts) partial maxima
// itself, then scales its share by the power of two that brings the maximum into
// [0.5, 1).
constexpr int kAbsParts = 1024;

__device__ __forceinline__ float block_max(float m, float* lds) {
    for (int d = 32; d >= 1; d >>= 1) m = fmaxf(m, __shfl_down(m, d, 64));
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = m;
    __syncthreads();
    m = lds[0];
    for (int w = 1; w < kThreads / 64; ++w) m = fmaxf(m, lds[w]);
    return m;
}

__global__ __launch_bounds__(kThreads) void k_absmax_c64(const float2* __restrict__ x, int64_t n,
                                                         float* __restrict__ parts) {
    __shared__ float lds[kThreads / 64];
    float m = 0.0f;
    const int64_t stride = int64_t(gridDim.x) * blockDim.x;
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
        m = fmaxf(m, fmaxf(fabsf(x[i].x), fabsf(x[i].y)));
    m = block_max(m, lds);
    if (threadIdx.x == 0) parts[blockIdx.x] = m;
}

__global__ __launch_bounds__(kThreads) void k_rescale_c64(float2* __restrict__ x, int64_t n,
                                                          const float* __restrict__ parts, int n_parts,
                                                          const int32_t* __restrict__ ea,
                                                          const int32_t* __restrict__ eb, int32_t* __restrict__ ec) {
    __shared__ float lds[kThreads / 64];
    float m = 0.0f;
    for (int j = threadIdx.x; j < n_parts; j += kThreads) m = fmaxf(m, parts[j]);
    m = block_max(m, lds);
    int e = 0;
    if (m > 0.0f && isfinite(m)) (void)frexpf(m, &e);  // m = f 2^e, f in [0.5, 1)
    const float s = ldexpf(1.0f, -e);                 // exact power of two
    const int64_t stride = int64_t(gridDim.x) * blockDim.x;
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
        x[i] = float2{x[i].x * s, x[i].y * s};
    if (blockIdx.x == 0 && threadIdx.x == 0) *ec = (ea ? *ea : 0) + (eb ? *eb : 0) + e;
}

// tensors of up to kRescaleSmall elements: the maximum, the scale and the exponent in
// one single-workgroup launch
constexpr int64_t kRescaleSmall = 1 << 14;
__global__ __launch_bounds__(kThreads) void k_rescale_small_c64(float2* __restrict__ x, int64_t n,
                                                                const int32_t* __restrict__ ea,
                                                                const int32_t* __restrict__ eb,
                                                                int32_t* __restrict__ ec) {
    __shared__ float part[kThreads / 64];
    float m = 0.0f;
    for (int64_t i = threadIdx.x; i < n; i += kThreads) m = fmaxf(m, fmaxf(fabsf(x[i].x), fabsf(x[i].y)));
    for (int d = 32; d >= 1; d >>= 1) m = fmaxf(m, __shfl_down(m, d, 64));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    m = part[0];
    for (int w = 1; w < kThreads / 64; ++w) m = fmaxf(m, part[w]);
    int e = 0;
    if (m > 0.0f && isfinite(m)) (void)frexpf(m, &e);
    const float s = ldexpf(1.0f, -e);
    for (int64_t i = threadIdx.x; i < n; i += kThreads) x[i] = float2{x[i].x * s, x[i].y * s};
    if (threadIdx.x == 0) *ec = (ea ? *ea : 0) + (eb ? *eb : 0) + e;
}


template <class V>
__global__ void k_accumulate(const V* __restrict__ t, const int32_t* __restrict__ e, double2* __restrict__ acc) {
    const int x = e ? *e : 0;
    const double2 a = *acc;
    *acc = double2{a.x + ldexp(double(t->x), x), a.y + ldexp(double(t->y), x)};
}

}  // namespace

qt_status accumulate_scalar(Ctx* c, const Tensor* t, Tensor* acc) {
    const int32_t* e = t->exp_slot >= 0 ? c->d_exp + t->exp_slot : nullptr;
    if (t->dtype == QT_DTYPE_C128)
        hipLaunchKernelGGL(k_accumulate<double2>, dim3(1), dim3(1), 0, c->stream,
                           static_cast<const double2*>(t->data), e, static_cast<double2*>(acc->data));
    else
        hipLaunchKernelGGL(k_accumulate<float2>, dim3(1), dim3(1), 0, c->stream, static_cast<const float2*>(t->data),
                           e, static_cast<double2*>(acc->data));
    return check_hip(c, hipGetLastError(), "k_accumulate");
}

// The device exponent table (first use) and a slot of it for C.
qt_status acquire_exponent(Ctx* c, Tensor* C) {
    if (!c->d_exp) {
        c->exp_cap = 1 << 20;
        qt_status s = check_hip(c, hipMalloc(reinterpret_cast<void**>(&c->d_exp), size_t(c->exp_cap) * 4), "exponents");
        if (s == QT_OK)
            s = check_hip(c, hipMalloc(reinterpret_cast<void**>(&c->d_absmax), kAbsParts * sizeof(float)), "absmax");
        if (s != QT_OK) return s;
        for (int32_t i = c->exp_cap - 1; i >= 0; --i) c->exp_free.push_back(i);
    }
    if (C->exp_slot < 0) {
        if (c->exp_free.empty()) return set_error(c, QT_OOM, "rescale: exponent slots exhausted");
        C->exp_slot = c->exp_free.back();
        c->exp_free.pop_back();
    }
    return QT_OK;
}

namespace {

__global__ void k_carry_exponent(const int32_t* __restrict__ ea, const int32_t* __restrict__ eb,
                                 int32_t* __restrict__ ec) {
    *ec = (ea ? *ea : 0) + (eb ? *eb : 0);
}

}  // namespace

qt_status carry_exponent(Ctx* c, const Tensor* A, const Tensor* B, Tensor* C) {
    if (A->exp_slot < 0 && B->exp_slot < 0) {
        release_exponent(c, C);  // C holds plain values
        return QT_OK;
    }
    qt_status s = acquire_exponent(c, C);
    if (s != QT_OK) return s;
    const int32_t* ea = A->exp_slot >= 0 ? c->d_exp + A->exp_slot : nullptr;
    const int32_t* eb = B->exp_slot >= 0 ? c->d_exp + B->exp_slot : nullptr;
    hipLaunchKernelGGL(k_carry_exponent, dim3(1), dim3(1), 0, c->stream, ea, eb, c->d_exp + C->exp_slot);
    return check_hip(c, hipGetLastError(), "k_carry_exponent");
}

qt_status rescale_c64(Ctx* c, const Tensor* A, const Tensor* B, Tensor* C) {
    qt_status st = acquire_exponent(c, C);
    if (st != QT_OK) return st;
    const int64_t n = C->numel;
    float2* x = static_cast<float2*>(C->data);
    const int32_t* ea = A->exp_slot >= 0 ? c->d_exp + A->exp_slot : nullptr;
    const int32_t* eb = B->exp_slot >= 0 ? c->d_exp + B->exp_slot : nullptr;
    if (n <= kRescaleSmall) {
        hipLaunchKernelGGL(k_rescale_small_c64, dim3(1), dim3(kThreads), 0, c->stream, x, n, ea, eb,
                           c->d_exp + C->exp_slot);
        return check_hip(c, hipGetLastError(), "k_rescale_small_c64");
    }
    const unsigned parts = grid_for(n, kThreads, kAbsParts);
    hipLaunchKernelGGL(k_absmax_c64, dim3(parts), dim3(kThreads), 0, c->stream, x, n, c->d_absmax);
    hipLaunchKernelGGL(k_rescale_c64, dim3(grid_for(n, kThreads, 4096)), dim3(kThreads), 0, c->stream, x, n,
                       c->d_absmax, int(parts), ea, eb, c->d_exp + C->exp_slot);
    return check_hip(c, hipGetLastError(), "k_rescale_c64");
}

qt_status read_exponent(Ctx* c, const Tensor* t, int32_t* e) {
    *e = 0;
    if (t->exp_slot < 0) return QT_OK;
    qt_status s = check_hip(c, hipStreamSynchronize(c->stream), "sync");
    if (s != QT_OK) return s;
    return check_hip(c, hipMemcpy(e, c->d_exp + t->exp_slot, 4, hipMemcpyDeviceToHost), "exponent");
}

void release_exponent(Ctx* c, Tensor* t) {
    if (t->exp_slot >= 0) c->exp_free.push_back(t->exp_slot);
    t->exp_slot = -1;
}

qt_status launch_fill_zero(Ctx* c, void* p, size_t bytes) {
    const int64_t n16 = int64_t((bytes + 15) / 16);  // pool blocks are >= 256 B, 16 B aligned
    hipLaunchKernelGGL(k_fill_zero, dim3(grid_for(n16, 256, 8192)), dim3(256), 0, c->stream,
                       static_cast<uint4*>(p), n16);
    return check_hip(c, hipGetLastError(), "k_fill_zero");
}

namespace {

// Large steps: permute into GEMM layout (skipped when already there), MFMA GEMM.
template <class V, int MODE>
qt_status run_gemm(Ctx* c, const Tensor* A, const Tensor* B, Tensor* C, const BitMap& m, int mbits,
                   const Workspace* ws) {
    // operand permutes: tiles of up to 2^12 elements (64 KB of LDS in complex128)
    constexpr int kPermTileBits = 12;
    const int nbits_n = m.nbits_c - mbits;
    const int sb = m.nbits_s;
    int src_a[64], src_b[64];
    for (int j = 0; j < mbits; ++j) src_a[j] = m.c_src[j];
    for (int j = 0; j < sb; ++j) src_a[mbits + j] = m.s_a[j];
    for (int j = 0; j < nbits_n; ++j) src_b[j] = m.c_src[mbits + j] - 64;
    for (int j = 0; j < sb; ++j) src_b[nbits_n + j] = m.s_b[j];
    const V* ap = static_cast<const V*>(A->data);
    const V* bp = static_cast<const V*>(B->data);
    void* abuf = nullptr;
    void* bbuf = nullptr;
    bool perm_a = !is_identity(src_a, mbits + sb), perm_b = !is_identity(src_b, nbits_n + sb);
    // bf16x3 with whole 128 x 128 x 32 tiles: the permutes write bf16 planes, the lowest
    // three summed bits first (k_gemm_bf16x3).  Each operand then needs scratch of its own
    // size, also one that is in place, so not with a caller's workspace, and where there is
    // no room for both, k_gemm_c64 takes the operands as they are.  An operand in place
    // pays a pass over it for the planes, so there the product has to be large.  us without
    // and with planes (2^m x 2^n over 2^k):
    //   both in place, below 2^30 MACs:  7,7,5 5.3, 15.0;  9,9,8 24, 34;  11,11,7 32, 35
    //   from there:                      10,10,10 84, 60;  13,13,5 181, 147
    //   one in place, 2^8 or more terms: 7,7,8 37, 32;     10,10,9 55, 47 (7,7,5 10.3, 14.8;
    //     10,10,6 17, 21); 32 times the other operand: 12,7,10 50, 54
    //   both permuted:                   7,7,5 14.3, 14.9; 8,8,10 52, 39; 10,10,12 320, 147
    const bool one_permuted = perm_a != perm_b;
    const int excess = perm_a ? nbits_n - mbits : mbits - nbits_n;  // of the one in place, in bits
    bool planes = MODE == MODE_BF16X3 && !ws && mbits >= 7 && nbits_n >= 7 && sb >= 5 &&
                  ((perm_a && perm_b) || m.nbits_c + sb >= 30 || (one_permuted && sb >= 8 && excess <= 3));
    if (planes) {
        hipError_t e = hipSuccess;
        abuf = c->pool.alloc(A->bytes, &e);
        if (abuf) bbuf = c->pool.alloc(B->bytes, &e);
        if (!bbuf) {
            c->pool.release(abuf);
            abuf = nullptr;
            planes = false;
        }
    }
    if (planes) {
        auto lowest_first = [&](int* src, int free_bits, const uint8_t* sum) {
            for (int j = free_bits - 1; j >= 0; --j) src[j + 3] = src[j];
            for (int j = 0; j < 3; ++j) src[j] = sum[j];
        };
        lowest_first(src_a, mbits, m.s_a);
        lowest_first(src_b, nbits_n, m.s_b);
        perm_a = perm_b = true;
    }
    auto rewrite = [&](const Tensor* t, void* out, int nbits, const int* src) {
        const PermPlan p = make_perm_plan(nbits, src, kPermTileBits);
        if constexpr (MODE == MODE_BF16X3)
            if (planes) return run_permute_split(c, static_cast<const float2*>(t->data), out, p);
        return permute(c, t->data, out, t->dtype, p);
    };
    // a workspace holds A's permute at its start and B's after it (256-byte aligned)
    const size_t ws_b = perm_a ? (A->bytes + 255) / 256 * 256 : 0;
    if (ws && ws_b + (perm_b ? B->bytes : 0) > ws->bytes)
        return set_error(c, QT_INVALID_INPUT, "gemm: operand permutes exceed the workspace");
    qt_status s = QT_OK;
    if (perm_a) {
        hipError_t e = hipSuccess;
        if (!abuf) abuf = ws ? static_cast<void*>(ws->base) : c->pool.alloc(A->bytes, &e);
        if (!abuf) return check_hip(c, e, "gemm scratch A");
        s = rewrite(A, abuf, mbits + sb, src_a);
        ap = static_cast<const V*>(abuf);
    }
    if (s == QT_OK && perm_b) {
        hipError_t e = hipSuccess;
        if (!bbuf) bbuf = ws ? static_cast<void*>(ws->base + ws_b) : c->pool.alloc(B->bytes, &e);
        if (!bbuf) {
            if (!ws) c->pool.release(abuf);
            return check_hip(c, e, "gemm scratch B");
        }
        s = rewrite(B, bbuf, nbits_n + sb, src_b);
        bp = static_cast<const V*>(bbuf);
    }
    if (s == QT_OK) {
        const int64_t M = int64_t(1) << mbits, N = int64_t(1) << nbits_n, K = int64_t(1) << sb;
        const int64_t tiles = (M / GM) * (N / GN);
        const unsigned gx = unsigned(tiles < 65536 ? tiles : 65536);
        const unsigned gy = unsigned((tiles + gx - 1) / gx);
        if constexpr (MODE == MODE_PLAIN) {
            // as for complex64 below: fewer than 512 tiles (64 x 64 here) split K
            int S = 1;
            if (!ws && K % GK == 0)
                while (tiles * S < 512 && K / (2 * S) >= kSplitRows && S < 64) S *= 2;
            double2* part = nullptr;
            if (S > 1) {
                hipError_t e = hipSuccess;
                part = static_cast<double2*>(c->pool.alloc(size_t(S) * size_t(M * N) * sizeof(double2), &e));
                if (!part) {
                    (void)hipGetLastError();  // no room: one product, unsplit
                    S = 1;
                }
            }
            double2* out = S > 1 ? part : static_cast<double2*>(C->data);
            hipLaunchKernelGGL(k_gemm_c128, dim3(gx, gy, unsigned(S)), dim3(kThreads), 0, c->stream, ap, bp, out, M,
                               N, K / S);
            s = check_hip(c, hipGetLastError(), "k_gemm_c128");
            if (S > 1) {
                const int64_t n = M * N;
                if (s == QT_OK) {
                    hipLaunchKernelGGL(k_sum_splits_c128, dim3(unsigned((n + kThreads - 1) / kThreads)), dim3(kThreads),
                                       0, c->stream, part, static_cast<double2*>(C->data), n, S);
                    s = check_hip(c, hipGetLastError(), "k_sum_splits_c128");
                }
                c->pool.release(part);
            }
        } else {
            bool done = false;
            if ((MODE == MODE_BF16X3 ? planes : K % BK == 0) && M >= BT && N >= BT) {
                const int64_t big = (M / BT) * (N / BT);
                const unsigned bx = unsigned(big < 65536 ? big : 65536);
                const unsigned by = unsigned((big + bx - 1) / bx);
                // fewer output tiles than two per CU: split K (at least kSplitRows
                // summed rows per split) into S partial products, then add them in
                // order; not with a caller's workspace, which holds no room for them
                int S = 1;
                if (!ws)
                    while (big * S < 512 && K / (2 * S) >= kSplitRows && S < 64) S *= 2;
                float2* part = nullptr;
                if (S > 1) {
                    hipError_t e = hipSuccess;
                    part = static_cast<float2*>(c->pool.alloc(size_t(S) * size_t(M * N) * sizeof(float2), &e));
                    if (!part) {
                        (void)hipGetLastError();  // no room: one product, unsplit
                        S = 1;
                    }
                }
                float2* out = S > 1 ? part : static_cast<float2*>(C->data);
                if constexpr (MODE == MODE_BF16X3)
                    hipLaunchKernelGGL(k_gemm_bf16x3, dim3(bx, by, unsigned(S)), dim3(kThreads), 0, c->stream,
                                       reinterpret_cast<const uint4*>(ap), reinterpret_cast<const uint4*>(bp), out, M,
                                       N, K / S, K);
                else
                    hipLaunchKernelGGL((k_gemm_c64_big<MODE>), dim3(bx, by, unsigned(S)), dim3(kThreads), 0, c->stream,
                                       ap, bp, out, M, N, K / S);
                s = check_hip(c, hipGetLastError(), "k_gemm_c64_big");
                if (S > 1) {
                    const int64_t n4 = M * N / 2;
                    if (s == QT_OK) {
                        hipLaunchKernelGGL(k_sum_splits, dim3(unsigned((n4 + kThreads - 1) / kThreads)),
                                           dim3(kThreads), 0, c->stream, reinterpret_cast<const float4*>(part),
                                           reinterpret_cast<float4*>(C->data), n4, S);
                        s = check_hip(c, hipGetLastError(), "k_sum_splits");
                    }
                    c->pool.release(part);
                }
                done = true;
            }
            if (!done) {
                // fewer than 512 tiles (64 x 64 here): split K as above
                int S = 1;
                if (!ws && K % HK == 0)
                    while (tiles * S < 512 && K / (2 * S) >= kSplitRows && S < 64) S *= 2;
                float2* part = nullptr;
                if (S > 1) {
                    hipError_t e = hipSuccess;
                    part = static_cast<float2*>(c->pool.alloc(size_t(S) * size_t(M * N) * sizeof(float2), &e));
                    if (!part) {
                        (void)hipGetLastError();  // no room: one product, unsplit
                        S = 1;
                    }
                }
                float2* out = S > 1 ? part : static_cast<float2*>(C->data);
                hipLaunchKernelGGL((k_gemm_c64<MODE>), dim3(gx, gy, unsigned(S)), dim3(kThreads), 0, c->stream, ap, bp,
                                   out, M, N, K / S);
                s = check_hip(c, hipGetLastError(), "k_gemm_c64");
                if (S > 1) {
                    const int64_t n4 = M * N / 2;
                    if (s == QT_OK) {
                        hipLaunchKernelGGL(k_sum_splits, dim3(unsigned((n4 + kThreads - 1) / kThreads)), dim3(kThreads),
                                           0, c->stream, reinterpret_cast<const float4*>(part),
                                           reinterpret_cast<float4*>(C->data), n4, S);
                        s = check_hip(c, hipGetLastError(), "k_sum_splits");
                    }
                    c->pool.release(part);
                }
            }
        }
    }
    // stream-ordered reuse: later work on this stream may take these blocks
    if (!ws) {
        c->pool.release(abuf);
        c->pool.release(bbuf);
    }
    return s;
}

// a split C (A's free bits low, B's high) with at most 5 bits on one side and at
// least 10 on the other
inline bool skinny_shape(const BitMap& m, bool split, int mbits) {
    const int nbits_n = m.nbits_c - mbits;
    return split && std::min(mbits, nbits_n) <= 5 && std::max(mbits, nbits_n) >= 10;
}

// Sums long enough to be split over a workgroup's lanes, into few outputs: from 2^9 summed
// indices up to 2^11 outputs, from 2^11 up to 2^16.  k_direct and k_skinny run one lane
// per output (or per 2 to 32 outputs), which leaves most of the chip idle there: 2^12
// outputs over 2^12 summed indices (a state projected on 12 qubits, complex64) took
// 1,244 us on k_skinny, 2^7 over 2^15 (complex128) 389 us on k_direct; here about 50 and
// 20 us.  At the corners, shuffled axes, us before and here (complex128; complex64 4M):
// one output over 2^9 31, 8.4 (21, 7.4); 2^11 over 2^9 75, 6.3 (75, 9.3); one over 2^11 116,
// 7.4 (80, 7.4); 2^16 over 2^11 2,260, 84 (1,356, 43); none of 484 shapes and forms was slower.
// With a caller's workspace only the sums that have always split (2^6 outputs, 2^13 terms)
// do: the others need no scratch on k_direct and k_skinny, and calls that share the
// workspace may overlap there.
inline bool reduce_shape(const BitMap& m, const Workspace* ws) {
    if (ws) return m.nbits_s >= 13 && m.nbits_c <= 6;
    return (m.nbits_s >= 11 && m.nbits_c <= 16) || (m.nbits_s >= 9 && m.nbits_c <= 11);
}

template <class V, int MODE>
qt_status dispatch_small(Ctx* c, const Tensor* A, const Tensor* B, Tensor* C, const BitMap& m, bool split,
                         int mbits, const Workspace* ws) {
    const V* a = static_cast<const V*>(A->data);
    const V* b = static_cast<const V*>(B->data);
    V* cc = static_cast<V*>(C->data);
    if (reduce_shape(m, ws)) {
        bool no_room = false;  // then as sums too short to split, which need no scratch
        const qt_status s = run_reduce<V, MODE>(c, a, b, cc, m, ws, &no_room);
        if (!no_room) return s;
    }
    if (skinny_shape(m, split, mbits)) return run_skinny<V, MODE>(c, a, b, cc, m, mbits);
    return run_direct<V, MODE>(c, a, b, cc, m);
}

}  // namespace

qt_status contract_pair(Ctx* c, const Tensor* A, const Tensor* B, Tensor* C, const BitMap& m,
                        int precision, const Workspace* ws) {
    // GEMM shape: C's low bits all from A, high bits all from B
    int mbits = 0;
    while (mbits < m.nbits_c && m.c_src[mbits] < 64) ++mbits;
    bool split = true;
    for (int i = mbits; i < m.nbits_c; ++i)
        if (m.c_src[i] < 64) split = false;
    const int nbits_n = m.nbits_c - mbits;
    const bool gemm = split && mbits >= 6 && nbits_n >= 6;
    // short summed extents (8, or 16 in complex64: below a k-tile) take the GEMM, with
    // the last k-tile zero-filled, when the output is large: k_direct would re-read
    // the operands once per output element of the other side (measured: from 2^16
    // outputs in complex64, from 2^24 in complex128)
    if (A->dtype == QT_DTYPE_C128) {
        const bool short_k = m.nbits_s >= 3 && m.nbits_c >= 24;
        if (gemm && (m.nbits_s >= 4 || short_k)) return run_gemm<double2, MODE_PLAIN>(c, A, B, C, m, mbits, ws);
        return dispatch_small<double2, MODE_PLAIN>(c, A, B, C, m, split, mbits, ws);
    }
    const bool short_k = m.nbits_s >= 3 && m.nbits_c >= 16;
    const bool gemm64 = gemm && (m.nbits_s >= 5 || short_k);  // k-tiles of 32
    switch (precision) {
        case QT_C64_4M:
            return gemm64 ? run_gemm<float2, MODE_4M>(c, A, B, C, m, mbits, ws)
                          : dispatch_small<float2, MODE_4M>(c, A, B, C, m, split, mbits, ws);
        case QT_C64_3M:
            return gemm64 ? run_gemm<float2, MODE_3M>(c, A, B, C, m, mbits, ws)
                          : dispatch_small<float2, MODE_3M>(c, A, B, C, m, split, mbits, ws);
        default:
            return gemm64 ? run_gemm<float2, MODE_BF16X3>(c, A, B, C, m, mbits, ws)
                          : dispatch_small<float2, MODE_BF16X3>(c, A, B, C, m, split, mbits, ws);
    }
}

}  // namespace qt
