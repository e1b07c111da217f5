// Chains of thin contraction steps in one pass over the large tensor (libqtorch_hip.so).
//
// A circuit sweep contracts one growing tensor with a small tensor at a time: each step
// sums one or two index bits of it and adds up to two.  Step by step (k_thin) every step
// reads and writes the whole tensor.  k_chain takes several consecutive steps: a workgroup
// loads a tile of the tensor into LDS, namely every value of the bits that the steps sum
// and of the lowest bits (whole cache lines), runs the steps on it there, and writes the
// result's tile.  Each step does k_thin's arithmetic in its order, so the results have
// the bits that the steps one by one give.
//
// Rescaled passes keep their range between the steps: a tile whose largest value leaves
// [2^-16, 2^16] is scaled by a power of two in LDS (k_chain), and k_chain_scale brings
// the tiles to the result's one exponent afterwards.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "qt_internal.h"
#include "qt_mac.h"

namespace qt {

namespace {

constexpr int kMaxLinks = 8;     // steps of one pass
constexpr int kThreadBits = 8;  // two workgroups a CU (LDS); 512 threads measured 4 %, 1,024 35 % slower
constexpr int kChainThreads = 1 << kThreadBits;
constexpr int kMaxTileBits = 12; // complex64; one less in complex128 (two buffers of 32 KB)

struct ChainStep {
    int32_t ns, nb;       // summed bits (1 or 2) and added bits (0 to 2)
    int32_t lb;           // tile bits before the step
    int32_t adj;          // the summed bit at tile position 0, or -1
    int32_t ins[2];       // tile positions of the summed bits, ascending
    int32_t off[4];       // tile offset of summed index j
    int32_t g_small[4];   // small operand offset of summed index j
    int32_t g_free[4];    // small operand offset of its free part o
};

// Tile bits are the tensor's bits in increasing position; each step takes its summed bits
// away and adds the new ones on top, as in the step's result.
struct ChainPlan {
    int32_t n_steps, tb_in, tb_out, n_rest;
    int32_t in_pos[kMaxTileBits], out_pos[kMaxTileBits];
    int32_t rest_in[48], rest_out[48];
    ChainStep step[kMaxLinks];
};

struct ChainArgs {
    ChainPlan p;
    const void* g[kMaxLinks];
};

// Two neighbouring elements of a tile: 16-byte LDS accesses in complex64.
template <class V>
struct alignas(16) Pair {
    V a, b;
};

// Largest |re|, |im| so far; infinite once a value is, NaN passed over.
template <class V>
__device__ __forceinline__ void grow_max(float& m, V v) {
    m = fmaxf(m, fmaxf(fabsf(float(v.x)), fabsf(float(v.y))));
}

// Largest over the workgroup (lds: one float per wave).
__device__ __forceinline__ float tile_max(float m, float* lds) {
    for (int d = 32; d >= 1; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = m;
    __syncthreads();
    m = lds[0];
    for (int w = 1; w < kChainThreads / 64; ++w) m = fmaxf(m, lds[w]);
    return m;
}

// The same over the finite values of a tile.
__device__ __forceinline__ float tile_max_finite(const float2* t, int n, float* lds) {
    float m = 0.0f;
    for (int i = threadIdx.x; i < n; i += kChainThreads) {
        const float x = fabsf(t[i].x), y = fabsf(t[i].y);
        if (x < INFINITY) m = fmaxf(m, x);
        if (y < INFINITY) m = fmaxf(m, y);
    }
    return tile_max(m, lds);
}

// A thread makes the outputs of two neighbouring free parts t.  ADJ: the summed bit (0 or 1
// of the summed index) at tile position 0, whose two values are neighbours, or -1: then the
// two t are.
// SCALED: m grows to the outputs' largest |re|, |im|.
template <class V, int MODE, bool SCALED, int NS, int NB, int ADJ>
__device__ __forceinline__ void chain_step(const V* in, V* out, const V* gl, const ChainStep& s, int tid, float& m) {
    constexpr int NJ = 1 << NS, NO = 1 << NB;
    V g[NO][NJ];
#pragma unroll
    for (int o = 0; o < NO; ++o)
#pragma unroll
        for (int j = 0; j < NJ; ++j) g[o][j] = gl[o * 4 + j];
    const int nf = 1 << (s.lb - NS);
    const int lo0 = (1 << s.ins[0]) - 1, lo1 = (1 << s.ins[1]) - 1;
    auto expand = [&](int t) {
        int x = ((t & ~lo0) << 1) | (t & lo0);
        if constexpr (NS == 2) x = ((x & ~lo1) << 1) | (x & lo1);
        return x;
    };
    auto pair = [&](int x) { return *reinterpret_cast<const Pair<V>*>(in + x); };
    for (int t = 2 * tid; t < nf; t += 2 * kChainThreads) {
        V xs[2][NJ];
        if constexpr (ADJ >= 0) {
            constexpr int kAdj = 1 << ADJ, kOther = kAdj == 1 ? 2 : 1;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int x = expand(t + h);
                const Pair<V> v = pair(x);
                xs[h][0] = v.a;
                xs[h][kAdj] = v.b;
                if constexpr (NS == 2) {
                    const Pair<V> w = pair(x + s.off[kOther]);
                    xs[h][kOther] = w.a;
                    xs[h][3] = w.b;
                }
            }
        } else {
            const int x = expand(t);
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const Pair<V> v = pair(x + s.off[j]);
                xs[0][j] = v.a;
                xs[1][j] = v.b;
            }
        }
        Acc<V, MODE> acc[2][NO];
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int o = 0; o < NO; ++o) mac<V, MODE>(acc[h][o], xs[h][j], g[o][j]);
#pragma unroll
        for (int o = 0; o < NO; ++o) {
            const Pair<V> v{finish<V, MODE>(acc[0][o]), finish<V, MODE>(acc[1][o])};
            if constexpr (SCALED) {
                grow_max(m, v.a);
                grow_max(m, v.b);
            }
            *reinterpret_cast<Pair<V>*>(out + t + o * nf) = v;
        }
    }
}

template <class V, int MODE, bool SCALED, int NS, int ADJ>
__device__ __forceinline__ void chain_step_nb(const V* in, V* out, const V* gl, const ChainStep& s, int tid,
                                              float& m) {
    if (s.nb == 0) chain_step<V, MODE, SCALED, NS, 0, ADJ>(in, out, gl, s, tid, m);
    else if (s.nb == 1) chain_step<V, MODE, SCALED, NS, 1, ADJ>(in, out, gl, s, tid, m);
    else chain_step<V, MODE, SCALED, NS, 2, ADJ>(in, out, gl, s, tid, m);
}

// Exponents of a rescaled pass's tiles: the stored values times 2^scale are the tile's, the
// largest of which lies in [2^(top - 1), 2^top) (kNoTop: no nonzero finite value).
struct TileExp {
    int32_t scale, top;
};
constexpr int kNoTop = INT32_MIN;

// A pass reads and writes the tensor once in HBM, and each step once in LDS: at 8 steps
// the two and the multiply-adds take about as long as each other, and two workgroups a CU
// overlap them in part.  The 48-qubit depth-14 sweep (456 steps on tensors of up to 2^29
// complex64, 1,517 GB step by step, 181 GB in passes): 271.7 ms with k_thin, 99.6 ms;
// complex128 544 and 225 ms.  Tiles of 2^11 (four workgroups a CU, shorter passes): 103.8
// and 292 ms.
// SCALED: complex64 values may not leave FP32's range between the steps, so a tile whose
// largest |re|, |im| a step leaves outside [2^-16, 2^16] is scaled by the power of two that
// brings it into [0.5, 1) (exact; the test is one maximum a value and two ballots a wave, and
// a tile of gate-sized values never scales).  Step by step every result is scaled, so the
// values are the same.
template <class V, int MODE, bool SCALED>
__global__ __launch_bounds__(kChainThreads) void k_chain(const V* __restrict__ X, V* __restrict__ C, ChainArgs a,
                                                         TileExp* __restrict__ tile_exp) {
    static_assert(!SCALED || sizeof(V) == 8, "complex64 values are rescaled");
    constexpr int kTile = (8 << kMaxTileBits) / int(sizeof(V));
    const ChainPlan& p = a.p;
    __shared__ V gl[kMaxLinks][16];
    __shared__ __align__(16) V tiles[2][kTile];
    V *buf = tiles[0], *alt = tiles[1];
    const int tid = threadIdx.x;
    if (tid < p.n_steps * 16) {
        const ChainStep& s = p.step[tid >> 4];
        const int o = (tid >> 2) & 3, j = tid & 3;
        if (o < (1 << s.nb) && j < (1 << s.ns))
            gl[tid >> 4][tid & 15] = static_cast<const V*>(a.g[tid >> 4])[s.g_free[o] + s.g_small[j]];
    }
    const int64_t id = int64_t(blockIdx.x) + int64_t(blockIdx.y) * gridDim.x;
    int64_t base_in = 0, base_out = 0;
    for (int i = 0; i < p.n_rest; ++i)
        if ((id >> i) & 1) {
            base_in += int64_t(1) << p.rest_in[i];
            base_out += int64_t(1) << p.rest_out[i];
        }
    // 16 bytes per access: P low bits of a tile index are one load's or store's elements
    // (positions 0 to P - 1 are in the tile on both sides).  Thread bits, then up to
    // 4 step bits, whose offsets are read before the first load
    constexpr int P = sizeof(V) == 8 ? 1 : 0, hi = kThreadBits + P, kStepBits = 4;
    struct alignas(16) Pack {
        V v[1 << P];
    };
    {
        int64_t off_t = base_in, off_s[kStepBits];
        for (int b = P; b < hi && b < p.tb_in; ++b)
            if ((tid >> (b - P)) & 1) off_t += int64_t(1) << p.in_pos[b];
#pragma unroll
        for (int k = 0; k < kStepBits; ++k) off_s[k] = hi + k < p.tb_in ? int64_t(1) << p.in_pos[hi + k] : 0;
        const int n = 1 << p.tb_in;
        if ((tid << P) < n)
#pragma unroll 4
            for (int q = 0; (q << hi) < n; ++q) {
                int64_t off = off_t;
#pragma unroll
                for (int k = 0; k < kStepBits; ++k)
                    if ((q >> k) & 1) off += off_s[k];
                *reinterpret_cast<Pack*>(buf + (tid << P) + (q << hi)) = *reinterpret_cast<const Pack*>(X + off);
            }
    }
    __syncthreads();
    __shared__ int wave_range[2][kChainThreads / 64];  // of the step before and this one
    __shared__ float wave_max[kChainThreads / 64];
    float m = 0.0f;
    int scale = 0;
    bool empty = false;  // no nonzero finite value left: nothing to scale from here on
    for (int i = 0; i < p.n_steps; ++i) {
        const ChainStep& s = p.step[i];
        m = 0.0f;
        switch (s.ns * 4 + s.adj) {
            case 3: chain_step_nb<V, MODE, SCALED, 1, -1>(buf, alt, gl[i], s, tid, m); break;
            case 4: chain_step_nb<V, MODE, SCALED, 1, 0>(buf, alt, gl[i], s, tid, m); break;
            case 7: chain_step_nb<V, MODE, SCALED, 2, -1>(buf, alt, gl[i], s, tid, m); break;
            case 8: chain_step_nb<V, MODE, SCALED, 2, 0>(buf, alt, gl[i], s, tid, m); break;
            default: chain_step_nb<V, MODE, SCALED, 2, 1>(buf, alt, gl[i], s, tid, m); break;
        }
        V* const t = buf;
        buf = alt;
        alt = t;
        if constexpr (SCALED) {
            const int r = (__any(m >= 0x1p-16f) ? 1 : 0) | (__any(m > 0x1p16f) ? 2 : 0);
            if ((tid & 63) == 0) wave_range[i & 1][tid >> 6] = r;
        }
        __syncthreads();
        if constexpr (SCALED) {
            int r = 0;
            for (int w = 0; w < kChainThreads / 64; ++w) r |= wave_range[i & 1][w];
            if (r != 1 && !empty) {  // the same in every thread
                const int n = 1 << (s.lb - s.ns + s.nb);
                const float top = tile_max_finite(buf, n, wave_max);
                int e = 0;
                empty = top == 0.0f;
                if (!empty) (void)frexpf(top, &e);
                scale += e;
                for (int k = tid; k < n && e != 0; k += kChainThreads)
                    buf[k] = V{ldexpf(buf[k].x, -e), ldexpf(buf[k].y, -e)};
                m = ldexpf(m, -e);
                __syncthreads();
            }
        }
    }
    if constexpr (SCALED) {
        float top = tile_max(m, wave_max);  // of the last step's values
        if (!(top < INFINITY)) {
            __syncthreads();
            top = tile_max_finite(buf, 1 << p.tb_out, wave_max);
        }
        int e = 0;
        (void)frexpf(top, &e);
        if (tid == 0) tile_exp[id] = TileExp{scale, top > 0.0f ? scale + e : kNoTop};
    }
    int64_t off_t = base_out, off_s[kStepBits];
    for (int b = P; b < hi && b < p.tb_out; ++b)
        if ((tid >> (b - P)) & 1) off_t += int64_t(1) << p.out_pos[b];
#pragma unroll
    for (int k = 0; k < kStepBits; ++k) off_s[k] = hi + k < p.tb_out ? int64_t(1) << p.out_pos[hi + k] : 0;
    const int n = 1 << p.tb_out;
    if ((tid << P) < n)
#pragma unroll 4
        for (int q = 0; (q << hi) < n; ++q) {
            int64_t off = off_t;
#pragma unroll
            for (int k = 0; k < kStepBits; ++k)
                if ((q >> k) & 1) off += off_s[k];
            *reinterpret_cast<Pack*>(C + off) = *reinterpret_cast<const Pack*>(buf + (tid << P) + (q << hi));
        }
}

// Largest top of a rescaled pass's tiles in one workgroup (0 if no tile has one), and C's
// exponent with X's added.
constexpr int kTopThreads = 1024;
__global__ __launch_bounds__(kTopThreads) void k_chain_top(const TileExp* __restrict__ tile_exp, int64_t n,
                                                           const int32_t* __restrict__ ex, int32_t* __restrict__ ec,
                                                           int32_t* __restrict__ top) {
    __shared__ int wave_top[kTopThreads / 64];
    int t = kNoTop;
    for (int64_t i = threadIdx.x; i < n; i += kTopThreads) t = max(t, tile_exp[i].top);
    for (int d = 32; d >= 1; d >>= 1) t = max(t, __shfl_xor(t, d, 64));
    if ((threadIdx.x & 63) == 0) wave_top[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int w = 1; w < kTopThreads / 64; ++w) t = max(t, wave_top[w]);
    if (t == kNoTop) t = 0;
    *top = t;
    *ec = (ex ? *ex : 0) + t;
}

// The tiles of C brought to the exponent *top: one workgroup a tile, in k_chain's order.
__global__ __launch_bounds__(kChainThreads) void k_chain_scale(float2* __restrict__ C, ChainPlan p,
                                                               const TileExp* __restrict__ tile_exp,
                                                               const int32_t* __restrict__ top) {
    const int64_t id = int64_t(blockIdx.x) + int64_t(blockIdx.y) * gridDim.x;
    const int e = tile_exp[id].scale - *top;
    if (e == 0) return;
    int64_t off_t = 0;
    for (int i = 0; i < p.n_rest; ++i)
        if ((id >> i) & 1) off_t += int64_t(1) << p.rest_out[i];
    constexpr int hi = kThreadBits + 1;  // two neighbours a thread, then up to 3 step bits
    const int tid = threadIdx.x;
    for (int b = 1; b < hi && b < p.tb_out; ++b)
        if ((tid >> (b - 1)) & 1) off_t += int64_t(1) << p.out_pos[b];
    const int n = 1 << p.tb_out;
    if (2 * tid >= n) return;
    for (int q = 0; (q << hi) < n; ++q) {
        int64_t off = off_t;
        for (int b = hi; b < p.tb_out; ++b)
            if ((q >> (b - hi)) & 1) off += int64_t(1) << p.out_pos[b];
        float4* const at = reinterpret_cast<float4*>(C + off);
        const float4 v = *at;
        *at = make_float4(ldexpf(v.x, e), ldexpf(v.y, e), ldexpf(v.z, e), ldexpf(v.w, e));
    }
}

// The bits of the tensor through the links, in position order: the input position each comes
// from, -1 for a bit that a step added.
struct Bits {
    int n = 0;
    int x[64];  // 40 input bits, and a step adds one at most

    // summed bits (their positions ascending) taken away, `added` new ones on top
    void step(const int* summed, int ns, int added) {
        int m = 0;
        for (int b = 0; b < n; ++b)
            if (b != summed[0] && (ns < 2 || b != summed[1])) x[m++] = x[b];
        for (int b = 0; b < added; ++b) x[m++] = -1;
        n = m;
    }
};

// The plan of the first n links (desc / axes as qt_contract_chain takes them), or false when
// they cannot share a pass.
bool plan_chain(int nx, int dl, bool c128, int n, const int32_t* desc, const int32_t* axes, ChainPlan* out) {
    if (n < 1 || n > kMaxLinks || nx < 1 || nx > 40) return false;
    ChainPlan p;
    std::memset(&p, 0, sizeof p);
    p.n_steps = n;
    Bits bits;
    for (bits.n = 0; bits.n < nx; ++bits.n) bits.x[bits.n] = bits.n;
    bool in_tile[64] = {false};   // input bits of the tile: first those summed in the chain
    int summed[kMaxLinks][2];     // current positions, ascending
    int s_x[kMaxLinks][2];        // the same in the pairs' own order
    const int32_t* ax = axes;
    for (int s = 0; s < n; ++s) {
        const int rg = desc[3 * s], k = desc[3 * s + 1], rc = desc[3 * s + 2];
        if (k < 1 || k > 2 || rg < k || rg > k + 2) return false;
        const int rx = bits.n / dl, kb = k * dl, nb = (rg - k) * dl;
        if (kb > 2 || nb > 2 || k > rx || rc != rx + rg - 2 * k) return false;
        const int32_t *px = ax, *pg = ax + k, *fs = ax + 2 * k;
        ax += 2 * k + rc;
        bool used_x[64] = {false}, used_g[8] = {false};
        ChainStep& st = p.step[s];
        st.ns = kb;
        st.nb = nb;
        // digit j of the summed index belongs to pair k - 1 - j (src/Network.h:912-916)
        int s_g[2] = {0, 0};
        s_x[s][0] = s_x[s][1] = 0;
        for (int i = 0; i < k; ++i) {
            if (px[i] < 0 || px[i] >= rx || pg[i] < 0 || pg[i] >= rg || used_x[px[i]] || used_g[pg[i]]) return false;
            used_x[px[i]] = used_g[pg[i]] = true;
            for (int t = 0; t < dl; ++t) {
                s_x[s][(k - 1 - i) * dl + t] = px[i] * dl + t;
                s_g[(k - 1 - i) * dl + t] = pg[i] * dl + t;
            }
        }
        summed[s][0] = kb == 2 ? std::min(s_x[s][0], s_x[s][1]) : s_x[s][0];
        summed[s][1] = kb == 2 ? std::max(s_x[s][0], s_x[s][1]) : 0;
        for (int j = 0; j < (1 << kb); ++j)
            for (int b = 0; b < kb; ++b)
                if ((j >> b) & 1) st.g_small[j] += 1 << s_g[b];
        // free axes: the tensor's in their order, then the small operand's
        int prev = -1, f = 0;
        for (; f < rc && (fs[f] & QT_FROM_A); ++f) {
            const int axis = fs[f] & ~QT_FROM_A;
            if (axis <= prev || axis >= rx || used_x[axis]) return false;
            prev = axis;
        }
        if (f != rx - k) return false;
        int g_bit[2] = {0, 0}, ng = 0;
        for (; f < rc; ++f) {
            if ((fs[f] & QT_FROM_A) || fs[f] < 0 || fs[f] >= rg || used_g[fs[f]]) return false;
            used_g[fs[f]] = true;
            for (int t = 0; t < dl; ++t) g_bit[ng++] = fs[f] * dl + t;
        }
        for (int o = 0; o < (1 << nb); ++o)
            for (int b = 0; b < nb; ++b)
                if ((o >> b) & 1) st.g_free[o] += 1 << g_bit[b];
        for (int b = 0; b < kb; ++b)
            if (bits.x[summed[s][b]] >= 0) in_tile[bits.x[summed[s][b]]] = true;
        bits.step(summed[s], kb, nb);
    }
    // the tile: the summed input bits, the four lowest bits of the input (three in
    // complex128: 128 bytes) and of the result, then the lowest others up to the size that
    // the largest intermediate allows
    const int line = c128 ? 3 : 4;
    for (int i = 0; i < line && i < nx; ++i) in_tile[i] = true;
    for (int i = 0; i < line && i < bits.n; ++i)
        if (bits.x[i] >= 0) in_tile[bits.x[i]] = true;
    int grow = 0, most = 0;  // the largest excess of an intermediate over the input tile
    for (int s = 0; s < n; ++s) {
        grow += p.step[s].nb - p.step[s].ns;
        most = std::max(most, grow);
    }
    int tb = 0;
    for (int i = 0; i < nx; ++i) tb += in_tile[i];
    // at least 2^8 tiles where the tensor is small, and a tile that fills the workgroup
    const int cap = std::min(c128 ? kMaxTileBits - 1 : kMaxTileBits, std::max(9, nx - 8));
    if (tb + most > cap || tb + grow < 2) return false;
    for (int i = 0; i < nx && tb + most < cap; ++i)
        if (!in_tile[i]) {
            in_tile[i] = true;
            ++tb;
        }
    p.tb_in = tb;
    p.tb_out = tb + grow;
    int k = 0;
    for (int i = 0; i < nx; ++i)
        if (in_tile[i]) p.in_pos[k++] = i;
    k = 0;
    int r = 0;
    for (int i = 0; i < bits.n; ++i) {
        if (bits.x[i] < 0 || in_tile[bits.x[i]]) {
            p.out_pos[k++] = i;
        } else {
            p.rest_in[r] = bits.x[i];
            p.rest_out[r++] = i;
        }
    }
    p.n_rest = r;
    if (k != p.tb_out || r > 48) return false;
    // tile positions of the summed bits: their rank among the tile's bits at that step
    Bits cur;
    for (cur.n = 0; cur.n < nx; ++cur.n) cur.x[cur.n] = cur.n;
    for (int s = 0; s < n; ++s) {
        ChainStep& st = p.step[s];
        int rank_of[64], lb = 0;
        for (int b = 0; b < cur.n; ++b) rank_of[b] = cur.x[b] < 0 || in_tile[cur.x[b]] ? lb++ : -1;
        st.lb = lb;
        if (lb - st.ns < 1) return false;  // a thread takes two free parts
        st.adj = -1;
        for (int b = 0; b < st.ns; ++b)
            if (rank_of[s_x[s][b]] == 0) st.adj = b;
        for (int i = 0; i < st.ns; ++i) st.ins[i] = rank_of[summed[s][i]];
        for (int j = 0; j < (1 << st.ns); ++j)
            for (int b = 0; b < st.ns; ++b)
                if ((j >> b) & 1) st.off[j] += 1 << rank_of[s_x[s][b]];
        cur.step(summed[s], st.ns, st.nb);
    }
    *out = p;
    return true;
}

// One workgroup a tile.
dim3 tile_grid(const ChainPlan& p) {
    const int64_t tiles = int64_t(1) << p.n_rest;
    const unsigned gx = unsigned(std::min<int64_t>(tiles, 65536));
    return dim3(gx, unsigned(tiles / gx));
}

template <class V, int MODE>
qt_status launch_chain(Ctx* c, const Tensor* X, Tensor* C, const ChainArgs& a) {
    hipLaunchKernelGGL((k_chain<V, MODE, false>), tile_grid(a.p), dim3(kChainThreads), 0, c->stream,
                       static_cast<const V*>(X->data), static_cast<V*>(C->data), a, static_cast<TileExp*>(nullptr));
    return check_hip(c, hipGetLastError(), "k_chain");
}

// The same with C scaled: its largest |re|, |im| in [0.5, 1), exponent on the device.
template <int MODE>
qt_status launch_chain_scaled(Ctx* c, const Tensor* X, Tensor* C, const ChainArgs& a) {
    qt_status s = acquire_exponent(c, C);
    if (s != QT_OK) return s;
    const int64_t tiles = int64_t(1) << a.p.n_rest;
    hipError_t e = hipSuccess;
    auto* const exps = static_cast<TileExp*>(c->pool.alloc(size_t(tiles) * sizeof(TileExp) + 256, &e));
    if (!exps) return check_hip(c, e, "qt_contract_chain: tile exponents");
    auto* const top = reinterpret_cast<int32_t*>(exps + tiles);
    auto* const out = static_cast<float2*>(C->data);
    hipLaunchKernelGGL((k_chain<float2, MODE, true>), tile_grid(a.p), dim3(kChainThreads), 0, c->stream,
                       static_cast<const float2*>(X->data), out, a, exps);
    const int32_t* const ex = X->exp_slot >= 0 ? c->d_exp + X->exp_slot : nullptr;
    hipLaunchKernelGGL(k_chain_top, dim3(1), dim3(kTopThreads), 0, c->stream, exps, tiles, ex, c->d_exp + C->exp_slot,
                       top);
    hipLaunchKernelGGL(k_chain_scale, tile_grid(a.p), dim3(kChainThreads), 0, c->stream, out, a.p, exps, top);
    s = check_hip(c, hipGetLastError(), "k_chain (rescaled)");
    c->pool.release(exps);  // later work on this stream may take it
    return s;
}

}  // namespace

// Smaller tensors go step by step: their steps take a launch's time each, and a tile per
// workgroup would leave most of the chip idle.
constexpr int kChainMinBits = 16;

}  // namespace qt

using qt::set_error;

extern "C" {

int qt_chain_links(int rank_x, int dim_log2, int dtype, int n, const int32_t* desc, const int32_t* axes) {
    if (n < 1 || !desc || !axes || rank_x < 0 || (dim_log2 != 1 && dim_log2 != 2) || rank_x * dim_log2 > 40 ||
        rank_x * dim_log2 < qt::kChainMinBits)
        return 0;
    for (int m = std::min(n, qt::kMaxLinks); m >= 2; --m) {
        qt::ChainPlan p;
        if (qt::plan_chain(rank_x * dim_log2, dim_log2, dtype == QT_DTYPE_C128, m, desc, axes, &p)) return m;
    }
    return 0;
}

qt_status qt_contract_chain(qt_ctx* cx, const qt_tensor* X, int rank_x, int n, const qt_tensor* const* G,
                            const int32_t* desc, const int32_t* axes, qt_tensor* C, int precision) {
    if (!cx) return QT_INVALID_INPUT;
    auto* ctx = &cx->impl;
    if (!X || !C || !G || !desc || !axes || n < 1 || n > qt::kMaxLinks)
        return set_error(ctx, QT_INVALID_INPUT, "qt_contract_chain: null argument or too many links");
    const qt::Tensor& x = X->impl;
    qt::Tensor& c = C->impl;
    const bool c128 = x.dtype == QT_DTYPE_C128, rescale = (precision & QT_RESCALE) != 0;
    const int form = precision & ~QT_RESCALE;
    if ((c128 && (form != QT_PLAIN_C128 || rescale)) ||
        (!c128 && form != QT_C64_4M && form != QT_C64_3M && form != QT_C64_BF16X3))
        return set_error(ctx, QT_INVALID_INPUT, "qt_contract_chain: precision does not fit dtype");
    if (x.rank != rank_x || c.rank != desc[3 * (n - 1) + 2] || c.dtype != x.dtype || c.dim_log2 != x.dim_log2 || &x == &c)
        return set_error(ctx, QT_INVALID_INPUT, "qt_contract_chain: C or X does not match the links");
    qt::ChainArgs a;
    std::memset(&a, 0, sizeof a);
    for (int s = 0; s < n; ++s) {
        if (!G[s] || G[s]->impl.rank != desc[3 * s] || G[s]->impl.dtype != x.dtype ||
            G[s]->impl.dim_log2 != x.dim_log2 || &G[s]->impl == &c)
            return set_error(ctx, QT_INVALID_INPUT, "qt_contract_chain: a small tensor does not match its link");
        if (G[s]->impl.exp_slot >= 0)
            return set_error(ctx, QT_UNSUPPORTED, "qt_contract_chain: a small tensor carries an exponent");
        a.g[s] = G[s]->impl.data;
    }
    if (!qt::plan_chain(rank_x * x.dim_log2, x.dim_log2, c128, n, desc, axes, &a.p))
        return set_error(ctx, QT_UNSUPPORTED, "qt_contract_chain: the links do not fit one pass");
    std::lock_guard<std::recursive_mutex> g(ctx->mu);
    qt_status s = qt::check_deadline(ctx, "qt_contract_chain");
    if (s != QT_OK) return s;
    (void)hipSetDevice(ctx->device);
    if (rescale)
        switch (form) {
            case QT_C64_4M: return qt::launch_chain_scaled<qt::MODE_4M>(ctx, &x, &c, a);
            case QT_C64_3M: return qt::launch_chain_scaled<qt::MODE_3M>(ctx, &x, &c, a);
            default: return qt::launch_chain_scaled<qt::MODE_BF16X3>(ctx, &x, &c, a);
        }
    switch (form) {
        case QT_PLAIN_C128: s = qt::launch_chain<double2, qt::MODE_PLAIN>(ctx, &x, &c, a); break;
        case QT_C64_4M: s = qt::launch_chain<float2, qt::MODE_4M>(ctx, &x, &c, a); break;
        case QT_C64_3M: s = qt::launch_chain<float2, qt::MODE_3M>(ctx, &x, &c, a); break;
        default: s = qt::launch_chain<float2, qt::MODE_BF16X3>(ctx, &x, &c, a); break;
    }
    if (s == QT_OK) s = qt::carry_exponent(ctx, &x, &G[0]->impl, &c);
    return s;
}

}  // extern "C"
