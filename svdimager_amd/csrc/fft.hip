// Batched 2D inverse DFT (sign +, unnormalised) of the moment planes, replacing
// cufftPlanMany + cufftExecC2C(CUFFT_INVERSE) (SVDIntegratedImager.cu:1658-1676, 1713).
//
// Two LDS-staged passes of a mixed-radix Stockham FFT (radices of 2 to 16, for lengths with prime
// factors up to 13).  G = ceil(3N/2) is 3 * 2^k for the usual image sizes; 1536, 3072 and 6144 have
// passes of their own around a 1536-point transform held by one wavefront.
// Only the central N x N of each transformed G x G plane is read by the image pass, so the row
// pass keeps the central `cols` output columns and the column pass transforms just those
// columns and keeps the central `rows` outputs.
#include "svdi_internal.hpp"

#include <algorithm>
#include <cmath>

namespace svdi {
namespace {

constexpr int kMaxStages = 24;

// Quotient q = n / d for 0 <= n < 2^27 and d <= 2^13 as (n * ceil(2^40 / d)) >> 40: the error
// term n / 2^40 stays below 1 / d, so the floor is exact without an integer divide.
struct FastDiv {
    uint64_t mul;
    __host__ __device__ uint32_t div(uint32_t n) const { return static_cast<uint32_t>((n * mul) >> 40); }
};

inline FastDiv make_fastdiv(uint32_t d) {
    FastDiv f;
    f.mul = ((1ull << 40) + d - 1) / d;
    return f;
}

struct FftStages {
    int n;
    int count;
    int radix[kMaxStages];
    FastDiv by_m[kMaxStages];      // m = n / R of the stage
    FastDiv by_ns[kMaxStages];     // ns = product of the earlier radices
};

// LDS index of element i of a transform: one float2 of padding per 32 keeps the radix-R
// Stockham writes (stride R) off shared banks.
__device__ __forceinline__ int pidx(int i) { return i + (i >> 5); }
__host__ __device__ inline size_t padded_len(size_t n) { return n + n / 32 + 1; }

// Complex values are float2, or double2 where a butterfly is formed in FP64 (the convolutions).
template <class V> __device__ __forceinline__ V cmul(V a, V b) { return V(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
template <class V> __device__ __forceinline__ V cadd(V a, V b) { return V(a.x + b.x, a.y + b.y); }
template <class V> __device__ __forceinline__ V csub(V a, V b) { return V(a.x - b.x, a.y - b.y); }
template <class V> __device__ __forceinline__ V mul_i(V a) { return V(-a.y, a.x); }   // i * a

// out[k] = sum_r v[r] e^{+2 pi i r k / R}
template <class V>
__device__ __forceinline__ void dft2(V* v) {
    const V a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
}

__device__ __forceinline__ void dft3(float2* v) {
    const float c = -0.5f, s = 0.86602540378443864676f;   // e^{2 pi i / 3} = c + i s
    const float2 t1 = cadd(v[1], v[2]);
    const float2 t2 = csub(v[1], v[2]);
    const float2 m = make_float2(v[0].x + c * t1.x, v[0].y + c * t1.y);
    const float2 is = make_float2(-s * t2.y, s * t2.x);
    v[0] = cadd(v[0], t1);
    v[1] = cadd(m, is);
    v[2] = csub(m, is);
}

template <class V>
__device__ __forceinline__ void dft4(V* v) {
    const V y0 = cadd(v[0], v[2]), y1 = csub(v[0], v[2]);
    const V y2 = cadd(v[1], v[3]), y3 = mul_i(csub(v[1], v[3]));
    v[0] = cadd(y0, y2);
    v[2] = csub(y0, y2);
    v[1] = cadd(y1, y3);
    v[3] = csub(y1, y3);
}

// cos and sin of 2 pi num / den, for constants.
constexpr double turn_cos(int num, int den) {
    num %= den;
    if (2 * num > den) num = den - num;                // cos(-x) = cos x
    const bool neg = 4 * num > den;                    // cos(pi - x) = -cos x
    const double x = 6.283185307179586476925 * (neg ? 0.5 - static_cast<double>(num) / den : static_cast<double>(num) / den);
    double term = 1.0, sum = 1.0;
    for (int k = 1; k <= 12; ++k) {
        term *= -x * x / ((2 * k - 1) * (2 * k));
        sum += term;
    }
    return neg ? -sum : sum;
}
constexpr double turn_sin(int num, int den) { return turn_cos(4 * num + 3 * den, 4 * den); }   // sin x = cos(x - pi/2)

// Odd prime P: out_k, out_{P-k} = v_0 + sum_j cos(2 pi j k / P) (v_j + v_{P-j}) +- i sum_j sin(2 pi j k / P)
// (v_j - v_{P-j}).
template <int P, class T = float>
struct TurnTable {
    T c[P], s[P];
    constexpr TurnTable() : c(), s() {
        for (int i = 0; i < P; ++i) {
            c[i] = static_cast<T>(turn_cos(i, P));
            s[i] = static_cast<T>(turn_sin(i, P));
        }
    }
};
template <int P>
__device__ __forceinline__ void dft_prime(float2* v) {
    constexpr TurnTable<P> t;
    constexpr int H = (P - 1) / 2;
    float2 a[H], b[H];
    const float2 x0 = v[0];
    float2 all = x0;
#pragma unroll
    for (int j = 0; j < H; ++j) {
        a[j] = cadd(v[j + 1], v[P - 1 - j]);
        b[j] = csub(v[j + 1], v[P - 1 - j]);
        all = cadd(all, a[j]);
    }
    v[0] = all;
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        float2 m = x0, n = make_float2(0.f, 0.f);
#pragma unroll
        for (int j = 0; j < H; ++j) {
            const int i = (j + 1) * k % P;
            m.x += t.c[i] * a[j].x;
            m.y += t.c[i] * a[j].y;
            n.x += t.s[i] * b[j].x;
            n.y += t.s[i] * b[j].y;
        }
        const float2 in = mul_i(n);
        v[k] = cadd(m, in);
        v[P - k] = csub(m, in);
    }
}

template <class V>
__device__ __forceinline__ void dft8(V* v) {
    const decltype(v->x) h = 0.70710678118654752440;
    V a[4], b[4];
    for (int r = 0; r < 4; ++r) {
        a[r] = cadd(v[r], v[r + 4]);
        b[r] = csub(v[r], v[r + 4]);
    }
    // b[r] *= e^{+2 pi i r / 8}
    b[1] = V(h * (b[1].x - b[1].y), h * (b[1].x + b[1].y));
    b[2] = mul_i(b[2]);
    b[3] = V(-h * (b[3].x + b[3].y), h * (b[3].x - b[3].y));
    dft4(a);
    dft4(b);
    for (int m = 0; m < 4; ++m) {
        v[2 * m] = a[m];
        v[2 * m + 1] = b[m];
    }
}

template <int R, class V>
__device__ __forceinline__ void dft_fixed(V* v);

// R = A^2: X[k1 + A k2] = sum_{n2 < A} W_A^{n2 k2} (W_R^{n2 k1} sum_{n1 < A} W_A^{n1 k1} v[A n1 + n2]).
template <int A, class V>
__device__ __forceinline__ void dft_square(V* v) {
    constexpr TurnTable<A * A, decltype(v->x)> t;
    V y[A][A];
#pragma unroll
    for (int n2 = 0; n2 < A; ++n2) {
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) y[n2][n1] = v[A * n1 + n2];
        dft_fixed<A>(y[n2]);
#pragma unroll
        for (int k1 = 1; k1 < A; ++k1)
            if (n2 != 0) y[n2][k1] = cmul(y[n2][k1], V(t.c[n2 * k1], t.s[n2 * k1]));
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
        V z[A];
#pragma unroll
        for (int n2 = 0; n2 < A; ++n2) z[n2] = y[n2][k1];
        dft_fixed<A>(z);
#pragma unroll
        for (int k2 = 0; k2 < A; ++k2) v[k1 + A * k2] = z[k2];
    }
}

// R = A B with A and B coprime (Good and Thomas): with n = B n1 + A n2 mod R and k = k1 mod A = k2 mod B,
// W_R^{n k} = W_A^{n1 k1} W_B^{n2 k2}: no twiddles, so no roundings but those of the factors.
template <int A, int B>
__device__ __forceinline__ void dft_coprime(float2* v) {
    float2 y[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) y[n2][n1] = v[(B * n1 + A * n2) % (A * B)];
        dft_fixed<A>(y[n2]);
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
        float2 z[B];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) z[n2] = y[n2][k1];
        dft_fixed<B>(z);
#pragma unroll
        for (int k = 0; k < A * B; ++k)
            if (k % A == k1) v[k] = z[k % B];
    }
}

template <int R, class V>
__device__ __forceinline__ void dft_fixed(V* v) {
    if constexpr (R == 2) dft2(v);
    else if constexpr (R == 4) dft4(v);
    else if constexpr (R == 8) dft8(v);
    else if constexpr (R == 3) dft3(v);
    else if constexpr (R == 5 || R == 7 || R == 11 || R == 13) dft_prime<R>(v);
    else if constexpr (R == 16) dft_square<4>(v);
    else if constexpr (R == 9) dft_square<3>(v);
    else if constexpr (R == 15) dft_coprime<3, 5>(v);
    else if constexpr (R == 12) dft_coprime<4, 3>(v);
    else dft_coprime<2, R / 2>(v);                     // 6, 10, 14
}

// put(t, get(t)) for t = threadIdx.x, + blockDim.x, ... < n, with the gets of kCopyBatch
// consecutive steps issued before their puts (several global loads in flight per thread).
constexpr int kCopyBatch = 8;
template <class Get, class Put>
__device__ __forceinline__ void copy_batched(int n, Get&& get, Put&& put) {
    const int step = static_cast<int>(blockDim.x);
    int t = static_cast<int>(threadIdx.x);
    for (; t + (kCopyBatch - 1) * step < n; t += kCopyBatch * step) {
        float2 v[kCopyBatch];
#pragma unroll
        for (int j = 0; j < kCopyBatch; ++j) v[j] = get(t + j * step);
#pragma unroll
        for (int j = 0; j < kCopyBatch; ++j) put(t + j * step, v[j]);
    }
    for (; t < n; t += step) put(t, get(t));
}

__device__ __forceinline__ const float2* load_twiddles(float2* lds, const float2* __restrict__ tw, int n) {
    copy_batched(n, [&](int t) { return tw[t]; }, [&](int t, float2 v) { lds[t] = v; });
    return lds;
}

// Barrier for data exchanged through LDS: global loads and stores stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Passes of the lengths without a kernel of their own.  A workgroup takes ntrans transforms (rows, or
// neighbouring columns) through the Stockham stages; the first stage's butterflies are read from
// memory and the last one's written to memory, so that a length of two to four stages goes through
// LDS one to three times.  Bound by LDS traffic and index arithmetic, which go with the number of stages, and by
// how many wavefronts hide them: radices of up to 16 in registers keep the stages few, and the registers of
// one or two butterflies (kHoldLess or kHoldMore elements a thread, held between reading and writing, as a
// stage is in place) keep the wavefronts many.  Rows + columns of eight planes, before (radices of up to 8,
// every stage from and to LDS; 7 and above a loop over a private array) and now: 768^2 31 + 21 -> 21 + 15
// us, 1500^2 103 + 81 -> 77 + 50, 2304^2 480 -> 133 + 173 (both), 3024^2 3590 -> 309 + 292 (both).
constexpr int kHoldLess = 16, kHoldMore = 20;
constexpr int kPassThreads = 1024;
constexpr int kPassElems = 6200;                   // of a workgroup's transforms, if it can choose
constexpr size_t kPassLds = 160 << 10;
constexpr int kRadices[] = {16, 15, 14, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};

// Padding of a pass's LDS: one float2 per 16, so that first stages with an even radix (stride R) spread
// over the banks, and transforms an odd multiple of four apart, so that four neighbouring elements
// of eight columns do.
__device__ __forceinline__ int pass_idx(int i) { return i + (i >> 4); }
__host__ __device__ inline int pass_len(int n) { return ((n + n / 16 + 1 + 3) & ~7) + 4; }

template <int R, int kHold, bool kRows, class Get, class Put>
__device__ __forceinline__ void pass_stage(float2* buf, int ntrans, int n, int pn, int ns, FastDiv by_m, FastDiv by_ns,
                                           const float2* tw, bool first, bool last, Get&& get, Put&& put) {
    constexpr int B = kHold / R;
    const int m = n / R, tstep = n / (ns * R), total = ntrans * m;
    const int threads = static_cast<int>(blockDim.x);
    // (Opaque, so that no radix's index arithmetic is moved out of the loop over tiles, where those of
    // all radices together would not fit the registers.)
    int tid = static_cast<int>(threadIdx.x);
    asm volatile("" : "+v"(tid));
    float2 v[B][R];
    int at[B], tr_of[B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int t = tid + b * threads;
        at[b] = -1;
        if (t < total) {
            // Rows: consecutive threads take consecutive elements; columns: consecutive columns.
            const int tr = kRows ? static_cast<int>(by_m.div(t)) : t & (ntrans - 1);
            const int j = kRows ? t - tr * m : t >> (31 - __builtin_clz(ntrans));
            tr_of[b] = tr;
            if (first) {
#pragma unroll
                for (int r = 0; r < R; ++r) v[b][r] = get(tr, j + r * m);
                at[b] = j * R;
            } else {
                const int jq = static_cast<int>(by_ns.div(j)), jm = j - jq * ns;
                const float2* in = buf + tr * pn;
                v[b][0] = in[pass_idx(j)];
#pragma unroll
                for (int r = 1; r < R; ++r) v[b][r] = cmul(in[pass_idx(j + r * m)], tw[jm * r * tstep]);
                at[b] = jq * ns * R + jm;
            }
        }
    }
#pragma unroll
    for (int b = 0; b < B; ++b)
        if (b * threads < total) dft_fixed<R>(v[b]);   // (the same for the whole workgroup)
    if (last) {
#pragma unroll
        for (int b = 0; b < B; ++b)
            if (at[b] >= 0)
#pragma unroll
                for (int r = 0; r < R; ++r) put(tr_of[b], at[b] + r * ns, v[b][r]);
        return;
    }
    lds_barrier();                                 // the stage (or the last tile) has been read
#pragma unroll
    for (int b = 0; b < B; ++b)
        if (at[b] >= 0)
#pragma unroll
            for (int r = 0; r < R; ++r) buf[tr_of[b] * pn + pass_idx(at[b] + r * ns)] = v[b][r];
    lds_barrier();
}

template <int kHold, bool kRows, class Get, class Put>
__device__ __forceinline__ void pass_transforms(float2* buf, int ntrans, const FftStages& st, const float2* tw, Get&& get,
                                                Put&& put) {
    const int n = st.n, pn = pass_len(n);
    int ns = 1;
    for (int stage = 0; stage < st.count; ++stage) {
        const FastDiv bm = st.by_m[stage], bn = st.by_ns[stage];
        const bool first = stage == 0, last = stage == st.count - 1;
        const int R = st.radix[stage];
        auto run = [&](auto radix) {
            pass_stage<decltype(radix)::value, kHold, kRows>(buf, ntrans, n, pn, ns, bm, bn, tw, first, last, get, put);
        };
        switch (R) {
            case 2: run(std::integral_constant<int, 2>()); break;
            case 3: run(std::integral_constant<int, 3>()); break;
            case 4: run(std::integral_constant<int, 4>()); break;
            case 5: run(std::integral_constant<int, 5>()); break;
            case 6: run(std::integral_constant<int, 6>()); break;
            case 7: run(std::integral_constant<int, 7>()); break;
            case 8: run(std::integral_constant<int, 8>()); break;
            case 9: run(std::integral_constant<int, 9>()); break;
            case 10: run(std::integral_constant<int, 10>()); break;
            case 11: run(std::integral_constant<int, 11>()); break;
            case 12: run(std::integral_constant<int, 12>()); break;
            case 13: run(std::integral_constant<int, 13>()); break;
            case 14: run(std::integral_constant<int, 14>()); break;
            case 15: run(std::integral_constant<int, 15>()); break;
            default: run(std::integral_constant<int, 16>()); break;
        }
        ns *= R;
    }
}

// One 1536-point inverse transform per wavefront (G = 24 x 64), held in registers.  With
// n = 64 n1 + l and k = k1 + 24 k2 (Cooley-Tukey, W = e^{+2 pi i / 1536}):
//   lane l:  Y[k1] = W^{l k1} sum_{n1} x[64 n1 + l] W_24^{n1 k1}   (24-point DFT as 8 x 3),
//   X[k1 + 24 k2] = sum_l Y_l[k1] W_64^{l k2},
// the 64-point DFTs across lanes done as 8 x 8 (l = 8a + b, k2 = c + 8d) through one padded LDS
// tile per wavefront: pass A takes (k1, b) and transforms over a, times W_64^{b c}; pass B takes
// (k1, c) and transforms over b, giving X[k1 + 24 c + 192 d].  load(n) reads x[n] (lane l asks
// for n = 64 n1 + l); store(k, X[k]) is called for every k, lane l holding k = l + 64 j + 192 d.
constexpr int kFftWaves = 4;                 // wavefronts (transforms) per workgroup
constexpr int kTileStride = 65;              // float2 per k1 row of the LDS tile (64 + 1 pad)

__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Twiddles of the 1536-point wavefront transform in the order in which lanes ask for them, so that
// each request reads 64 consecutive entries (from the one table of W_1536^m the lanes of a request
// lie up to 64 lines apart, which bound the passes): W^{l k1} at [k1][l], W_64^{b c} at [c][q], q = 24 b +
// k1 (the place of (k1, b) below), and W_24^{v s} at [8 v + s].
struct Fft1536Tables {
    const float2 *lane, *cross, *w24;
};
constexpr int kTabLane = 24 * 64, kTabCross = 8 * 192, kTab24 = 24;
constexpr int kTabAll = kTabLane + kTabCross + kTab24;
__device__ __forceinline__ Fft1536Tables fft1536_tables(const float2* __restrict__ t) {
    return {t, t + kTabLane, t + kTabLane + kTabCross};
}

// fft1536_wave_regs takes the lane's inputs already in registers: y[v][u] = x[64 (3u + v) + l].
template <class Store>
__device__ __forceinline__ void fft1536_wave_regs(float2 (&y)[3][8], float2* tile, const Fft1536Tables& tw,
                                                  int lane, Store&& store) {
    // 24-point DFT over n1 = 3u + v, k1 = s + 8t: 8-point DFTs over u, times W_24^{v s}, then
    // 3-point DFTs over v.
#pragma unroll
    for (int v = 0; v < 3; ++v) dft8(y[v]);
#pragma unroll
    for (int v = 1; v < 3; ++v)
#pragma unroll
        for (int s8 = 1; s8 < 8; ++s8) y[v][s8] = cmul(y[v][s8], tw.w24[8 * v + s8]);
#pragma unroll
    for (int s8 = 0; s8 < 8; ++s8) {
        float2 t3[3] = {y[0][s8], y[1][s8], y[2][s8]};
        dft3(t3);
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const int k1 = s8 + 8 * t;
            // times W^{l k1} (l k1 < 1536), into the tile at [k1][l]
            tile[k1 * kTileStride + lane] = k1 == 0 ? t3[t] : cmul(t3[t], tw.lane[k1 * 64 + lane]);
        }
    }
    wave_lds_fence();
    // Pass A: q = lane + 64 j -> (k1, b) = (q % 24, q / 24); 8-point DFT over a, times W_64^{b c}.
    float2 w[3][8];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int q = lane + 64 * j, k1 = q % 24, b = q / 24;
#pragma unroll
        for (int a = 0; a < 8; ++a) w[j][a] = tile[k1 * kTileStride + 8 * a + b];
    }
    wave_lds_fence();
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int q = lane + 64 * j, k1 = q % 24, b = q / 24;
        dft8(w[j]);
#pragma unroll
        for (int c = 1; c < 8; ++c) w[j][c] = cmul(w[j][c], tw.cross[c * 192 + q]);
#pragma unroll
        for (int c = 0; c < 8; ++c) tile[k1 * kTileStride + 8 * b + c] = w[j][c];
    }
    wave_lds_fence();
    // Pass B: p = lane + 64 j -> (k1, c) = (p % 24, p / 24); 8-point DFT over b gives X[p + 192 d].
    // Every value is read before the first store (the stores may go to the tile's memory).
    float2 z[3][8];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int p = lane + 64 * j, k1 = p % 24, c = p / 24;
#pragma unroll
        for (int b = 0; b < 8; ++b) z[j][b] = tile[k1 * kTileStride + 8 * b + c];
    }
    wave_lds_fence();
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int p = lane + 64 * j;
        dft8(z[j]);
#pragma unroll
        for (int d = 0; d < 8; ++d) store(p + 192 * d, z[j][d]);
    }
}

template <class Load, class Store>
__device__ __forceinline__ void fft1536_wave(float2* tile, const Fft1536Tables& tw, int lane,
                                             Load&& load, Store&& store) {
    float2 y[3][8];                                // y[v][u] = x[64 (3u + v) + l]
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int v = 0; v < 3; ++v) y[v][u] = load(64 * (3 * u + v) + lane);
    wave_lds_fence();                              // the tile may be where the loads came from
    fft1536_wave_regs(y, tile, tw, lane, store);
}

// Workgroups are dealt to the 8 XCDs round-robin in launch order, each XCD with its own L2.
// Remapped so that consecutive logical tiles (neighbouring column strips, which share cache
// lines) run on the same XCD at about the same time.
// A bijection of [0, total): XCD x takes the contiguous tiles [x q + min(x, r), ...), q + 1 of
// them for x < r and q otherwise (q = total / 8, r = total % 8).
__device__ __forceinline__ int xcd_local_tile(int linear, int total) {
    constexpr int kXcds = 8;
    const int q = total / kXcds, r = total % kXcds;
    const int x = linear % kXcds, local = linear / kXcds;
    return x * q + min(x, r) + local;
}

// G = 1536 s, s = 1, 2 or 4: the column direction's radix-s step (decimation in frequency) is done
// in the row pass, on the row-transformed rows x_n, x_{n + 1536}, ...: sub-plane q holds
// y_q[n] = W^{n q} sum_m W_s^{m q} x_{n + 1536 m}, n < 1536, W = e^{2 pi i / G}, and its 1536-point
// column transform gives the output rows s k + q.  Between the passes element (n, c) of sub-plane i lies
// at i sub_stride + n row_stride + (c / 8) block_stride + c % 8.  For s > 1 the columns are in blocks,
// [sub-plane][block][n][8], which the column pass reads as contiguous runs (48 planes of 3072^2: rows 1.49
// + columns 0.87 ms, against 1.34 + 1.17 row-major); for s = 1 the planes are row-major (8 planes of
// 1536^2: 54 + 51 us, against 62 + 47 in blocks).
constexpr int kBlockCols = 8;                      // 64-byte row segments
constexpr int kSub = 1536;
struct MidLayout {
    size_t sub_stride;
    int row_stride, block_stride;
    __device__ __forceinline__ size_t row(size_t sub, int n) const { return sub * sub_stride + static_cast<size_t>(n) * row_stride; }
    __device__ __forceinline__ size_t col(int kc) const {
        return static_cast<size_t>(kc / kBlockCols) * block_stride + kc % kBlockCols;
    }
};

// Row pass for G = 1536: one wavefront per row of the P x G rows; loads stride 64 per lane are
// coalesced; only the columns col_lo .. col_lo + cols - 1 are stored.
__global__ void __launch_bounds__(64 * kFftWaves)
k_fft_rows_1536(const float2* __restrict__ in, float2* __restrict__ out, const float2* __restrict__ tab,
                int total_rows, int col_lo, int cols, MidLayout mid) {
    constexpr int G = 1536;
    __shared__ float2 tile_all[kFftWaves][24 * kTileStride];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int row = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x * kFftWaves + wave));
    if (row >= total_rows) return;                 // whole wavefronts; no workgroup barrier below
    const float2* src = in + static_cast<size_t>(row) * G;
    const int plane = row / G, n = row - plane * G;
    float2* dst = out + mid.row(plane, n);
    fft1536_wave(tile_all[wave], fft1536_tables(tab), lane, [&](int m) { return src[m]; },
                 [&](int k, float2 v) {
                     const int kc = k - col_lo;
                     if (kc >= 0 && kc < cols) dst[mid.col(kc)] = v;
                 });
}

// Column pass of the 1536-point transforms of column blocks (s sub-planes per plane), bound by memory:
// persistent workgroups, one per CU, a wavefront per column of the block.  The block is read into LDS, each
// wavefront transforms one column in place (the column's LDS region is also its exchange tile), and
// the output rows s k + q in the window row_lo .. row_lo + rows - 1 are written.  The next block's
// loads are issued before the transforms, which take their twiddles from LDS so that they wait
// for no global load, and stay in flight across the barriers: with one workgroup per CU the memory
// pipe is otherwise idle while it computes (with a workgroup per block and the twiddles gathered from
// global memory: 8 planes of 1536^2 56 us, now 52; 48 of 3072^2 1.48 ms, 0.89; 8 of 6144^2, which then
// had half transforms by pairs of wavefronts, 1.86 ms, 0.59).  Output element (row r, column c) of plane p goes to
// p plane_stride + (c / 8) block_stride + r row_stride + c % 8 in a row-major plane (split_rows = 0), or,
// with row_stride = 8 and split_rows = rows / s, to row q split_rows + k of its column block
// (FftWindow).
constexpr int kColLen = 24 * kTileStride;          // float2 per column region (>= 1536)
constexpr size_t kColsLds = sizeof(float2) * (kBlockCols * kColLen + kTabLane + kTabCross);
struct ColsOut {
    size_t plane_stride, block_stride;
    int row_stride, split_rows;
};

__global__ void __launch_bounds__(64 * kBlockCols)
k_fft_cols_1536(const float2* __restrict__ in, float2* __restrict__ out, const float2* __restrict__ tab,
                int s, int tiles, int nblk, int cols, int row_lo, int rows, MidLayout mid, ColsOut o) {
    constexpr int H = kSub, kThreadsC = 64 * kBlockCols, kLoads = H / 64;
    extern __shared__ float2 cols_lds[];
    float2* strip = cols_lds;
    float2* tab_lds = cols_lds + kBlockCols * kColLen;
    for (int t = threadIdx.x; t < kTabLane + kTabCross; t += kThreadsC) tab_lds[t] = tab[t];
    const Fft1536Tables tw = {tab_lds, tab_lds + kTabLane, tab + kTabLane + kTabCross};
    // Tiles (plane, q, block) are dealt so that an XCD's workgroups work on neighbouring blocks.
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int c = threadIdx.x % kBlockCols, r0 = threadIdx.x / kBlockCols;
    // Element (r, c) of a block: thread t = (r mod 64) kBlockCols + c loads rows r0 + 64 j.
    float2 v[kLoads];
    auto load = [&](int tile) {
        const int sub = tile / nblk;
        const float2* src = in + mid.row(sub, r0) + static_cast<size_t>(tile - sub * nblk) * mid.block_stride + c;
#pragma unroll
        for (int j = 0; j < kLoads; ++j) v[j] = src[static_cast<size_t>(64 * j) * mid.row_stride];
    };
    int tile = xcd_local_tile(blockIdx.x, gridDim.x);
    if (tile < tiles) load(tile);
    for (; tile < tiles; tile += gridDim.x) {
        lds_barrier();                             // the block before this one has been written out
#pragma unroll
        for (int j = 0; j < kLoads; ++j) strip[c * kColLen + r0 + 64 * j] = v[j];
        lds_barrier();
        if (tile + static_cast<int>(gridDim.x) < tiles) load(tile + gridDim.x);
        {
            float2* col = strip + wave * kColLen;
            fft1536_wave(col, tw, lane, [&](int n) { return col[n]; }, [&](int k, float2 x) { col[k] = x; });
        }
        lds_barrier();
        // Transform outputs k_lo .. k_lo + nk - 1 land in the window.
        const int sub = tile / nblk, blk = tile - sub * nblk;
        const int plane = sub / s, q = sub - plane * s;
        const int k_lo = max(0, (row_lo - q + s - 1) / s);
        const int nk = min(H, (row_lo + rows - q + s - 1) / s) - k_lo;
        if (blk * kBlockCols + c < cols) {
            float2* dst = out + plane * o.plane_stride + blk * o.block_stride + c;
#pragma unroll 8
            for (int k = r0; k < nk; k += kThreadsC / kBlockCols) {
                const int r = o.split_rows != 0 ? q * o.split_rows + k : s * (k_lo + k) + q - row_lo;
                dst[static_cast<size_t>(r) * o.row_stride] = strip[c * kColLen + k_lo + k];
            }
        }
    }
}

// Row pass for G = 3072: one workgroup per (plane, n < 1536) transforms rows n and n + 1536, a
// pair of wavefronts per row, by decimation in time: E and O are the transforms of the even and odd
// samples (each into its own LDS tile), X[k] = E[k] + W^k O[k] and X[k + 1536] = E[k] - W^k O[k],
// W = e^{2 pi i / 3072}.  The column direction's step gives a_n = x_n + x_{n + 1536} and
// b_n = (x_n - x_{n + 1536}) W^n, stored as row n of the plane's two sub-planes (the columns col_lo ..
// col_lo + cols - 1).  (Decimation in frequency, whose loads are whole runs, took 1.61 ms for 1.51: its
// extra LDS exchange costs more than the half-used lines, which the second wavefront finds in L2.)
// As the 6144-point pass: persistent workgroups of two tiles at a time, the next tiles' rows requested as soon as the
// transforms have taken the present ones, every twiddle in LDS (48 planes: a workgroup per tile 1.50 ms,
// now 1.34).
constexpr int kRows3Tiles = 2, kRows3Threads = 256 * kRows3Tiles;
constexpr size_t kRows3Lds = sizeof(float2) * (4 * kRows3Tiles * 24 * kTileStride + kTabLane + kTabCross + kSub);
__global__ void __launch_bounds__(kRows3Threads)
k_fft_rows_3072(const float2* __restrict__ in, float2* __restrict__ out, const float2* __restrict__ tw,
                const float2* __restrict__ tab, int pairs, int col_lo, int cols, MidLayout mid) {
    constexpr int G = 3072, H = kSub, kTile = 24 * kTileStride;
    extern __shared__ float2 rows3_lds[];          // [tile][row n or n + 1536][even or odd][kTile], tables, W^k
    float2* tab_lds = rows3_lds + 4 * kRows3Tiles * kTile;
    float2* step_tw = tab_lds + kTabLane + kTabCross;
    for (int t = threadIdx.x; t < kTabLane + kTabCross; t += kRows3Threads) tab_lds[t] = tab[t];
    for (int t = threadIdx.x; t < H; t += kRows3Threads) step_tw[t] = tw[t];
    const Fft1536Tables tables = {tab_lds, tab_lds + kTabLane, tab + kTabLane + kTabCross};
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int which = (wave >> 1) & 1, half = wave & 1;         // row n or n + 1536; even or odd
    float2* const tile_lds = rows3_lds + wave * kTile;
    const float2* const pair_lds = rows3_lds + (wave & ~3) * kTile;
    float2 x[3][8];
    auto load = [&](int pair) {
        const int tile_id = kRows3Tiles * pair + (wave >> 2), plane = tile_id / H, n = tile_id - plane * H;
        const float2* src = in + (static_cast<size_t>(plane) * G + n + which * H) * G + half;
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int v = 0; v < 3; ++v) x[v][u] = src[2 * (64 * (3 * u + v) + lane)];
    };
    int pair = xcd_local_tile(blockIdx.x, gridDim.x);
    if (pair < pairs) load(pair);
    lds_barrier();                                 // the tables
    for (; pair < pairs; pair += gridDim.x) {
        fft1536_wave_regs(x, tile_lds, tables, lane, [&](int k, float2 v) { tile_lds[k] = v; });
        if (pair + static_cast<int>(gridDim.x) < pairs) load(pair + gridDim.x);
        lds_barrier();
        const int tile_id = kRows3Tiles * pair + (wave >> 2), plane = tile_id / H, n = tile_id - plane * H;
        const float2 wn = tw[n];
        float2* dst_a = out + mid.row(2 * static_cast<size_t>(plane), n);
        float2* dst_b = out + mid.row(2 * static_cast<size_t>(plane) + 1, n);
#pragma unroll
        for (int k = threadIdx.x & 255; k < H; k += 256) {
            const float2 wk = step_tw[k];
            const float2 en = pair_lds[k], on = cmul(pair_lds[kTile + k], wk);
            const float2 em = pair_lds[2 * kTile + k], om = cmul(pair_lds[3 * kTile + k], wk);
            const float2 xn0 = cadd(en, on), xn1 = csub(en, on);      // row n at columns k, k + 1536
            const float2 xm0 = cadd(em, om), xm1 = csub(em, om);      // row n + 1536
            if (k >= col_lo && k < col_lo + cols) {
                const size_t i = mid.col(k - col_lo);
                dst_a[i] = cadd(xn0, xm0);
                dst_b[i] = cmul(csub(xn0, xm0), wn);
            }
            const int k1 = k + H;
            if (k1 >= col_lo && k1 < col_lo + cols) {
                const size_t i = mid.col(k1 - col_lo);
                dst_a[i] = cadd(xn1, xm1);
                dst_b[i] = cmul(csub(xn1, xm1), wn);
            }
        }
        lds_barrier();                             // the rows have been read
    }
}

// Row pass for G = 6144 = 4 x 1536: one workgroup per (plane, n < 1536) transforms the four rows
// n + 1536 m, two at a time with four wavefronts each: wavefront j of a row transforms the samples
// x[4 i + j] (i < 1536, the 1536-point wavefront transform) into F_j,
// then a radix-4 step along the row: with W = e^{2 pi i / 6144} and k = k0 + 1536 p (k0 < 1536,
// p < 4), X[k] = sum_j W^{j k} F_j[k0] = sum_j i^{j p} (W^{j k0} F_j[k0]).  Every thread keeps the
// sums of the column direction's radix-4 step for its twelve columns k = threadIdx.x + 512 i in
// registers over the four rows and stores them as row n of the plane's four sub-planes (the columns
// col_lo .. col_lo + cols - 1).  A row pass that took two rows had left half of the column step to the
// column pass (8 planes: 1.20 + 1.86 ms for both passes, then 1.39 + 0.59).
// Bound by memory, as the column pass: persistent workgroups, one per CU, request the next two rows
// as soon as a transform has taken the present ones into LDS, and keep every twiddle in LDS, so that nothing
// waits behind those loads (eight planes: a workgroup per tile, twiddles from memory 1.39 ms, now
// 1.12).
constexpr int kRows6Threads = 512;
constexpr size_t kRows6Lds = sizeof(float2) * (8 * 24 * kTileStride + kTabLane + kTabCross + 3 * kSub);
__global__ void __launch_bounds__(kRows6Threads)
k_fft_rows_6144(const float2* __restrict__ in, float2* __restrict__ out, const float2* __restrict__ tw,
                const float2* __restrict__ tab, int tiles, int col_lo, int cols, MidLayout mid) {
    constexpr int G = 6144, H = kSub, kTile = 24 * kTileStride, kPer = H / kRows6Threads;
    extern __shared__ float2 rows6_lds[];          // [row of the pair][residue j][kTile], tables, W^{j k}
    float2* tab_lds = rows6_lds + 8 * kTile;
    float2* step_tw = tab_lds + kTabLane + kTabCross;
    for (int t = threadIdx.x; t < kTabLane + kTabCross; t += kRows6Threads) tab_lds[t] = tab[t];
    for (int t = threadIdx.x; t < H; t += kRows6Threads)
        for (int j = 1; j < 4; ++j) step_tw[(j - 1) * H + t] = tw[j * t];
    const Fft1536Tables tables = {tab_lds, tab_lds + kTabLane, tab + kTabLane + kTabCross};
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    float2* const tile_lds = rows6_lds + wave * kTile;
    // Samples of row n + (half + 2 (wave / 4)) H of the tile's plane, residue wave % 4.
    float2 x0[3][8];
    auto load = [&](int tile_id, int half) {
        const int plane = tile_id / H, n = tile_id - plane * H;
        const float2* src = in + (static_cast<size_t>(plane) * G + n + (half + 2 * (wave >> 2)) * H) * G + (wave & 3);
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int v = 0; v < 3; ++v) x0[v][u] = src[4 * (64 * (3 * u + v) + lane)];
    };
    int tile_id = xcd_local_tile(blockIdx.x, gridDim.x);
    if (tile_id < tiles) load(tile_id, 0);
    lds_barrier();                                 // the tables
    for (; tile_id < tiles; tile_id += gridDim.x) {
    const int plane = tile_id / H, n = tile_id - plane * H;
    const int tile_next = tile_id + static_cast<int>(gridDim.x);
    float2 y[4][kPer][4];                          // [q][i][p]
#pragma unroll
    for (int half = 0; half < 2; ++half) {         // rows m = half and half + 2
        fft1536_wave_regs(x0, tile_lds, tables, lane, [&](int k, float2 v) { tile_lds[k] = v; });
        if (half == 0) load(tile_id, 1);
        else if (tile_next < tiles) load(tile_next, 0);
        lds_barrier();
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int k0 = threadIdx.x + kRows6Threads * i;
            float2 x[2][4];                        // the pair's rows at k0 + 1536 p
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const float2* t = rows6_lds + 4 * r * kTile;
                const float2 g0 = t[k0];
                const float2 g1 = cmul(t[kTile + k0], step_tw[k0]);
                const float2 g2 = cmul(t[2 * kTile + k0], step_tw[H + k0]);
                const float2 g3 = cmul(t[3 * kTile + k0], step_tw[2 * H + k0]);
                const float2 s02 = cadd(g0, g2), d02 = csub(g0, g2);
                const float2 s13 = cadd(g1, g3), id13 = mul_i(csub(g1, g3));
                x[r][0] = cadd(s02, s13);
                x[r][1] = cadd(d02, id13);
                x[r][2] = csub(s02, s13);
                x[r][3] = csub(d02, id13);
            }
            // y_0 and y_2 take +- (x_1 + x_3), y_1 and y_3 take +- i (x_1 - x_3).
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const float2 sum = cadd(x[0][p], x[1][p]), dif = csub(x[0][p], x[1][p]);
                if (half == 0) {
                    y[0][i][p] = sum;
                    y[1][i][p] = dif;
                } else {
                    const float2 s = y[0][i][p], d = y[1][i][p], id = mul_i(dif);
                    y[0][i][p] = cadd(s, sum);
                    y[2][i][p] = csub(s, sum);
                    y[1][i][p] = cadd(d, id);
                    y[3][i][p] = csub(d, id);
                }
            }
        }
        lds_barrier();                             // the rows have been read
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        float2* dst = out + mid.row(4 * static_cast<size_t>(plane) + q, n);
        const float2 wq = tw[q * n];
#pragma unroll
        for (int i = 0; i < kPer; ++i)
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const int kc = threadIdx.x + kRows6Threads * i + H * p - col_lo;
                if (kc >= 0 && kc < cols)
                    dst[mid.col(kc)] = q == 0 ? y[q][i][p] : cmul(y[q][i][p], wq);
            }
    }
    }
}

// Row pass of the other lengths: planes [P][G][G] -> row_out [P][G][cols] (output columns col_lo ..
// col_lo + cols - 1), `batch` rows of the P G at a time.  Workgroups walk the tiles, so that the twiddle
// table is loaded once for several.
template <int kHold>
__global__ void __launch_bounds__(kPassThreads)
k_fft_rows(const float2* __restrict__ in, float2* __restrict__ out, FftStages st, const float2* __restrict__ tw_g,
           int total_rows, int batch, int tiles, int col_lo, int cols) {
    extern __shared__ float2 lds[];
    const int G = st.n;
    const float2* tw = load_twiddles(lds, tw_g, G);
    float2* buf = lds + G;
    lds_barrier();
    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const int row0 = tile * batch;
        const float2* src = in + static_cast<size_t>(row0) * G;
        float2* dst = out + static_cast<size_t>(row0) * cols - col_lo;
        pass_transforms<kHold, true>(buf, min(batch, total_rows - row0), st, tw,
                              [&](int tr, int i) { return src[static_cast<size_t>(tr) * G + i]; },
                              [&](int tr, int k, float2 v) {
                                  if (k >= col_lo && k < col_lo + cols) dst[static_cast<size_t>(tr) * cols + k] = v;
                              });
    }
}

// Column pass: row_out [P][G][cols] -> out [P][rows][cols] (output rows row_lo .. row_lo + rows - 1).  A
// tile is a strip of `width` (a power of two) columns of a plane, dealt XCD-locally; the last strip of a
// plane repeats its last column in place of those past the end.
template <int kHold>
__global__ void __launch_bounds__(kPassThreads)
k_fft_cols(const float2* __restrict__ in, float2* __restrict__ out, FftStages st, const float2* __restrict__ tw_g,
           int width, int strips, int tiles, int cols, int row_lo, int rows) {
    extern __shared__ float2 lds[];
    const int G = st.n;
    const float2* tw = load_twiddles(lds, tw_g, G);
    float2* buf = lds + G;
    lds_barrier();
    for (int tile = xcd_local_tile(blockIdx.x, gridDim.x); tile < tiles; tile += gridDim.x) {
        const int plane = tile / strips, c0 = (tile - plane * strips) * width;
        const float2* src = in + plane * static_cast<size_t>(G) * cols + c0;
        float2* dst = out + plane * static_cast<size_t>(rows) * cols + c0;
        const int nc = cols - c0;
        pass_transforms<kHold, false>(buf, width, st, tw,
                               [&](int tr, int i) { return src[static_cast<size_t>(i) * cols + min(tr, nc - 1)]; },
                               [&](int tr, int k, float2 v) {
                                   const int r = k - row_lo;
                                   if (r >= 0 && r < rows && tr < nc) dst[static_cast<size_t>(r) * cols + tr] = v;
                               });
    }
}

// Lengths with a prime factor above 13, as a convolution (Bluestein): with c[n] = e^{i pi n^2 / G},
// n k = (n^2 + k^2 - (k - n)^2) / 2 gives X[k] = c[k] sum_n (x[n] c[n]) conj(c[k - n]), a circular
// convolution of length M = 2^m >= 2 G - 1, done by two + transforms of length M in LDS:
// z = conj(F(x c) B), X[k] = c[k] conj(F(z)[k]), where B = F(conj(c)) / M, conj(c) continued evenly.
// The first stage is read from memory and the last one written to it; the last stage of the first
// transform, the product with B and the first stage of the second, which takes the same elements, are one.
// Rows + columns of the planes of a 301^2 image (453^2): 27 + 20 us; with every stage from and to LDS 54 + 37, as
// direct DFTs 518 + 304.  The butterflies are FP64 (which runs at the rate of plain FP32 here) and rounded once a
// stage: with FP32 ones the transform's error was already below the direct sums' (2.3e-7 rms of white planes'
// output for 5.4e-7, now 1.5e-7), but the image's was 3 % above theirs, now 24 % below.
struct BlueTables {
    const float2 *chirp, *tw, *spec;               // c[G], W_M[M], B[M]
};
__device__ __forceinline__ double2 widen(float2 a) { return make_double2(a.x, a.y); }
__device__ __forceinline__ double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
__device__ __forceinline__ float2 narrow(double2 a) { return make_float2(static_cast<float>(a.x), static_cast<float>(a.y)); }

// Radices of the first transform of length 2^E; the second's are the same in reverse.
template <int E>
struct BlueRadices {
    static constexpr int count = E < 8 ? 2 : E < 12 ? 3 : 4;
    static constexpr int r[4] = {E == 8 ? 4 : E == 9 || E == 10 || E == 12 ? 8 : 16, E == 10 || E == 11 ? 16 : 8,
                                 E < 8 ? 1 : 8, E < 12 ? 1 : 8};
    static constexpr int least = E == 8 ? 4 : 8;
    static constexpr int per_transform = (1 << E) / least;         // threads
};

// The transforms of `ntrans` sequences (per_transform threads each): get(tr, n) reads x[n], put(tr, k, X[k])
// takes the outputs k_lo .. k_lo + nk - 1.  kUnitN: consecutive threads take consecutive elements of x
// and X (else transforms).
template <int E, bool kUnitN, class Get, class Put>
__device__ __forceinline__ void blue_transforms(float2* lds, const BlueTables& tb, int G, int ntrans, int k_lo, int nk,
                                                Get&& get, Put&& put) {
    using L = BlueRadices<E>;
    constexpr int M = 1 << E;
    const int pn = static_cast<int>(padded_len(M));
    const float2* tw = load_twiddles(lds, tb.tw, M);
    float2* buf = lds + M;
    const int tid = static_cast<int>(threadIdx.x);
    lds_barrier();
    // Butterfly j of transform tr of a stage with m butterflies a transform.
    auto place = [&](int m, bool unit, int& tr, int& j) {
        tr = unit ? tid / m : tid % ntrans;
        j = unit ? tid % m : tid / ntrans;
        return tr < ntrans && j < m;
    };
    auto write = [&](auto radix, int tr, int d, int ns, const double2* x, bool active) {
        constexpr int R = decltype(radix)::value;
        lds_barrier();                             // the stage has been read
        if (active)
#pragma unroll
            for (int r = 0; r < R; ++r) buf[tr * pn + pidx(d + r * ns)] = narrow(x[r]);
        lds_barrier();
    };
    auto read = [&](auto radix, int tr, int j, int ns, double2* x) {
        constexpr int R = decltype(radix)::value, m = M / R;
        const int jm = j & (ns - 1), tstep = M / (ns * R);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            x[r] = widen(buf[tr * pn + pidx(j + r * m)]);
            if (r > 0) x[r] = cmul(x[r], widen(tw[jm * r * tstep]));
        }
    };
    auto middle = [&](auto radix, int ns) {
        constexpr int R = decltype(radix)::value;
        int tr, j;
        const bool active = place(M / R, true, tr, j);
        double2 x[R];
        if (active) {
            read(radix, tr, j, ns, x);
            dft_fixed<R>(x);
        }
        write(radix, tr, (j & ~(ns - 1)) * R + (j & (ns - 1)), ns, x, active);
    };
    using First = std::integral_constant<int, L::r[0]>;
    using Last = std::integral_constant<int, L::r[L::count - 1]>;
    {
        constexpr int R = First::value, m = M / R;
        int tr, j;
        const bool active = place(m, kUnitN, tr, j);
        double2 x[R];
        if (active) {
            float2 v[R];
#pragma unroll
            for (int r = 0; r < R; ++r) v[r] = j + r * m < G ? get(tr, j + r * m) : make_float2(0.f, 0.f);
#pragma unroll
            for (int r = 0; r < R; ++r)
                x[r] = j + r * m < G ? cmul(widen(v[r]), widen(tb.chirp[j + r * m])) : make_double2(0.0, 0.0);
            dft_fixed<R>(x);
        }
        write(First(), tr, j * R, 1, x, active);
    }
    if constexpr (L::count > 2) middle(std::integral_constant<int, L::r[1]>(), L::r[0]);
    if constexpr (L::count > 3) middle(std::integral_constant<int, L::r[2]>(), L::r[0] * L::r[1]);
    {
        constexpr int R = Last::value, m = M / R;
        int tr, j;
        const bool active = place(m, true, tr, j);
        double2 x[R];
        if (active) {
            read(Last(), tr, j, m, x);
            dft_fixed<R>(x);
#pragma unroll
            for (int r = 0; r < R; ++r) x[r] = cconj(cmul(x[r], widen(tb.spec[j + r * m])));
            dft_fixed<R>(x);
        }
        write(Last(), tr, j * R, 1, x, active);
    }
    if constexpr (L::count > 3) middle(std::integral_constant<int, L::r[2]>(), L::r[3]);
    if constexpr (L::count > 2) middle(std::integral_constant<int, L::r[1]>(), M / (L::r[0] * L::r[1]));
    {
        constexpr int R = First::value, m = M / R;
        int tr, j;
        if (!place(m, kUnitN, tr, j)) return;
        double2 x[R];
        read(First(), tr, j, m, x);
        dft_fixed<R>(x);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int k = j + r * m - k_lo;
            if (k >= 0 && k < nk) put(tr, k, narrow(cmul(cconj(x[r]), widen(tb.chirp[k_lo + k]))));
        }
    }
}

// Threads of a workgroup: several transforms' where that leaves several workgroups to a CU; columns twice the
// rows', for longer row segments.
template <int E>
constexpr int blue_threads(bool rows) { return E == 13 ? 1024 : E == 12 || !rows ? 512 : 256; }

template <int E>
__global__ void __launch_bounds__(blue_threads<E>(true))
k_blue_rows(const float2* __restrict__ in, float2* __restrict__ out, BlueTables tb, int G, int total_rows, int batch,
            int col_lo, int cols) {
    extern __shared__ float2 lds[];
    const int row0 = blockIdx.x * batch;
    const float2* src = in + static_cast<size_t>(row0) * G;
    float2* dst = out + static_cast<size_t>(row0) * cols;
    blue_transforms<E, true>(lds, tb, G, min(batch, total_rows - row0), col_lo, cols,
                             [&](int tr, int n) { return src[static_cast<size_t>(tr) * G + n]; },
                             [&](int tr, int k, float2 v) { dst[static_cast<size_t>(tr) * cols + k] = v; });
}

template <int E>
__global__ void __launch_bounds__(blue_threads<E>(false))
k_blue_cols(const float2* __restrict__ in, float2* __restrict__ out, BlueTables tb, int G, int width, int cols, int row_lo,
            int rows, int strips) {
    extern __shared__ float2 lds[];
    const int tile = xcd_local_tile(blockIdx.x, gridDim.x);
    const size_t plane = tile / strips;
    const int c0 = (tile - static_cast<int>(plane) * strips) * width;
    const float2* src = in + plane * G * static_cast<size_t>(cols) + c0;
    float2* dst = out + plane * rows * static_cast<size_t>(cols) + c0;
    blue_transforms<E, false>(lds, tb, G, min(width, cols - c0), row_lo, rows,
                              [&](int tr, int n) { return src[static_cast<size_t>(n) * cols + tr]; },
                              [&](int tr, int k, float2 v) { dst[static_cast<size_t>(k) * cols + tr] = v; });
}

// The tables of BlueTables, contiguous, from FP64: one workgroup, B by a radix-2 transform in LDS (M
// double2).  M = 2^log_m <= 8192.
constexpr int kBlueThreads = 1024;
constexpr size_t kBlueMax = 8192;
__global__ void __launch_bounds__(kBlueThreads)
k_blue_tables(float2* __restrict__ tab, int G, int log_m) {
    extern __shared__ double2 zd[];
    const int M = 1 << log_m;
    float2 *chirp = tab, *tw = tab + G, *spec = tw + M;
    for (int t = threadIdx.x; t < M; t += kBlueThreads) {
        double sn, cs;
        sincospi(2.0 * t / M, &sn, &cs);
        tw[t] = make_float2(static_cast<float>(cs), static_cast<float>(sn));
        // conj(c) at +-n into the bit-reversed place, zero between
        const int n = min(t, M - t);
        double2 z = make_double2(0.0, 0.0);
        if (n < G) {
            sincospi(static_cast<double>(static_cast<long>(n) * n % (2 * G)) / G, &sn, &cs);
            if (t < G) chirp[t] = make_float2(static_cast<float>(cs), static_cast<float>(sn));
            z = make_double2(cs, -sn);
        }
        zd[__brev(static_cast<unsigned>(t)) >> (32 - log_m)] = z;
    }
    for (int l = 0; l < log_m; ++l) {
        __syncthreads();
        for (int t = threadIdx.x; t < M / 2; t += kBlueThreads) {
            const int h = 1 << l, j = t & (h - 1), i = ((t - j) << 1) + j;
            double sn, cs;
            sincospi(static_cast<double>(j) / h, &sn, &cs);
            const double2 a = zd[i], b = zd[i + h];
            const double2 wb = make_double2(b.x * cs - b.y * sn, b.x * sn + b.y * cs);
            zd[i] = make_double2(a.x + wb.x, a.y + wb.y);
            zd[i + h] = make_double2(a.x - wb.x, a.y - wb.y);
        }
    }
    __syncthreads();
    for (int t = threadIdx.x; t < M; t += kBlueThreads)
        spec[t] = make_float2(static_cast<float>(zd[t].x / M), static_cast<float>(zd[t].y / M));
}

// Direct O(G^2) DFT (rows then columns) for the other lengths that the Stockham passes do not take:
// below kBlueMin, where
// both take as long and the sums have the smaller error, and those whose convolution exceeds kBlueMax.
// sum_n src[n stride] W^{n k}, in partial sums of 64 terms.
__device__ __forceinline__ float2 direct_sum(const float2* __restrict__ src, size_t stride, int G, int k,
                                             const float2* __restrict__ tw) {
    float2 acc = make_float2(0.f, 0.f);
    for (int n0 = 0, t = 0; n0 < G; n0 += 64) {
        float2 part = make_float2(0.f, 0.f);
        const int end = min(G, n0 + 64);
        for (int n = n0; n < end; ++n) {
            part = cadd(part, cmul(src[n * stride], tw[t]));
            t += k;                                // n k mod G
            if (t >= G) t -= G;
        }
        acc = cadd(acc, part);
    }
    return acc;
}

__global__ void k_dft_rows_naive(const float2* __restrict__ in, float2* __restrict__ out, int G,
                                 const float2* __restrict__ tw, int col_lo, int cols) {
    const size_t plane = blockIdx.z;
    const int r = blockIdx.y;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= cols) return;
    const int k = col_lo + c;
    const float2* src = in + (plane * G + r) * static_cast<size_t>(G);
    out[(plane * G + r) * static_cast<size_t>(cols) + c] = direct_sum(src, 1, G, k, tw);
}

__global__ void k_dft_cols_naive(const float2* __restrict__ in, float2* __restrict__ out, int G,
                                 const float2* __restrict__ tw, int cols, int row_lo, int rows) {
    const size_t plane = blockIdx.z;
    const int r = blockIdx.y;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= cols) return;
    const int k = row_lo + r;
    const float2* src = in + plane * G * static_cast<size_t>(cols) + c;
    out[(plane * rows + r) * static_cast<size_t>(cols) + c] = direct_sum(src, static_cast<size_t>(cols), G, k, tw);
}

void stage_divisors(FftStages& st) {
    int ns = 1;
    for (int i = 0; i < st.count; ++i) {
        st.by_m[i] = make_fastdiv(static_cast<uint32_t>(st.n / st.radix[i]));
        st.by_ns[i] = make_fastdiv(static_cast<uint32_t>(ns));
        ns *= st.radix[i];
    }
}

// n in as few of the radices as do, of those the ones with the smallest sum, odd ones first (the first
// stage's LDS writes, a stride of its radix apart, then meet no bank twice).  False: n has a prime factor above
// 13 or is out of range.
constexpr int kPassMax = 8192;                     // (twiddles and one transform: 134 KB of LDS)
bool factorize(int n, FftStages& st) {
    if (n < 2 || n > kPassMax) return false;
    int best[kMaxStages], pick[kMaxStages], best_count = kMaxStages, best_sum = 0;
    auto search = [&](auto&& self, int rest, int depth, int sum, size_t from) -> void {
        if (rest == 1) {
            if (depth < best_count || (depth == best_count && sum < best_sum)) {
                best_count = depth;
                best_sum = sum;
                std::copy(pick, pick + depth, best);
            }
            return;
        }
        if (depth == best_count || depth + 1 == kMaxStages) return;
        for (size_t i = from; i < sizeof kRadices / sizeof kRadices[0]; ++i) {
            if (rest % kRadices[i] != 0) continue;
            pick[depth] = kRadices[i];
            self(self, rest / kRadices[i], depth + 1, sum + kRadices[i], i);
        }
    };
    search(search, n, 0, 0, 0);
    if (best_count == kMaxStages) return false;
    std::stable_partition(best, best + best_count, [](int r) { return r % 2 != 0; });
    st.n = n;
    st.count = best_count;
    std::copy(best, best + best_count, st.radix);
    stage_divisors(st);
    return true;
}

}  // namespace

// Twiddles e^{2 pi i t / G}, t < G, from FP64 sincospi, rounded to FP32, and behind them (for G = 1536
// s) the tables of the 1536-point wavefront transform (Fft1536Tables).
__global__ void k_twiddles(float2* __restrict__ tw, int G, int total) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= total) return;
    double turn = static_cast<double>(t) / static_cast<double>(G);
    if (t >= G) {
        const int i = t - G, j = i - kTabLane, m = j - kTabCross;
        int k;                                     // W_1536^k
        if (j < 0) k = (i / 64) * (i % 64);
        else if (m < 0) k = 24 * (j / 192) * (j % 192 / 24);
        else k = 64 * (m / 8) * (m % 8);
        turn = static_cast<double>(k) / kSub;
    }
    double sn, cs;
    sincospi(2.0 * turn, &sn, &cs);
    tw[t] = make_float2(static_cast<float>(cs), static_cast<float>(sn));
}

// The split s of G = 1536 s (0: another G).
static int fft_split(size_t G) { return G == 1536 ? 1 : G == 3072 ? 2 : G == 6144 ? 4 : 0; }
// The convolution length of G (0: G is not transformed by a convolution).
constexpr size_t kBlueMin = 51;
static size_t blue_len(size_t G) {
    FftStages st;
    if (G < kBlueMin || 2 * G - 1 > kBlueMax || factorize(static_cast<int>(G), st)) return 0;
    size_t M = 32;
    while (M < 2 * G - 1) M *= 2;
    return M;
}
static size_t twiddle_elems(size_t G) { return G + (fft_split(G) != 0 ? kTabAll : 2 * blue_len(G)); }

// The twiddle table of G in the context's workspace, computed on the stream (no host copy, no
// synchronisation) when G or the table's address changed since the last call.
void fft_prepare(svdi_context* ctx, size_t G) {
    const size_t total = twiddle_elems(G);
    float2* d = static_cast<float2*>(ctx->ws.get(Workspace::kTwiddles, total * sizeof(float2)));
    if (ctx->twiddle_n == G && ctx->twiddle_at == d) return;
    if (const size_t M = blue_len(G)) {
        const size_t lds = M * sizeof(double2);
        allow_dynamic_lds(reinterpret_cast<const void*>(&k_blue_tables), lds);
        k_blue_tables<<<1, kBlueThreads, lds, ctx->stream>>>(d, static_cast<int>(G), __builtin_ctzll(M));
    } else {
        k_twiddles<<<static_cast<unsigned>((total + 255) / 256), 256, 0, ctx->stream>>>(d, static_cast<int>(G),
                                                                                 static_cast<int>(total));
    }
    SVDI_LAUNCH_CHECK();
    ctx->twiddle_n = G;
    ctx->twiddle_at = d;
}

size_t fft_row_elems(size_t G, size_t cols) {
    return G * (fft_split(G) != 0 ? (cols + kBlockCols - 1) / kBlockCols * kBlockCols : cols);
}

FftWindow fft_window(size_t G, size_t row_lo, size_t rows, size_t cols) {
    FftWindow w;
    w.rows = static_cast<int>(rows);
    w.cols = static_cast<int>(cols);
    const size_t s = static_cast<size_t>(fft_split(G));
    if (s != 0 && cols % kBlockCols == 0 && rows % s == 0 && row_lo % s == 0) w.split = static_cast<int>(s);
    return w;
}

void launch_fft2_inverse(svdi_context* ctx, const float2* planes, size_t P, size_t G,
                         size_t row_lo, size_t rows, size_t col_lo, size_t cols,
                         float2* row_out, float2* out, const FftWindow& win) {
    fft_prepare(ctx, G);
    const float2* tw = static_cast<const float2*>(ctx->ws.get(Workspace::kTwiddles, twiddle_elems(G) * sizeof(float2)));
    const float2* tab = tw + G;
    const int split = fft_split(G);
    if (split != 0) {
        const int nblk = static_cast<int>((cols + kBlockCols - 1) / kBlockCols);
        const int clo = static_cast<int>(col_lo), nc = static_cast<int>(cols);
        MidLayout mid;
        mid.sub_stride = static_cast<size_t>(kSub) * nblk * kBlockCols;
        mid.row_stride = split == 1 ? nblk * kBlockCols : kBlockCols;
        mid.block_stride = split == 1 ? kBlockCols : kSub * kBlockCols;
        if (split == 4) {
            allow_dynamic_lds(reinterpret_cast<const void*>(&k_fft_rows_6144), kRows6Lds);
            const int row_tiles = static_cast<int>(P) * kSub;
            k_fft_rows_6144<<<static_cast<unsigned>(std::min(row_tiles, std::max(1, ctx->cu_count))), kRows6Threads, kRows6Lds,
                              ctx->stream>>>(planes, row_out, tw, tab, row_tiles, clo, nc, mid);
        } else if (split == 2) {
            allow_dynamic_lds(reinterpret_cast<const void*>(&k_fft_rows_3072), kRows3Lds);
            const int pairs = static_cast<int>(P) * kSub / kRows3Tiles;
            k_fft_rows_3072<<<static_cast<unsigned>(std::min(pairs, std::max(1, ctx->cu_count))), kRows3Threads, kRows3Lds,
                              ctx->stream>>>(planes, row_out, tw, tab, pairs, clo, nc, mid);
        } else {
            const int total_rows = static_cast<int>(P * G);
            k_fft_rows_1536<<<static_cast<unsigned>((total_rows + kFftWaves - 1) / kFftWaves), 64 * kFftWaves, 0,
                              ctx->stream>>>(planes, row_out, tab, total_rows, clo, nc, mid);
        }
        SVDI_LAUNCH_CHECK();
        const int tiles = static_cast<int>(P) * split * nblk;
        ColsOut o;
        o.plane_stride = rows * cols;
        o.block_stride = win.split != 0 ? rows * kBlockCols : kBlockCols;
        o.row_stride = win.split != 0 ? kBlockCols : nc;
        o.split_rows = win.split != 0 ? static_cast<int>(rows) / split : 0;
        allow_dynamic_lds(reinterpret_cast<const void*>(&k_fft_cols_1536), kColsLds);
        const int grid = std::min(tiles, std::max(1, ctx->cu_count));
        k_fft_cols_1536<<<static_cast<unsigned>(grid), 64 * kBlockCols, kColsLds, ctx->stream>>>(
            row_out, out, tab, split, tiles, nblk, nc, static_cast<int>(row_lo), static_cast<int>(rows), mid, o);
        SVDI_LAUNCH_CHECK();
        return;
    }
    FftStages st;
    if (const size_t M = blue_len(G)) {
        const int g = static_cast<int>(G), nc = static_cast<int>(cols), total_rows = static_cast<int>(P * G);
        const BlueTables tb = {tw, tw + G, tw + G + M};
        auto run = [&](auto exponent) {
            constexpr int E = decltype(exponent)::value;
            using L = BlueRadices<E>;
            constexpr int kRowThreads = blue_threads<E>(true), kColThreads = blue_threads<E>(false);
            const int batch = std::min(16, kRowThreads / L::per_transform), width = std::min(16, kColThreads / L::per_transform);
            auto lds = [&](int n) { return (M + static_cast<size_t>(n) * padded_len(M)) * sizeof(float2); };
            allow_dynamic_lds(reinterpret_cast<const void*>(&k_blue_rows<E>), lds(batch));
            k_blue_rows<E><<<static_cast<unsigned>((total_rows + batch - 1) / batch), kRowThreads, lds(batch), ctx->stream>>>(
                planes, row_out, tb, g, total_rows, batch, static_cast<int>(col_lo), nc);
            SVDI_LAUNCH_CHECK();
            const int strips = (nc + width - 1) / width;
            allow_dynamic_lds(reinterpret_cast<const void*>(&k_blue_cols<E>), lds(width));
            k_blue_cols<E><<<static_cast<unsigned>(strips * P), kColThreads, lds(width), ctx->stream>>>(
                row_out, out, tb, g, width, nc, static_cast<int>(row_lo), static_cast<int>(rows), strips);
            SVDI_LAUNCH_CHECK();
        };
        switch (__builtin_ctzll(M)) {
            case 7: run(std::integral_constant<int, 7>()); break;
            case 8: run(std::integral_constant<int, 8>()); break;
            case 9: run(std::integral_constant<int, 9>()); break;
            case 10: run(std::integral_constant<int, 10>()); break;
            case 11: run(std::integral_constant<int, 11>()); break;
            case 12: run(std::integral_constant<int, 12>()); break;
            case 13: run(std::integral_constant<int, 13>()); break;
            default: throw std::logic_error("convolution length out of range");
        }
        return;
    }
    if (!factorize(static_cast<int>(G), st)) {
        dim3 gr(static_cast<unsigned>((cols + 127) / 128), static_cast<unsigned>(G), static_cast<unsigned>(P));
        k_dft_rows_naive<<<gr, 128, 0, ctx->stream>>>(planes, row_out, static_cast<int>(G), tw,
                                                      static_cast<int>(col_lo), static_cast<int>(cols));
        SVDI_LAUNCH_CHECK();
        dim3 gc(static_cast<unsigned>((cols + 127) / 128), static_cast<unsigned>(rows), static_cast<unsigned>(P));
        k_dft_cols_naive<<<gc, 128, 0, ctx->stream>>>(row_out, out, static_cast<int>(G), tw,
                                                      static_cast<int>(cols), static_cast<int>(row_lo),
                                                      static_cast<int>(rows));
        SVDI_LAUNCH_CHECK();
        return;
    }
    // Transforms per workgroup: about kPassElems elements, so that two workgroups and more share a CU and one's
    // loads run beside the other's stages; columns at least four (32-byte row segments) unless the LDS does
    // not hold them; fewer where the workgroups would not fill the chip twice.  The threads: up to 512 with a
    // butterfly or so each, more where 512 could not hold a stage or a CU holds one workgroup.
    const int n = static_cast<int>(G);
    int held[2] = {kHoldLess, kHoldMore};          // elements per thread, the least of the stages
    for (int i = 0; i < st.count; ++i) {
        held[0] = std::min(held[0], kHoldLess / st.radix[i] * st.radix[i]);
        held[1] = std::min(held[1], kHoldMore / st.radix[i] * st.radix[i]);
    }
    const size_t one = static_cast<size_t>(pass_len(n)) * sizeof(float2), twb = G * sizeof(float2);
    auto lds_of = [&](int ntrans) { return twb + ntrans * one; };
    auto fit = [&](int most, int least, size_t transforms) {
        int ntrans = most;
        while (ntrans > least && (ntrans * n > kPassElems || transforms / ntrans < 2 * static_cast<size_t>(ctx->cu_count)))
            ntrans /= 2;
        while (ntrans > 1 && (ntrans * n > kPassThreads * std::max(held[0], held[1]) || lds_of(ntrans) > kPassLds)) ntrans /= 2;
        return ntrans;
    };
    struct Shape {
        int threads;
        bool more;                                 // kHoldMore
    };
    auto shape_of = [&](int ntrans) {
        const int elems = ntrans * n;
        Shape s = {128, false};
        while (s.threads < 512 && elems > s.threads * 8) s.threads *= 2;
        if (elems > s.threads * held[0] && elems <= s.threads * held[1]) s.more = true;
        while (elems > s.threads * held[s.more]) {
            s.more = false;
            s.threads *= 2;
            if (s.threads == kPassThreads && elems > s.threads * held[0]) s.more = true;
        }
        // (With one workgroup to a CU nothing else hides its waits: 8 planes of 5000^2 rows + columns 2.43 ms with 512 threads,
        // 2.25 so; of 7200^2 2.36 and 2.07.)
        if (s.threads < kPassThreads && 2 * lds_of(ntrans) > kPassLds) s = {kPassThreads, elems > kPassThreads * held[0]};
        return s;
    };
    auto grid_of = [&](int tiles, int ntrans, int threads) {
        const int per_cu = static_cast<int>(std::min<size_t>(kPassLds / lds_of(ntrans), 2048 / threads));
        return static_cast<unsigned>(std::min(tiles, std::max(1, ctx->cu_count * per_cu)));
    };
    const int c_lo = static_cast<int>(col_lo), nc = static_cast<int>(cols), nr = static_cast<int>(rows);
    auto launch = [&](auto less, auto more, int ntrans, int tiles, auto... args) {
        const Shape shape = shape_of(ntrans);
        const auto kernel = shape.more ? more : less;
        allow_dynamic_lds(reinterpret_cast<const void*>(kernel), lds_of(ntrans));
        kernel<<<grid_of(tiles, ntrans, shape.threads), shape.threads, lds_of(ntrans), ctx->stream>>>(args...);
        SVDI_LAUNCH_CHECK();
    };
    const int total_rows = static_cast<int>(P * G), batch = fit(16, 1, P * G), row_tiles = (total_rows + batch - 1) / batch;
    launch(&k_fft_rows<kHoldLess>, &k_fft_rows<kHoldMore>, batch, row_tiles, planes, row_out, st, tw, total_rows, batch,
           row_tiles, c_lo, nc);
    const int width = fit(8, 4, P * cols), strips = (nc + width - 1) / width, col_tiles = strips * static_cast<int>(P);
    launch(&k_fft_cols<kHoldLess>, &k_fft_cols<kHoldMore>, width, col_tiles, static_cast<const float2*>(row_out), out, st, tw,
           width, strips, col_tiles, nc, static_cast<int>(row_lo), nr);
}

}  // namespace svdi
