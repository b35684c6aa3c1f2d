// MFMA gridder: the ES gridding of Chebyshev moments (fused_gridding, SVDIntegratedImager.cu:
// 1218-1293; gridding, archive/FIPkernels.cu:391-452) recast as dense contractions over
// output-stationary 16 x 16 windows of the grid.
//
// For a window W and the samples r whose footprint meets it, every (term k, re/im, cell) of W is
//   D[m][(a, b)] = sum_r c[m][r] * ku_r[a] * kv_r[b],   m = 2k + ri,
//   c[2k + ri][r] = T_k(s_r) * (Re | Im) v_r / |det|,   ku_r[a] = ES((a - p1_r) / 4) (0 off support),
// with (a, b) the window's cells and p_r the sample's position relative to the window.  For each
// window row a, D_a = C * B_a runs on v_mfma_f32_16x16x32_f16, with C = c (16 x 32 samples) and
// B_a[r][b] = ku_r[a] kv_r[b] (32 samples x 16 columns), the 16 row blocks (64 FP32 accumulators
// per lane) staying in registers across the window's samples.  Half windows that hold many samples
// are contracted by workgroups instead, sorted by footprint column (k_win_dense); their partial
// sums are added in piece order by k_win_reduce, and no atomics touch the planes.
// Precision: c and the ES factors are split into f16 hi + lo and each product taken as
// hi*hi + lo*hi + hi*lo with FP32 accumulation (~22 significant bits per product); c is scaled by
// a power of two fixed from the largest |v| of the call and the ES factors by 2^7 each, so
// nothing overflows f16; the scales are undone exactly at write-out.
//
// Binning by row class: with class height c (4, or 8 when the finer histogram does not fit in
// LDS), a sample whose (clipped) first footprint row a0 lies in [c h, c h + c) is in row class h,
// and its footprint rows lie in [c h, c h + c + 8).  Window row wa (rows [16 wa, 16 wa + 16))
// therefore reads the 24 / c classes h = (16 / c) wa + d, d = -8 / c .. 16 / c - 1, class d
// touching only the window rows [c d, c d + c + 7].  Records are binned by (slab, window
// column, row class) with the class fastest, so a window's records are one contiguous range
// ordered by class, each record is written once per window column it meets, and a chunk of 32
// records drawn from neighbouring classes skips the 4-row quarters of the window that none of
// them touches (with c = 4, 12 of 16 rows per class).  Counting uses block-local
// LDS histograms kept per block; a prefix over the blocks and a scan of the bin totals give each
// block its first slot in every bin, and one more pass over its samples writes the records
// (position relative to the class's home window row / the window column, s, v).  When the bins
// do not fit in one LDS histogram, runs of eight classes are binned together first and each such
// coarse bin's records are then sorted by class (k_sub_bins).  Coarse bins that still do not fit are
// split into bands of consecutive bins, and each band is a separate set of workgroups that reads the
// block's samples and handles only its own bins.
#include "sample.hpp"
#include "scan.hpp"
#include "es_poly.hpp"
#include "records.hpp"
#include "work_shape.hpp"

#include <cstring>
#include <type_traits>

namespace svdi {
namespace {

constexpr int kWin = 16;                 // window side in cells
constexpr int kMaxClasses = 6;           // classes per window: 24 / class height (4 or 8)
constexpr int kBinThreads = 1024;        // binning blocks
constexpr int kBinRowsLeast = 64, kBinRowsMost = 512;   // rows of a block, snapshot input
constexpr int kBinPerThreadMost = 16;    // samples per thread, preprocessed input: 1 .. 16
constexpr int kLdsBins = 36864;          // largest block-local histogram (144 KB of LDS)
constexpr size_t kMaxBlockHistBytes = size_t(1) << 31;   // per-block histograms of all bands
constexpr int kSupLog2 = 3;              // row classes binned together when the bins pass kLdsBins
constexpr int kSup = 1 << kSupLog2;
constexpr int kChunk = 32;               // samples per MFMA reduction step
constexpr int kStride = 36;              // floats per c staging row (32 samples + pad)
constexpr int kStrideH = 40;             // halves per ES staging row (32 samples + pad, 16-byte rows)
constexpr int kPad = 8;                  // ES staging rows beyond each window edge (-8 .. 23)
constexpr int kStageRows = kWin + 2 * kPad;
constexpr int kPlaneHalves = kStageRows * kStrideH;               // one ES plane (hi or lo)
constexpr int kEsScaleLog2Sq = 14;      // ES factors scaled by 2^7 per axis (in the polynomial table)

// Operand precision of the window contraction D_a += C B_a (C = c, B_a = ku_a kv).
enum WinPrec : int {
    kPrecSplit3 = 0,   // c and both ES factors in f16 hi + lo; B_a's product error kept:
                       // hi*hi + lo*hi + hi*lo, ~22 significant bits per product, 3 MFMAs per row
    kPrecSplitC = 1,   // c in f16 hi + lo, B_a = f16(f16(ku) f16(kv)): 2 MFMAs per row
    kPrecSingle = 2,   // c and B_a single f16: 1 MFMA per row
    kPrecBf16 = 3,     // c and B_a in bf16 hi + lo, B_a's product formed in FP32: hi*hi + lo*hi +
                       // hi*lo on the bf16 MFMA, ~16 significant bits per product
};
constexpr int kStrideF = 36;                               // floats per FP32 ES staging row
constexpr int kPlaneFloats = kStageRows * kStrideF;        // one FP32 ES plane
template <int P>
struct WinTraits {
    static constexpr bool kBf16 = P == kPrecBf16;          // FP32 ES planes, bf16 operands
    static constexpr bool kEsLo = P == kPrecSplit3;        // ES factors staged as f16 hi + lo planes
    static constexpr bool kCLo = P != kPrecSingle;         // c split into hi + lo
    static constexpr bool kDither = P == kPrecSplitC || P == kPrecSingle;   // single-f16 ES product
    static constexpr int kPlanes = kEsLo ? 4 : 2;
    // Per wavefront: the ES planes (ku hi [lo], kv hi [lo], f16; or ku, kv in FP32), then c[16]
    // (f32).
    static constexpr int kStageFloats =
        (kBf16 ? 2 * kPlaneFloats : (kPlanes * kPlaneHalves) / 2) + kWin * kStride;
    // Wavefronts per workgroup (one workgroup per CU): as many as the staging allows.  At 12 the
    // kernel keeps its ~150 registers without spills; 16 (four per SIMD) would need 128 and a
    // staging area without row padding, which measured slower (542 against 500 us for split3).
    static constexpr int kWaves = (kEsLo || kBf16) ? 12 : 16;
};
// ES(1) 2^7, the ninth footprint cell of an integer position, as f16 hi + lo.
constexpr _Float16 kEsPolyEdgeHi = static_cast<_Float16>(kEsPolyEdge);
constexpr _Float16 kEsPolyEdgeLo = static_cast<_Float16>(kEsPolyEdge - static_cast<float>(kEsPolyEdgeHi));

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

struct WinGeom {
    int nw;          // windows per grid axis
    int cls_log2;    // log2 of the row-class height (2 or 3)
    int ncls;        // classes per window: 24 >> cls_log2
    int nh;          // row classes: ceil(G / class height)
    int nwin;        // nw * nw
    int nwin_total;  // nslabs * nwin
    int nbins;       // nslabs * nw * nh, ordered (slab, window column, row class)
    int sup_log2;    // log2 of the row classes that are binned together (0, or kSupLog2)
    int sup_rows;    // ceil(nh / 2^sup_log2)
    int lbins;       // bins of the count and scatter passes: nslabs * nw * sup_rows
    int use_lds;     // block histograms in LDS (else one global atomic per record)
    int band_bins;   // bins per LDS band (<= kLdsBins); band y covers [y band_bins, ...) of lbins
    int block_size;  // binning blocks: rows (snapshot input), samples per thread (preprocessed)
    int set_rows;    // rows of a block read at a time (64 or 256; snapshot rows read one by one)
    WorkShape shape;     // records above which a half is dense, and per workgroup piece (asked for; fit_shape)
    uint32_t slots;      // partial slots (kAllSlotsFit: enough for any sizes of the halves)
};

// A work item of window `win`.  slot < 0: a wavefront item, the `count` records from `start` on
// that are not among [hole, hole + hole_len); bnd[j] (j = 1 .. ncls - 1) is the first record of the
// window's class j (d = j - 8 / c), records before bnd[1] are of class 0, and bnd[j] for j >= ncls
// is the window's end; skip (bits 0, 1, 2: the half above, the lower half, the upper half): records
// with a negative first column are skipped.  slot >= 0: the piece [start, start + count) of half
// `half`, whose share goes to partial slot `slot`; skip (0 or 1) as above.
struct WItem {
    int win, start, count, slot;
    int bnd[kMaxClasses];
    int hole, hole_len, half, skip;
    __device__ __forceinline__ int record(int j) const {      // absolute index of the item's record j
        const int i = start + j;
        return i + (i >= hole ? hole_len : 0);
    }
};

// Records: 16 bytes each (records.hpp), one aligned 16-byte access to write or read.
struct WRecords {
    uint4* r;

    __device__ __forceinline__ void put(uint32_t slot, const RecordWords& w) const {
        r[slot] = make_uint4(w.w[0], w.w[1], w.w[2], w.w[3]);
    }
    __device__ __forceinline__ uint4 get(int i) const { return r[i]; }
};

// Every (sample, bin) pair of this block's samples: one row class h = a0 / c (c the class
// height), and the window columns b0 / 16 .. (b0 + nb - 1) / 16 that the clipped footprint meets
// (at most two).  Snapshot input: block_size consecutive rows, in sets of set_rows, each row split over
// kBinThreads / set_rows threads that take every so many channels (a wavefront reads 64 consecutive
// rows of one channel: coalesced), loading four samples before working on the first.  Preprocessed
// input: block_size consecutive samples per thread, at a stride of kBinThreads.  kVis = false (snapshot
// input): neither visibilities nor weights are loaded and f.vw is zero; the bins depend on flags
// and geometry only (samples are kept unless both polarisations are flagged, V = 0 when the
// weights sum to zero), so both passes keep the same samples.
template <bool kSnap, bool kVis, class Fn>
__device__ __forceinline__ void for_sample_bins(const SampleInput& in, const GridParams& gp,
                                                const WinGeom& wg, size_t blk, Fn&& fn) {
    auto bins_of = [&](const Footprint& f) {
        // (a0, b0 >= 0: array coordinates of an in-grid footprint.)
        const int h = f.a0 >> wg.cls_log2;
        const int col0 = f.local_slab * wg.nw;
        const int wb0 = static_cast<int>(static_cast<uint32_t>(f.b0) / kWin);
        const int wb1 = static_cast<int>(static_cast<uint32_t>(f.b0 + f.nb - 1) / kWin);
        for (int wb = wb0; wb <= wb1; ++wb) fn(f, (col0 + wb) * wg.sup_rows + (h >> wg.sup_log2), h, wb);
    };
    if constexpr (kSnap) {
        if (in.quad_rows) {
            // Four consecutive rows of one channel per thread (one 16-byte load per FP32 array, which needs no
            // more than 4-byte alignment, and one of 4 bytes per flag array), block_size / 4 row quads x
            // as many channel groups as the threads are enough for; the next channel's loads are issued before
            // this one is binned.  The last quad of a row count that is not a multiple of 4 starts earlier and
            // leaves out the rows of the quad before it.  (5.2 M samples in 81,103 rows: scatter + count 128 us
            // one row per thread, 119 so.)
            const uint32_t quads = static_cast<uint32_t>(wg.block_size) / 4, quad_groups = kBinThreads / quads;
            const uint32_t group = threadIdx.x / quads;
            const size_t quad0 = blk * wg.block_size + 4 * (threadIdx.x - group * quads);
            if (group >= quad_groups || quad0 >= in.num_rows) return;
            const size_t row0 = min(quad0, in.num_rows - 4);
            const int first = static_cast<int>(quad0 - row0);
            struct QuadLoad {
                double nu;
                float4 v0r, v0i, v3r, v3i, w0, w3;
                uint32_t f0, f3;
            };
            const float4 one4 = make_float4(1.0f, 1.0f, 1.0f, 1.0f), zero4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            auto load = [&](size_t chan) {
                QuadLoad q;
                const size_t idx = row0 + chan * in.num_rows;
                q.nu = in.freq[chan];
                q.v0r = q.v0i = q.v3r = q.v3i = zero4;
                q.w0 = q.w3 = one4;
                if constexpr (kVis) {
                    __builtin_memcpy(&q.v0r, in.v0r + idx, 16);
                    __builtin_memcpy(&q.v0i, in.v0i + idx, 16);
                    __builtin_memcpy(&q.v3r, in.v3r + idx, 16);
                    __builtin_memcpy(&q.v3i, in.v3i + idx, 16);
                    if (in.w0) __builtin_memcpy(&q.w0, in.w0 + idx, 16);
                    if (in.w3) __builtin_memcpy(&q.w3, in.w3 + idx, 16);
                }
                __builtin_memcpy(&q.f0, in.f0 + idx, 4);
                __builtin_memcpy(&q.f3, in.f3 + idx, 4);
                return q;
            };
            auto lane4 = [](const float4& v, int r) { return r == 0 ? v.x : r == 1 ? v.y : r == 2 ? v.z : v.w; };
            size_t chan = group;
            if (chan >= in.num_channels) return;
            QuadLoad cur = load(chan);
            double geo[4][3];
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int k = 0; k < 3; ++k) geo[r][k] = in.rot[3 * (row0 + r) + k];
            for (; chan < in.num_channels; chan += quad_groups) {
                QuadLoad nxt = cur;
                if (chan + quad_groups < in.num_channels) nxt = load(chan + quad_groups);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (r < first) continue;
                    SnapLoad s;
                    s.nu = cur.nu;
                    s.v0r = lane4(cur.v0r, r);
                    s.v0i = lane4(cur.v0i, r);
                    s.v3r = lane4(cur.v3r, r);
                    s.v3i = lane4(cur.v3i, r);
                    s.w0 = lane4(cur.w0, r);
                    s.w3 = lane4(cur.w3, r);
                    s.f0 = static_cast<uint8_t>(cur.f0 >> (8 * r));
                    s.f3 = static_cast<uint8_t>(cur.f3 >> (8 * r));
                    Footprint f;
                    if (finish_snapshot_sample<true>(gp, geo[r][0], geo[r][1], geo[r][2], s, f)) bins_of(f);
                }
                cur = nxt;
            }
            return;
        }
        constexpr int kBatch = 4;
        const uint32_t groups = kBinThreads / static_cast<uint32_t>(wg.set_rows);
        for (int set = 0; set < wg.block_size; set += wg.set_rows) {
        const size_t row = blk * wg.block_size + set + (threadIdx.x & (wg.set_rows - 1));
        if (row >= in.num_rows) return;
        const double ru = in.rot[3 * row], rv = in.rot[3 * row + 1], rw = in.rot[3 * row + 2];
        for (size_t c0 = threadIdx.x / static_cast<uint32_t>(wg.set_rows); c0 < in.num_channels; c0 += kBatch * groups) {
            SnapLoad ld[kBatch] = {};
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                const size_t chan = c0 + u * groups;
                if (chan < in.num_channels) ld[u] = load_snapshot_sample<kVis, kVis>(in, row + chan * in.num_rows, chan);
            }
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                const size_t chan = c0 + u * groups;
                Footprint f;
                if (chan < in.num_channels && finish_snapshot_sample<true>(gp, ru, rv, rw, ld[u], f)) bins_of(f);
            }
        }
        }
    } else {
        const size_t base = blk * kBinThreads * wg.block_size + threadIdx.x;
        for (int j = 0; j < wg.block_size; ++j) {
            const size_t idx = base + static_cast<size_t>(j) * kBinThreads;
            if (idx >= in.num_samples) return;
            Footprint f;
            if (setup_sample<false>(in, gp, idx, 0, 0, f)) bins_of(f);
        }
    }
}

// Largest |Re v|, |Im v| of the block, folded into *vmax_bits (non-negative floats order as
// their bit patterns).
__device__ __forceinline__ void block_max_to(float m, uint32_t* vmax_bits) {
    __shared__ float s_max[kBinThreads / 64];
    for (int d = 32; d >= 1; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
    if ((threadIdx.x & 63) == 0) s_max[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        float b = s_max[0];
        for (int w = 1; w < kBinThreads / 64; ++w) b = fmaxf(b, s_max[w]);
        if (b > 0.0f && b <= 3.0e38f) atomicMax(vmax_bits, __float_as_uint(b));
    }
}

// Sum of v over the block's kBinThreads threads, returned to every thread (once per kernel).
__device__ __forceinline__ uint32_t block_sum(uint32_t v) {
    __shared__ uint32_t s_part[kBinThreads / 64];
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = v;
    __syncthreads();
    uint32_t t = 0;
    for (int w = 0; w < kBinThreads / 64; ++w) t += s_part[w];
    return t;
}

// Bins [lo, lo + n) of LDS band blockIdx.y.
__device__ __forceinline__ void lds_band(const WinGeom& wg, int& lo, int& n) {
    lo = static_cast<int>(blockIdx.y) * wg.band_bins;
    n = min(wg.band_bins, wg.lbins - lo);
}

// Bin counts: per (block, band) in an LDS histogram (dynamic LDS) written to
// blockhist[block * lbins + bin] for the band's bins, and the (block, band)'s record total to
// blocktot[band * blocks + block] (without LDS histograms the counts go straight to counts[bin]).
// kHist16: 16-bit counters, two bins per LDS word (bin b in the half b & 1 of word b / 2, added
// to by a 32-bit atomic of 1 << 16 (b & 1)), for blocks of fewer than 65536 samples: a sample
// adds at most one record to a bin, so no half carries into the other.  Half the LDS lets two
// workgroups share a CU.
template <bool kSnap, bool kHist16, typename CountT>
__global__ void __launch_bounds__(kBinThreads)
k_win_count(SampleInput in, GridParams gp, WinGeom wg, uint32_t* __restrict__ counts,
            CountT* __restrict__ blockhist, uint32_t* __restrict__ blocktot) {
    take_device_plan(gp);
    extern __shared__ uint32_t hist[];
    const size_t blk = blockIdx.x;
    if (!wg.use_lds) {
        for_sample_bins<kSnap, false>(in, gp, wg, blk, [&](const Footprint&, int bin, int, int) {
            atomicAdd(&counts[bin], 1u);
        });
        return;
    }
    int lo, n;
    lds_band(wg, lo, n);
    const int words = kHist16 ? (n + 1) / 2 : n;
    for (int w = threadIdx.x; w < words; w += kBinThreads) hist[w] = 0;
    __syncthreads();
    uint32_t cnt = 0;
    for_sample_bins<kSnap, false>(in, gp, wg, blk, [&](const Footprint&, int bin, int, int) {
        const uint32_t b = static_cast<uint32_t>(bin - lo);
        if (b < static_cast<uint32_t>(n)) {
            if constexpr (kHist16) atomicAdd(&hist[b >> 1], 1u << ((b & 1u) << 4));
            else atomicAdd(&hist[b], 1u);
            ++cnt;
        }
    });
    const uint32_t tot = block_sum(cnt);          // (its barrier also ends the histogram's atomics)
    if (threadIdx.x == 0) blocktot[static_cast<size_t>(blockIdx.y) * gridDim.x + blk] = tot;
    CountT* row = blockhist + blk * wg.lbins + lo;
    for (int b = threadIdx.x; b < n; b += kBinThreads)
        row[b] = static_cast<CountT>(kHist16 ? (hist[b >> 1] >> ((b & 1) << 4)) & 0xffffu : hist[b]);
}

// The per-block histograms turned into per-block record offsets without global atomics per
// (block, bin): the blocks are split into kBinSegs segments; k_bin_seg_sums forms each segment's
// count of every bin (and the bin totals), and after the scan of the totals k_bin_block_offsets
// writes offs[block][bin] = boff[bin] + the records of the bin in earlier blocks.  Each block's
// records of a bin therefore follow those of the blocks before it.  The counts are 16-bit when a
// block has fewer than 65536 samples (half the histogram traffic), and otherwise 32-bit words
// that the offsets then replace in place.
constexpr int kBinSegs = 8;

__device__ __forceinline__ void bin_segment(int nblocks, int seg, int& b0, int& b1) {
    const int per = (nblocks + kBinSegs - 1) / kBinSegs;
    b0 = min(seg * per, nblocks);
    b1 = min(b0 + per, nblocks);
}

template <typename CountT>
__global__ void __launch_bounds__(256)
k_bin_seg_sums(const CountT* __restrict__ blockhist, int nblocks, int nbins, uint32_t* __restrict__ segsum,
               uint32_t* __restrict__ counts) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= kBinSegs * nbins) return;
    const int seg = t / nbins, bin = t - seg * nbins;
    int b0, b1;
    bin_segment(nblocks, seg, b0, b1);
    const CountT* p = blockhist + bin;
    uint32_t sum = 0;
    int b = b0;
    for (; b + 8 <= b1; b += 8) {
        uint32_t v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = p[static_cast<size_t>(b + j) * nbins];
#pragma unroll
        for (int j = 0; j < 8; ++j) sum += v[j];
    }
    for (; b < b1; ++b) sum += p[static_cast<size_t>(b) * nbins];
    segsum[t] = sum;
    if (sum != 0) atomicAdd(&counts[bin], sum);
}

// The dense halves counted by size for fit_shape, half t by thread t of workgroups of 256; words: kShapeWords, zero
// before.
inline unsigned half_size_blocks(const WinGeom& wg) { return (2u * static_cast<unsigned>(wg.nwin_total) + 255) / 256; }
__device__ __forceinline__ void count_half_sizes(const uint32_t* __restrict__ boff, const WinGeom& wg, uint32_t* __restrict__ words) {
    __shared__ uint32_t s_words[kShapeWords];
    for (int i = threadIdx.x; i < kShapeWords; i += 256) s_words[i] = 0u;
    __syncthreads();
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t < 2 * wg.nwin_total) {
        const int per = 8 >> wg.cls_log2, col = t / (2 * wg.nw), h = (t - col * 2 * wg.nw) * per;
        const uint32_t* b = boff + static_cast<size_t>(col) * wg.nh;
        const uint32_t n = b[min(h + per, wg.nh)] - b[min(h, wg.nh)];
        if (n > wg.shape.coop_min) {
            const int k = 2 + 2 * shape_bucket(wg.shape.coop_min, n);
            atomicAdd(&s_words[0], 1u);
            atomicAdd(&s_words[1], n);
            atomicAdd(&s_words[k], 1u);
            atomicAdd(&s_words[k + 1], n);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kShapeWords; i += 256)
        if (s_words[i] != 0) atomicAdd(&words[i], s_words[i]);
}
__global__ void __launch_bounds__(256)
k_win_half_sizes(const uint32_t* __restrict__ boff, WinGeom wg, uint32_t* __restrict__ words) {
    count_half_sizes(boff, wg, words);
}

// cnt and offs may be the same words (32-bit counts): each is read before it is written.  The first size_blocks
// workgroups count the halves' sizes instead (boff holds the bins' offsets then).
template <typename CountT>
__global__ void __launch_bounds__(256)
k_bin_block_offsets(const CountT* cnt, uint32_t* offs, int nblocks, int nbins, const uint32_t* __restrict__ segsum,
                    const uint32_t* __restrict__ boff, unsigned size_blocks, WinGeom wg, uint32_t* __restrict__ words) {
    if (blockIdx.x < size_blocks) {
        count_half_sizes(boff, wg, words);
        return;
    }
    const int t = (blockIdx.x - size_blocks) * 256 + threadIdx.x;
    if (t >= kBinSegs * nbins) return;
    const int seg = t / nbins, bin = t - seg * nbins;
    int b0, b1;
    bin_segment(nblocks, seg, b0, b1);
    uint32_t run = boff[bin];
    for (int s = 0; s < seg; ++s) run += segsum[s * nbins + bin];
    const CountT* p = cnt + bin;
    uint32_t* o = offs + bin;
    int b = b0;
    for (; b + 8 <= b1; b += 8) {
        uint32_t v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = p[static_cast<size_t>(b + j) * nbins];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            o[static_cast<size_t>(b + j) * nbins] = run;
            run += v[j];
        }
    }
    for (; b < b1; ++b) {
        const uint32_t v = p[static_cast<size_t>(b) * nbins];
        o[static_cast<size_t>(b) * nbins] = run;
        run += v;
    }
}

// Records of this block's samples, in one pass per band: with LDS histograms the block's first
// slot of each of the band's bins comes from blockhist (the offsets of k_bin_block_offsets) and
// LDS cursors hand out the slots; otherwise every record takes a global cursor slot.
// `limit` (the record buffer's capacity) only bounds the writes.  With LDS histograms the
// (block, band)'s emitted records are checked against its count-pass total: a difference (the
// inputs changed between the passes) would leave slots unwritten, so it sets kErrBinMismatch in
// *err and the call fails instead of gridding stale records.
template <bool kSnap>
__global__ void __launch_bounds__(kBinThreads)
k_win_scatter(SampleInput in, GridParams gp, WinGeom wg, const uint32_t* __restrict__ blockhist,
              const uint32_t* __restrict__ blocktot, uint32_t* __restrict__ cursor, WRecords rec,
              uint32_t limit, uint32_t* __restrict__ vmax_bits, uint32_t* __restrict__ err) {
    take_device_plan(gp);
    extern __shared__ uint32_t hist[];
    const int off = gp.G / 2;
    float m = 0.0f;
    auto emit = [&](uint32_t slot, const Footprint& f, int h, int wb) {
        m = fmaxf(m, fmaxf(fabsf(f.vw.x), fabsf(f.vw.y)));
        if (slot >= limit) return;
        // Row position relative to the class's home window row (c h + 8) / 16: the row window
        // that reads the class at d < 8 / c (the row above reads it at d >= 8 / c).  Snapshot
        // input: q = p - (first footprint cell); preprocessed input: q = p (centred).
        const int home = ((h << wg.cls_log2) + 8) >> 4;
        const int base1 = kSnap ? f.a0 - home * kWin : off - home * kWin;
        const int base2 = kSnap ? f.b0 - wb * kWin : off - wb * kWin;
        RecordWords w = rec_encode(base1, f.q1, base2, f.q2, f.s, f.vw.x, f.vw.y);
        // A negative first column marks the copy of a record whose home is the window to the left.  A
        // position just above an integer that the encoding rounds to it (first cell one lower, F = 0)
        // keeps its home's first cell 0, with the largest fraction instead.
        if (wb > 0 && f.b0 >= wb * kWin && static_cast<int32_t>(w.w[3]) < 0)
            w.w[3] = (((1u << kRecFracBits) - 1u) << 8) | (w.w[3] & 0xffu);
        if (wg.sup_log2 != 0)
            rec_to_coarse(w, kWin * home - ((h >> wg.sup_log2) << (wg.sup_log2 + wg.cls_log2)));
        rec.put(slot, w);
    };
    const size_t blk = blockIdx.x;
    if (!wg.use_lds) {
        for_sample_bins<kSnap, true>(in, gp, wg, blk, [&](const Footprint& f, int bin, int h, int wb) {
            emit(atomicAdd(&cursor[bin], 1u), f, h, wb);
        });
        block_max_to(m, vmax_bits);
        return;
    }
    int lo, n;
    lds_band(wg, lo, n);
    const uint32_t* row = blockhist + blk * wg.lbins + lo;
    for (int b = threadIdx.x; b < n; b += kBinThreads) hist[b] = row[b];
    __syncthreads();
    uint32_t cnt = 0;
    for_sample_bins<kSnap, true>(in, gp, wg, blk, [&](const Footprint& f, int bin, int h, int wb) {
        const uint32_t b = static_cast<uint32_t>(bin - lo);
        if (b < static_cast<uint32_t>(n)) {
            emit(atomicAdd(&hist[b], 1u), f, h, wb);
            ++cnt;
        }
    });
    const uint32_t tot = block_sum(cnt);
    if (threadIdx.x == 0 && tot != blocktot[static_cast<size_t>(blockIdx.y) * gridDim.x + blk])
        atomicOr(err, kErrBinMismatch);
    block_max_to(m, vmax_bits);
}

// The records of the coarse bins (kSup row classes of a window column) sorted by class, and the
// offsets boff of all bins.  A wavefront takes a piece of at most kSubPiece records of one coarse
// bin into registers, ranks the records of each class by ballots and writes them to the class's range.
// A coarse bin of one piece needs nothing else; the classes of larger ones are counted first
// (kCount) in cls, and `used` hands out their slots to the pieces.  k_sub_list lists the pieces, those
// of the larger coarse bins from the front and the others from the back, so that the wavefronts share
// the few coarse bins near the uv centre, with thousands of pieces, evenly (16.7 M samples at 4096^2: 343 us;
// given out by a fixed rule over groups of 256 coarse bins 543).
// Bound by HBM: records read once (twice in coarse bins of several pieces) and written once.
constexpr int kSubLoads = 8;
constexpr int kSubPiece = 64 * kSubLoads;
constexpr int kSubWaves = 4;             // wavefronts per workgroup
constexpr int kSubGroupsPerCu = 4;

// (bin, first record of the bin, piece number, records of the piece; pieces of one-piece coarse bins,
// empty ones among them, are at the list's end.)
struct SubPiece {
    uint32_t bin, lo, piece, n;
};

// counts[0], [1]: pieces listed from the front and from the back.  A coarse bin of n records has
// max(1, ceil(n / kSubPiece)) pieces, so `cap` = lbins + max_records / kSubPiece holds them all.
__global__ void __launch_bounds__(256)
k_sub_list(const uint32_t* __restrict__ coff, WinGeom wg, uint32_t limit, SubPiece* __restrict__ list, uint32_t cap,
           uint32_t* __restrict__ counts, uint32_t* __restrict__ boff) {
    const int bin = blockIdx.x * 256 + threadIdx.x, lane = threadIdx.x & 63;
    if (bin == 0) boff[wg.nbins] = coff[wg.lbins];
    uint32_t lo = 0, n = 0;
    if (bin < wg.lbins) {
        lo = min(coff[bin], limit);
        n = min(coff[bin + 1], limit) - lo;
    }
    const bool single = bin < wg.lbins && n <= static_cast<uint32_t>(kSubPiece);
    const uint64_t singles = __ballot(single);
    uint32_t base = 0;
    if (lane == 0 && singles != 0) base = atomicAdd(&counts[1], static_cast<uint32_t>(__popcll(singles)));
    base = __builtin_amdgcn_readfirstlane(base);
    if (single) {
        const uint32_t at = base + __popcll(singles & ((1ull << lane) - 1));
        if (at < cap) list[cap - 1 - at] = {static_cast<uint32_t>(bin), lo, 0u, n};
    }
    // The larger ones' pieces: one reservation per wavefront, then all its lanes list a coarse bin's.
    const uint32_t pieces = bin < wg.lbins && !single ? (n + kSubPiece - 1) / kSubPiece : 0u;
    uint32_t incl = pieces;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t v = __shfl_up(incl, d, 64);
        if (lane >= d) incl += v;
    }
    base = 0;
    if (lane == 63 && incl != 0) base = atomicAdd(&counts[0], incl);
    const uint32_t first = __builtin_amdgcn_readlane(base, 63) + incl - pieces;
    uint64_t todo = __ballot(pieces != 0);
    while (todo != 0) {
        const int i = __builtin_ctzll(todo);
        todo &= todo - 1;
        const uint32_t b_lo = __builtin_amdgcn_readlane(lo, i), b_n = __builtin_amdgcn_readlane(n, i);
        const uint32_t b_first = __builtin_amdgcn_readlane(first, i), b_pieces = __builtin_amdgcn_readlane(pieces, i);
        for (uint32_t p = lane; p < b_pieces; p += 64)
            if (b_first + p < cap)
                list[b_first + p] = {static_cast<uint32_t>(bin - lane + i), b_lo, p,
                                     min(b_n - p * kSubPiece, static_cast<uint32_t>(kSubPiece))};
    }
}

template <bool kCount>
__global__ void __launch_bounds__(kSubWaves * 64)
k_sub_bins(const SubPiece* __restrict__ list, uint32_t cap, const uint32_t* __restrict__ counts, WinGeom wg,
           const uint4* __restrict__ coarse, uint32_t* __restrict__ cls, uint32_t* __restrict__ used,
           uint32_t* __restrict__ boff, WRecords rec, uint32_t limit) {
    const int lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * kSubWaves + (threadIdx.x >> 6));
    const uint32_t nwaves = gridDim.x * kSubWaves;
    const int my = lane & (kSup - 1);                      // the class that this lane counts
    const uint32_t multi = min(counts[0], cap);
    const uint32_t total = kCount ? multi : min(multi + counts[1], cap);
    // Lanes of class c among those whose class bits are (b0, b1, b2).
    auto among = [](uint64_t b0, uint64_t b1, uint64_t b2, int c) {
        return ((c & 1) ? b0 : ~b0) & ((c & 2) ? b1 : ~b1) & ((c & 4) ? b2 : ~b2);
    };
    auto piece = [&](uint32_t t) { return list[t < multi ? t : cap - 1 - (t - multi)]; };
    auto load = [&](const SubPiece& s, uint4 (&q)[kSubLoads]) {
        const uint4* src = coarse + s.lo + s.piece * kSubPiece;
#pragma unroll
        for (int r = 0; r < kSubLoads; ++r)
            if (64u * r + lane < s.n) q[r] = src[64 * r + lane];
    };
    uint32_t t = wave;
    if (t >= total) return;
    SubPiece s = piece(t), s_next = s;
    uint4 q[kSubLoads];
    load(s, q);
    if (t + nwaves < total) s_next = piece(t + nwaves);
    for (;;) {
        // The classes, then (the row cells are not needed for anything else) the records as they are
        // written, so that the next piece's loads can be requested behind them.
        int c[kSubLoads];
        uint32_t cnt = 0;
        const int col = static_cast<int>(s.bin) / wg.sup_rows, sup = static_cast<int>(s.bin) - col * wg.sup_rows;
#pragma unroll
        for (int r = 0; r < kSubLoads; ++r) {
            const bool valid = 64u * r + lane < s.n;
            c[r] = valid ? min(max(rec_coarse_row(q[r].z, q[r].w) >> wg.cls_log2, 0), kSup - 1) : 0;
            const uint64_t b0 = __ballot(c[r] & 1), b1 = __ballot(c[r] & 2), b2 = __ballot(c[r] & 4);
            cnt += __popcll(among(b0, b1, b2, my) & __ballot(valid));
        }
        if constexpr (kCount) {
            if (lane < kSup && cnt != 0) atomicAdd(&cls[kSup * s.bin + lane], cnt);
        } else {
            const bool single = t >= multi;
            const uint32_t tot = single ? cnt : cls[kSup * s.bin + my];
            uint32_t start = s.lo;                         // first slot of class `my`
#pragma unroll
            for (int k = 0; k < kSup - 1; ++k) {
                const uint32_t u = __builtin_amdgcn_readlane(tot, k);
                start += my > k ? u : 0u;
            }
            const int h = kSup * sup + my;
            if (s.piece == 0 && lane < kSup && h < wg.nh) boff[col * wg.nh + h] = start;
            if (!single && lane < kSup && cnt != 0) start += atomicAdd(&used[kSup * s.bin + lane], cnt);
#pragma unroll
            for (int r = 0; r < kSubLoads; ++r) {
                const bool valid = 64u * r + lane < s.n;
                const uint64_t b0 = __ballot(c[r] & 1), b1 = __ballot(c[r] & 2), b2 = __ballot(c[r] & 4);
                const uint64_t in = __ballot(valid);
                const uint64_t same = among(b0, b1, b2, c[r]) & in;
                const uint32_t rank = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(same >> 32),
                                                                __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(same), 0u));
                const uint32_t slot = __shfl(start, c[r], 64) + rank;
                if (valid && slot < limit) {
                    const int h0 = kSup * sup + c[r];
                    RecordWords w = {{q[r].x, q[r].y, q[r].z, q[r].w}};
                    rec_from_coarse(w, ((kSup * sup) << wg.cls_log2) - ((((h0 << wg.cls_log2) + 8) >> 4) * kWin));
                    rec.put(slot, w);
                }
                start += __popcll(among(b0, b1, b2, my) & in);
            }
        }
        t += nwaves;
        if (t >= total) break;
        s = s_next;
        load(s, q);
        if (t + nwaves < total) s_next = piece(t + nwaves);
    }
}

// Record range of window w (slab, wa, wb): bnd[j] = first record of the window's class j
// (h = (16 / c) wa - 8 / c + j, clamped to the column's classes [0, nh)), j = 0 .. ncls;
// bnd[0] = start, bnd[j] = end for j >= ncls.
struct WinRange {
    uint32_t bnd[kMaxClasses + 1];
    __device__ uint32_t start() const { return bnd[0]; }
};
__device__ __forceinline__ WinRange window_range(const uint32_t* __restrict__ boff, const WinGeom& wg, int w, uint32_t& end) {
    const int ls = w / wg.nwin, r = w - ls * wg.nwin;
    const int wa = r / wg.nw, wb = r - wa * wg.nw;
    const int base = (ls * wg.nw + wb) * wg.nh;
    const int h0 = (wa << (4 - wg.cls_log2)) - (8 >> wg.cls_log2);
    WinRange x;
#pragma unroll
    for (int j = 0; j <= kMaxClasses; ++j)
        x.bnd[j] = boff[base + min(max(h0 + min(j, wg.ncls), 0), wg.nh)];
    end = x.bnd[wg.ncls];
    return x;
}

// Work items.  A window's home records are those of the 16 / c classes whose first footprint row
// lies in the window; its halves are the two runs of classes of first rows 0 .. 7 and 8 .. 15.  A
// half with more than coop_min home records is dense: k_win_dense takes them, in pieces of at
// most coop_cap records, a workgroup each, and writes each piece's share of the 16 rows and 24
// columns that its footprints reach (the lower eight rows of the upper half and the last eight
// columns lie in the windows below and to the right) to a partial slot.  Every other record is read
// by the wavefront items of k_win_grid, one per window: the halves that are not dense and the
// upper half of the window above unless that is.  Either way the copies of records whose home is
// a dense half of the window to the left (negative first column) are skipped.  k_win_reduce then
// adds the partial slots, in piece order, to the windows that dense pieces reach (a window with
// no other records gets no wavefront item).  Both queues run largest first, by octave classes: class c
// holds items with count * 2^c <= cap < count * 2^(c+1) (cap = 3 coop_min for wavefront items,
// coop_cap for pieces; the last class also the smaller and empty ones), so that the wavefronts
// and workgroups finish together.
// icount: [kItemClasses][nwin_total] wavefront items, [kItemClasses][2 nwin_total] pieces of the
// halves, [2 nwin_total] partial slots, [nwin_total] windows that k_win_reduce completes; one exclusive
// scan gives the queue positions, slot numbers and places in k_win_reduce's list.  totals[0] = records, [1] = wavefront items, [2] = coop_min,
// [3] = pieces, [4] = max |v| bits, [6] = windows that k_win_reduce completes, [7] = coop_cap (the shape that fit_shape
// left), [8], [9] = the coarse bins' pieces, [kPieceHead ..] = the piece queue's heads.
constexpr int kPieceHead = 10;           // two words: blocks of eight terms, of sixteen
constexpr int kItemClasses = 8;

__device__ __forceinline__ int item_class(uint32_t count, uint32_t cap) {
    if (count == 0) return kItemClasses - 1;
    int c = 0;
    while (c < kItemClasses - 1 && (static_cast<uint64_t>(count) << (c + 1)) <= cap) ++c;
    return c;
}

// Home records of half `half` of window (wa, wb) of slab ls (0 outside the grid of windows).
__device__ __forceinline__ uint32_t half_records(const uint32_t* __restrict__ boff, const WinGeom& wg, int ls, int wa, int wb,
                                                 int half) {
    if (wa < 0 || wb < 0) return 0u;
    const int per = 8 >> wg.cls_log2;                      // classes per half
    const int base = (ls * wg.nw + wb) * wg.nh, h = (2 * wa + half) * per;
    return boff[base + min(h + per, wg.nh)] - boff[base + min(h, wg.nh)];
}

// How window w's records are shared out: [h[0], h[1]) and [h[1], h[2]) the home records of its two
// halves; [s0, s1) less [hole, hole + hole_len) the records of its wavefront item, s_count of them.
// up, left[2], up_left: the records of the dense halves that reach it from the windows above and
// to the left (0 where a half is not dense).
struct WinSplit {
    uint32_t h[3], s0, s1, hole, hole_len, s_count;
    uint32_t up, left[2], up_left;
    bool dense[2];
    __device__ bool reduced() const { return dense[0] || dense[1] || (up | left[0] | left[1] | up_left) != 0; }
    // Bit 0, 1, 2: skip the copies in the half above, the lower half and the upper half.
    __device__ int skip() const { return (up_left != 0 ? 1 : 0) | (left[0] != 0 ? 2 : 0) | (left[1] != 0 ? 4 : 0); }
};
__device__ __forceinline__ WinSplit window_split(const uint32_t* __restrict__ boff, const WinGeom& wg, int w,
                                                 const WinRange& x, uint32_t end) {
    const int ls = w / wg.nwin, r = w - ls * wg.nwin;
    const int wa = r / wg.nw, wb = r - wa * wg.nw;
    auto if_dense = [&](uint32_t n) { return n > wg.shape.coop_min ? n : 0u; };
    WinSplit s;
    s.h[0] = wg.cls_log2 == 2 ? x.bnd[2] : x.bnd[1];
    s.h[1] = wg.cls_log2 == 2 ? x.bnd[4] : x.bnd[2];
    s.h[2] = end;
    s.dense[0] = s.h[1] - s.h[0] > wg.shape.coop_min;
    s.dense[1] = s.h[2] - s.h[1] > wg.shape.coop_min;
    // (The classes below the home ones are the upper half of the window above; none at the top.)
    s.up = if_dense(s.h[0] - x.start());
    s.left[0] = if_dense(half_records(boff, wg, ls, wa, wb - 1, 0));
    s.left[1] = if_dense(half_records(boff, wg, ls, wa, wb - 1, 1));
    s.up_left = if_dense(half_records(boff, wg, ls, wa - 1, wb - 1, 1));
    s.s0 = s.up != 0 ? (s.dense[0] ? s.h[1] : s.h[0]) : x.start();
    s.s1 = s.dense[1] ? (s.dense[0] ? s.h[0] : s.h[1]) : s.h[2];
    if (s.s1 < s.s0) s.s1 = s.s0;                          // both halves and the one above are dense
    s.hole = s.h[0];
    s.hole_len = s.dense[0] && s.s0 <= s.h[0] && s.s1 >= s.h[1] ? s.h[1] - s.h[0] : 0u;
    s.s_count = s.s1 - s.s0 - s.hole_len;
    return s;
}

// The queue classes of a window's wavefront item (-1: it has none) and of a dense half's pieces.
__device__ __forceinline__ int wave_item_class(const WinGeom& wg, const WinSplit& s) {
    const uint32_t cap = 3u * min(wg.shape.coop_min, 0xffffffffu / 3u);
    return s.s_count > 0 || !s.reduced() ? item_class(s.s_count, cap) : -1;
}
__device__ __forceinline__ int piece_class(const WinGeom& wg, const Pieces& p) { return item_class(p.per, wg.shape.coop_cap); }

__global__ void __launch_bounds__(256)
k_win_item_counts(const uint32_t* __restrict__ boff, WinGeom wg, uint32_t* __restrict__ icount, uint32_t* __restrict__ totals,
                  const uint32_t* __restrict__ words) {
    const int w = blockIdx.x * 256 + threadIdx.x;
    const int nwt = wg.nwin_total;
    if (w >= nwt) return;
    uint32_t end;
    const WinRange x = window_range(boff, wg, w, end);
    fit_shape(words, wg.slots, wg.shape);
    if (w == 0) {
        totals[0] = boff[wg.nbins];
        totals[2] = wg.shape.coop_min;
        totals[7] = wg.shape.coop_cap;
    }
    const WinSplit s = window_split(boff, wg, w, x, end);
    const int wcls = wave_item_class(wg, s);
    for (int k = 0; k < kItemClasses; ++k) icount[k * nwt + w] = k == wcls ? 1u : 0u;
    uint32_t* half = icount + kItemClasses * nwt;
    for (int j = 0; j < 2; ++j) {
        int pcls = -1;
        Pieces p = {0u, 0u};
        if (s.dense[j]) {
            p = dense_pieces(s.h[j + 1] - s.h[j], wg.shape.coop_cap);
            pcls = piece_class(wg, p);
        }
        for (int k = 0; k <= kItemClasses; ++k)
            half[(2 * k + j) * nwt + w] = k == pcls || k == kItemClasses ? p.count : 0u;
    }
    half[(2 * kItemClasses + 2) * nwt + w] = s.reduced() ? 1u : 0u;
}

// A window that k_win_reduce completes: the partial slots of the halves that reach it (its lower
// and upper half, the upper half of the window above, the two halves of the window to the left, the
// upper half of the window above that), and whether the planes hold its wavefront item's sums.
struct WReduce {
    int win, add;
    uint32_t first[6], count[6];
};

// kItemLanes threads per window write its items at the places that the counts' offsets give them, the
// first one the wavefront item and, for a window that k_win_reduce completes, its entry there.  Bound by
// latency: two rounds of loads that no cache line serves twice, so few threads per window (SKA-Low
// snapshot, 9,216 windows: 11 us with two, 18 with eight; a thread per item that looks its window up by
// binary search over the offsets is a chain of 18 loads, 16 us).
constexpr int kItemLanes = 2;
__global__ void __launch_bounds__(256)
k_win_item_write(const uint32_t* __restrict__ boff, const uint32_t* __restrict__ ioff, WinGeom wg, WItem* __restrict__ items,
                 uint32_t max_items, WReduce* __restrict__ red, uint32_t* __restrict__ totals) {
    wg.shape = {totals[2], totals[7]};
    const int t = blockIdx.x * 256 + threadIdx.x;
    const int w = t / kItemLanes, sub = t % kItemLanes;
    const int nwt = wg.nwin_total;
    const int n = 3 * kItemClasses * nwt;
    if (w >= nwt) return;
    uint32_t end;
    const WinRange x = window_range(boff, wg, w, end);
    const WinSplit s = window_split(boff, wg, w, x, end);
    // Every offset that the window can need is requested at once (at a valid place where it does not need it),
    // not one behind another.  (n + j nwt + w: the slots of half j of window w.)
    const uint32_t records[6] = {s.dense[0] ? s.h[1] - s.h[0] : 0u, s.dense[1] ? s.h[2] - s.h[1] : 0u,
                                 s.up, s.left[0], s.left[1], s.up_left};
    const int at[6] = {n + w, n + nwt + w, n + nwt + w - wg.nw, n + w - 1, n + nwt + w - 1, n + nwt + w - wg.nw - 1};
    uint32_t slots[6], queue[2];
#pragma unroll
    for (int k = 0; k < 6; ++k) slots[k] = ioff[records[k] != 0 ? at[k] : n];
    Pieces pieces[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        pieces[j] = dense_pieces(records[j], wg.shape.coop_cap);
        queue[j] = ioff[records[j] != 0 ? (kItemClasses + 2 * piece_class(wg, pieces[j]) + j) * nwt + w : n];
    }
    const int wcls = wave_item_class(wg, s);
    const uint32_t wave_at = ioff[wcls >= 0 ? wcls * nwt + w : n], slot0 = ioff[n], red0 = ioff[n + 2 * nwt];
    const uint32_t red_at = ioff[n + 2 * nwt + w];
    if (sub == 0 && s.reduced()) {
        WReduce r;
        r.win = w;
        r.add = s.s_count > 0 ? 1 : 0;
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            r.count[k] = records[k] != 0 ? dense_pieces(records[k], wg.shape.coop_cap).count : 0u;
            r.first[k] = records[k] != 0 ? slots[k] - slot0 : 0u;
        }
        red[red_at - red0] = r;
    }
    WItem it;
    it.win = w;
#pragma unroll
    for (int j = 0; j < kMaxClasses; ++j) it.bnd[j] = static_cast<int>(x.bnd[j]);
    it.hole = static_cast<int>(s.hole);
    it.hole_len = static_cast<int>(s.hole_len);
    if (sub == 0 && wcls >= 0) {
        it.start = static_cast<int>(s.s0);
        it.count = static_cast<int>(s.s_count);
        it.slot = -1;
        it.half = 0;
        it.skip = s.skip();
        if (wave_at < max_items) items[wave_at] = it;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        if (records[j] == 0) continue;
        it.half = j;
        it.skip = (s.skip() >> (j + 1)) & 1;
        for (uint32_t q = sub; q < pieces[j].count; q += kItemLanes) {
            it.start = static_cast<int>(s.h[j] + q * pieces[j].per);
            it.count = static_cast<int>(min(pieces[j].per, records[j] - q * pieces[j].per));
            it.slot = static_cast<int>(slots[j] - slot0 + q);
            if (queue[j] + q < max_items) items[queue[j] + q] = it;
        }
    }
    if (t == 0) {
        const uint32_t nwave = ioff[kItemClasses * nwt], nitems = min(slot0, max_items);
        totals[1] = min(nwave, nitems);
        totals[3] = nitems - min(nwave, nitems);
        totals[6] = ioff[n + 3 * nwt] - red0;
    }
}

// Partial slots: [term][kDenseRows rows][kDenseCols columns] from the half's first row and the
// window's first column: a first cell in the half's 8 x 16, and eight cells more at most.
constexpr int kDenseRows = kWin / 2 + 8;
constexpr int kDenseCols = kWin + 8;
constexpr int kDenseCells = kDenseRows * kDenseCols;

// The windows that dense pieces reach: the sum of the pieces' shares, in piece order (of the window's
// own halves, then of those above and to the left), added to what the window's wavefront item
// wrote to the planes, if it has one; so the result does not depend on timing.  One unit =
// (listed window, term) per workgroup, a thread per cell.  Bound by latency (a unit's chain of
// descriptor, slots and planes), so many small workgroups are resident, and the densest windows,
// with over a hundred pieces, are read sixteen pieces at a time.
__global__ void __launch_bounds__(256)
k_win_reduce(const WReduce* __restrict__ red, const uint32_t* __restrict__ totals, WinGeom wg,
             int G, int K, uint32_t max_slots, const float2* __restrict__ partial, float2* __restrict__ planes) {
    const uint32_t units = totals[6] * static_cast<uint32_t>(K);
    const size_t plane_size = static_cast<size_t>(G) * G;
    const size_t piece_size = static_cast<size_t>(K) * kDenseCells;
    const int cell = threadIdx.x, row = cell / kWin, col = cell % kWin;
    for (uint32_t u = blockIdx.x; u < units; u += gridDim.x) {
        const WReduce& r = red[u / K];
        const int k = static_cast<int>(u % K), w = r.win;
        const int ls = w / wg.nwin, rem = w - ls * wg.nwin;
        const int wa = rem / wg.nw, wb = rem - wa * wg.nw;
        const int a = wa * kWin + row, b = wb * kWin + col;
        const bool in_grid = a < G && b < G;
        float2* dst = planes + (static_cast<size_t>(ls) * K + k) * plane_size + static_cast<size_t>(a) * G + b;
        // The sum is FP64: over a hundred FP32 additions one after another would cost half a digit
        // (6.3e-7 against 3.1e-7 of the signed SKA-Low image).
        double sx = 0.0, sy = 0.0;
        if (r.add != 0 && in_grid) {
            const float2 v = *dst;
            sx = v.x;
            sy = v.y;
        }
        auto add_pieces = [&](int j, bool reached, int at) {
            const uint32_t first = r.first[j], pieces = r.count[j];
            if (pieces == 0 || !reached || first + pieces > max_slots) return;   // (the slot count bounds the pieces)
            const float2* src = partial + first * piece_size + static_cast<size_t>(k) * kDenseCells + at;
            uint32_t p = 0;
            for (; p + 16 <= pieces; p += 16) {
                float2 v[16];
#pragma unroll
                for (int q = 0; q < 16; ++q) v[q] = src[(p + q) * piece_size];
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    sx += v[q].x;
                    sy += v[q].y;
                }
            }
            for (; p < pieces; ++p) {
                const float2 v = src[p * piece_size];
                sx += v.x;
                sy += v.y;
            }
        };
        const int at = row * kDenseCols + col;
        constexpr int kDown = (kWin / 2) * kDenseCols;     // eight rows
        add_pieces(0, true, at);
        add_pieces(1, row >= 8, at - kDown);
        add_pieces(2, row < 8, at + kDown);
        add_pieces(3, col < 8, at + kWin);
        add_pieces(4, col < 8 && row >= 8, at + kWin - kDown);
        add_pieces(5, col < 8 && row < 8, at + kWin + kDown);
        if (in_grid) *dst = make_float2(static_cast<float>(sx), static_cast<float>(sy));
    }
}

// (f16(a - h.x), f16(b - h.y)) with each difference formed exactly in FP32: one mixed-precision
// fma per value (v_fma_mixlo / mixhi: source 0 the f16 half of h, negated, times 1.0, plus the
// FP32 value).
__device__ __forceinline__ half2v residual_f16x2(half2v h, float a, float b) {
    half2v r;
    asm volatile("v_fma_mixlo_f16 %0, -%1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(a));
    asm volatile("v_fma_mixhi_f16 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(r) : "v"(h), "v"(b));
    return r;
}

// x = hi + lo: hi rounded to nearest by a packed conversion (two values per instruction), lo =
// f16(x - hi) by mixed-precision fmas: |x - hi - lo| <= 2^-12 |lo| <= 2^-23 |x| (x in f16's
// normal range).
__device__ __forceinline__ void split_hilo(const float4& x0, const float4& x1, half8& hi, half8& lo) {
    const float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        const half2v h = __builtin_convertvector((float2v){v[i], v[i + 1]}, half2v);
        const half2v l = residual_f16x2(h, v[i], v[i + 1]);
        hi[i] = h[0];
        hi[i + 1] = h[1];
        lo[i] = l[0];
        lo[i + 1] = l[1];
    }
}

// x = hi + lo in bf16: hi = RN(x), lo = RN(x - hi) (the difference exact in FP32), so
// |x - hi - lo| <= 2^-9 |x - hi| <= 2^-18 |x|; two values per packed conversion.
__device__ __forceinline__ void split_bf16(const float (&x)[8], bf16x8& hi, bf16x8& lo) {
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        const bf16x2 h = __builtin_convertvector((float2v){x[i], x[i + 1]}, bf16x2);
        const bf16x2 l = __builtin_convertvector((float2v){x[i] - static_cast<float>(h[0]),
                                                           x[i + 1] - static_cast<float>(h[1])}, bf16x2);
        hi[i] = h[0];
        hi[i + 1] = h[1];
        lo[i] = l[0];
        lo[i + 1] = l[1];
    }
}

// One window row a with bf16 operands: B_a = ku_a kv formed in FP32 and split into bf16 hi + lo,
// then D_a += C_hi B_hi + C_lo B_hi + C_hi B_lo.
__device__ __forceinline__ void window_row_bf16(floatx4& d, const float* __restrict__ u_row, const float (&vf)[8],
                                                const bf16x8& a_hi, const bf16x8& a_lo) {
    const float4 u0 = *reinterpret_cast<const float4*>(u_row), u1 = *reinterpret_cast<const float4*>(u_row + 4);
    const float p[8] = {u0.x * vf[0], u0.y * vf[1], u0.z * vf[2], u0.w * vf[3],
                        u1.x * vf[4], u1.y * vf[5], u1.z * vf[6], u1.w * vf[7]};
    bf16x8 b_hi, b_lo;
    split_bf16(p, b_hi, b_lo);
    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_hi, b_hi, d, 0, 0, 0);
    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_lo, b_hi, d, 0, 0, 0);
    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_hi, b_lo, d, 0, 0, 0);
}

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One window row a.  kPrecSplit3: B_a[r][b] = ku_r[a] kv_r[b] from the factors split into
// f16 hi + lo (ku = uh + ul, kv = vh + vl), in packed f16: P = f16(uh vh), E = uh vh - P exactly
// (an fma of 11-bit significands), lo = f16(uh vl + ul vh + E), hi = P, so |ku kv - hi - lo| <=
// 2^-11 |lo| + |ul vl| ~ 2^-22 |ku kv| (products below 2^-24 / 2^-22 of the largest lose bits to
// f16 subnormals: contributions under 1e-12 of the peak); then D_a += C B_a as hi*hi + lo*hi +
// hi*lo.  Otherwise B_a = f16(uh vh) (relative error <= 3 x 2^-11 against ku kv, from the three
// roundings) and D_a += C_hi B_a [+ C_lo B_a].
template <int P>
__device__ __forceinline__ void es_product(const half8& uh, const half8& ul, const half8& vh, const half8& vl, half8& b_hi,
                                           half8& b_lo) {
    b_hi = uh * vh;
    b_lo = b_hi;
    if constexpr (P == kPrecSplit3) {
        const half8 e = __builtin_elementwise_fma(uh, vh, -b_hi);
        b_lo = __builtin_elementwise_fma(ul, vh, __builtin_elementwise_fma(uh, vl, e));
    }
}
template <int P>
__device__ __forceinline__ void contract(floatx4& d, const half8& a_hi, const half8& a_lo, const half8& b_hi, const half8& b_lo) {
    d = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_hi, b_hi, d, 0, 0, 0);
    if constexpr (P != kPrecSingle) d = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_lo, b_hi, d, 0, 0, 0);
    if constexpr (P == kPrecSplit3) d = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_hi, b_lo, d, 0, 0, 0);
}

// The eight ES values (times 2^7, and times dith with kDith) of a footprint with fraction F = t +
// 1/2: cell j is at x = (F + j) / 4 - 1, for j < 8 the quarter-support polynomial pair (j, 7 - j)
// in t.
template <bool kDith>
__device__ __forceinline__ void es_cells(float t, float dith, float (&v)[8]) {
    const float t2 = t * t;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        float e = kEsPolyEven[j][kEsPolyDegree / 2];
#pragma unroll
        for (int i = kEsPolyDegree / 2 - 1; i >= 0; --i) e = fmaf(e, t2, kEsPolyEven[j][i]);
        float o = kEsPolyOdd[j][kEsPolyDegree / 2 - 1];
#pragma unroll
        for (int i = kEsPolyDegree / 2 - 2; i >= 0; --i) o = fmaf(o, t2, kEsPolyOdd[j][i]);
        if constexpr (kDith) {
            e *= dith;
            o *= dith;
        }
        v[j] = fmaf(t, o, e);
        v[7 - j] = fmaf(-t, o, e);
    }
}

// Per-wavefront constants of the window kernel.
struct WinLane {
    _Float16* s_kuh;    // ku hi, lo: [32 rows a = -8 .. 23][32 samples], f16 (lo: kPrecSplit3 only)
    _Float16* s_kul;
    _Float16* s_kvh;    // kv hi, lo: [32 columns b = -8 .. 23][32 samples], f16
    _Float16* s_kvl;
    float* s_c;         // [16 m][32 samples]
    _Float16* s_kh;     // this lane's axis (ku or kv): hi and lo planes
    _Float16* s_kl;
    float* s_kuf;       // FP32 ES planes (kPrecBf16): ku, kv, and this lane's axis
    float* s_kvf;
    float* s_kf;
    int lane, rl, axis, g8, n16;
    int vexp;           // log2 of the c scale
    float inv;
};

// One chunk: the records [c0, c0 + 32) of item `it` (this lane's record in q) contracted
// into the accumulators d for the terms kg .. kg + 7.
template <int P>
__device__ __forceinline__ void window_chunk(const WinLane& L, const WItem& it, int c0, int kg, int K,
                                             int cls_log2, const uint4& q, floatx4 (&d)[kWin]) {
    using T = WinTraits<P>;
    bool valid = c0 + L.rl < it.count;
    // Classes of the chunk's first and last records (wave-uniform), and the 4-row quarters of
    // the window that they touch: class j covers rows [c d, c d + c + 7], d = j - 8 / c.
    const int i0 = it.record(c0), i1 = it.record(min(it.count, c0 + kChunk) - 1) + 1;
    // (i >= bnd as the sign of bnd - 1 - i, so that the sums stay in scalar registers; bnd[j] for
    // j >= ncls is the window's end, which no record reaches.)
    int j_first = 0, j_last = 0;
#pragma unroll
    for (int j = 1; j < kMaxClasses; ++j) {
        j_first += static_cast<int>((static_cast<uint32_t>(it.bnd[j]) + ~static_cast<uint32_t>(i0)) >> 31);
        j_last += static_cast<int>((static_cast<uint32_t>(it.bnd[j]) - static_cast<uint32_t>(i1)) >> 31);
    }
    const int cls = 1 << cls_log2, dlo = -(8 >> cls_log2);
    const int q_lo = max(0, ((j_first + dlo) * cls) >> 2);
    const int q_hi = min(3, ((j_last + dlo) * cls + cls + 7) >> 2);
    // ES factors along this lane's axis, as f16 (hi + lo for kPrecSplit3): the axis' 32 lanes
    // zero the window's 16 rows / columns of the planes (a 64-byte row per lane, or half a row
    // with one plane), then every lane writes its sample's 9 cells ceil(p - 4) .. ceil(p - 4) + 8
    // (padded rows take those outside the window; the ninth is nonzero only for an integer p).
    {
        const uint4 z = make_uint4(0u, 0u, 0u, 0u);
        if constexpr (T::kBf16) {
            float* zrow = L.s_kf - L.rl + (kPad + (L.rl & 15)) * kStrideF + ((L.rl & 16) ? 16 : 0);
#pragma unroll
            for (int k = 0; k < 4; ++k) reinterpret_cast<uint4*>(zrow)[k] = z;
        } else if constexpr (T::kEsLo) {
            _Float16* zrow = ((L.rl & 16) ? L.s_kl : L.s_kh) - L.rl + (kPad + (L.rl & 15)) * kStrideH;
#pragma unroll
            for (int k = 0; k < 4; ++k) reinterpret_cast<uint4*>(zrow)[k] = z;
        } else {
            _Float16* zrow = L.s_kh - L.rl + (kPad + (L.rl & 15)) * kStrideH + ((L.rl & 16) ? 16 : 0);
#pragma unroll
            for (int k = 0; k < 2; ++k) reinterpret_cast<uint4*>(zrow)[k] = z;
        }
    }
    // Single-f16 B: each sample's two ES factors are scaled by its own factors du, dv in [1, 2)
    // (from the visibility and s bits of its record) and c by 1 / (du dv).  Rounding ku, kv and
    // their product to f16 then errs by an amount that is independent from sample to sample and
    // averages out over the samples of a cell; with a fixed scale the kernel's flat peak sits at
    // one f16 value for every sample and the rounding is biased (about 4e-6 of the gridded sum).
    float dith_u = 1.0f, dith_v = 1.0f;
    if constexpr (T::kDither) {
        const uint32_t h = (q.x ^ q.y ^ q.z) * 0x9E3779B1u;
        dith_u = 1.0f + static_cast<float>(h >> 24) * (1.0f / 256.0f);
        dith_v = 1.0f + static_cast<float>((h >> 16) & 0xffu) * (1.0f / 256.0f);
    }
    // A record's row position is relative to its class's home window row (the first window row
    // that reads the class); this window reads the classes j >= 16 / c as the row above their
    // home, 16 rows up.
    const int foreign = cls_log2 == 2 ? it.bnd[4] : it.bnd[2];
    const int i = it.record(c0 + L.rl);
    if (it.skip != 0 && rec_cell(q.w) < 0) {
        const int part = i >= foreign ? 4 : i >= (cls_log2 == 2 ? it.bnd[2] : it.bnd[1]) ? 2 : 1;
        valid = valid && (it.skip & part) == 0;
    }
    if (valid) {
        const uint32_t pw = L.axis ? q.w : q.z;
        const int fl = rec_cell(pw) + (L.axis == 0 && i >= foreign ? kWin : 0);
        const uint32_t fb = rec_frac_bits(pw);
        const int first = min(max(fl, -kPad), kWin - 1);
        // Cell j is at x = (F + j) / 4 - 1 (F the record's fraction in [0, 1)): for j < 8 the
        // quarter-support polynomial pair (j, 7 - j) in t = F - 1/2, for j = 8 ES(1) when F = 0
        // and zero otherwise.
        const float t = fmaf(static_cast<float>(fb), kRecFracInv, -0.5f);
        const float dith = L.axis ? dith_v : dith_u;
        float v[8];
        es_cells<T::kDither>(t, dith, v);
        if constexpr (T::kBf16) {
            float* df = L.s_kf + (first + kPad) * kStrideF;
#pragma unroll
            for (int j = 0; j < 8; ++j) df[j * kStrideF] = v[j];
            df[8 * kStrideF] = fb == 0u ? kEsPolyEdge : 0.0f;
        } else {
        _Float16* dh = L.s_kh + (first + kPad) * kStrideH;
        // hi of the pair (j, 7 - j) by one packed round-to-nearest conversion, each lo = f16(v - hi)
        // with the difference formed in FP32 (one mixed-precision fma per value).
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const half2v h = __builtin_convertvector((float2v){v[j], v[7 - j]}, half2v);
            dh[j * kStrideH] = h[0];
            dh[(7 - j) * kStrideH] = h[1];
            if constexpr (T::kEsLo) {
                _Float16* dl = L.s_kl + (first + kPad) * kStrideH;
                const half2v l = residual_f16x2(h, v[j], v[7 - j]);
                dl[j * kStrideH] = l[0];
                dl[(7 - j) * kStrideH] = l[1];
            }
        }
        const bool edge = fb == 0u;
        if constexpr (T::kEsLo) dh[8 * kStrideH] = edge ? kEsPolyEdgeHi : static_cast<_Float16>(0.0f);
        else dh[8 * kStrideH] = static_cast<_Float16>(edge ? kEsPolyEdge * dith : 0.0f);
        if constexpr (T::kEsLo) {
            _Float16* dl = L.s_kl + (first + kPad) * kStrideH;
            dl[8 * kStrideH] = edge ? kEsPolyEdgeLo : static_cast<_Float16>(0.0f);
        }
        }
    }
    // c rows 2k + axis for the terms kg .. kg + 7.  Terms k >= K (when K is not a multiple of 8)
    // are contracted like the others and dropped at write-out (T_k stays in [-1, 1]).
    {
        float vs = valid ? rec_v(L.axis ? q.y : q.x, q.w, L.vexp) : 0.0f;
        if constexpr (T::kDither) vs *= __builtin_amdgcn_rcpf(dith_u * dith_v);
        const float s = rec_s(q.x, q.y, q.z), s2 = 2.0f * s;
        float t0 = 1.0f, t1 = s;                      // T_k, T_{k+1}
        for (int k = 0; k < kg; ++k) {
            const float t2 = s2 * t1 - t0;
            t0 = t1;
            t1 = t2;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            L.s_c[(2 * j + L.axis) * kStride + L.rl] = t0 * vs;
            const float t2 = s2 * t1 - t0;
            t0 = t1;
            t1 = t2;
        }
    }
    wave_lds_sync();

    // A (16 x 32): lane holds A[n16][g8 + i]; B (32 x 16): lane holds B[g8 + i][n16];
    // D (16 x 16): lane holds D[4 (lane / 16) + i][n16].
    if constexpr (T::kBf16) {
        bf16x8 a_hi, a_lo;
        {
            const float* row = L.s_c + L.n16 * kStride + L.g8;
            const float4 x0 = *reinterpret_cast<const float4*>(row), x1 = *reinterpret_cast<const float4*>(row + 4);
            const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
            split_bf16(x, a_hi, a_lo);
        }
        float vf[8];
        {
            const float* vrow = L.s_kvf + (kPad + L.n16) * kStrideF + L.g8;
            const float4 v0 = *reinterpret_cast<const float4*>(vrow), v1 = *reinterpret_cast<const float4*>(vrow + 4);
            vf[0] = v0.x; vf[1] = v0.y; vf[2] = v0.z; vf[3] = v0.w;
            vf[4] = v1.x; vf[5] = v1.y; vf[6] = v1.z; vf[7] = v1.w;
        }
        const float* ub = L.s_kuf + kPad * kStrideF + L.g8;
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
            if (qd >= q_lo && qd <= q_hi) {
#pragma unroll
                for (int a = 4 * qd; a < 4 * qd + 4; ++a) window_row_bf16(d[a], ub + a * kStrideF, vf, a_hi, a_lo);
            }
        }
        wave_lds_sync();
        return;
    }
    half8 a_hi, a_lo;
    {
        const float* row = L.s_c + L.n16 * kStride + L.g8;
        const float4 x0 = *reinterpret_cast<const float4*>(row), x1 = *reinterpret_cast<const float4*>(row + 4);
        if constexpr (T::kCLo) {
            split_hilo(x0, x1, a_hi, a_lo);
        } else {
            a_hi = __builtin_convertvector((floatx8){x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w}, half8);
            a_lo = a_hi;
        }
    }
    const half8 vh = *reinterpret_cast<const half8*>(L.s_kvh + (kPad + L.n16) * kStrideH + L.g8);
    half8 vl = vh;
    if constexpr (T::kEsLo) vl = *reinterpret_cast<const half8*>(L.s_kvl + (kPad + L.n16) * kStrideH + L.g8);
    const _Float16* uhb = L.s_kuh + kPad * kStrideH + L.g8;
    const _Float16* ulb = T::kEsLo ? L.s_kul + kPad * kStrideH + L.g8 : uhb;
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
        if (qd >= q_lo && qd <= q_hi) {
            // Each row's ES values are requested one row ahead, so that their LDS latency
            // overlaps the previous row's products and MFMAs.
            half8 uh_n = *reinterpret_cast<const half8*>(uhb + 4 * qd * kStrideH);
            half8 ul_n = uh_n;
            if constexpr (T::kEsLo) ul_n = *reinterpret_cast<const half8*>(ulb + 4 * qd * kStrideH);
#pragma unroll
            for (int a = 4 * qd; a < 4 * qd + 4; ++a) {
                const half8 uh = uh_n, ul = ul_n;
                if (a + 1 < 4 * qd + 4) {
                    uh_n = *reinterpret_cast<const half8*>(uhb + (a + 1) * kStrideH);
                    if constexpr (T::kEsLo) ul_n = *reinterpret_cast<const half8*>(ulb + (a + 1) * kStrideH);
                }
                half8 b_hi, b_lo;
                es_product<P>(uh, ul, vh, vl, b_hi, b_lo);
                contract<P>(d[a], a_hi, a_lo, b_hi, b_lo);
            }
        }
    }
    wave_lds_sync();
}

// Destination of the window values of (row a, term k, column n16) in the planes; out-of-grid cells
// and k >= K go to the scratch line `trash` so that every lane issues the same stores.
struct WinOut {
    float2* base;
    int kstride, wa16, wb16;
};
__device__ __forceinline__ WinOut window_out(const WItem& it, const WinGeom& wg, int K, int G, float2* planes, int n16) {
    const int ls = it.win / wg.nwin, w = it.win - ls * wg.nwin;
    const int wa = w / wg.nw, wb = w - wa * wg.nw;
    const size_t plane_size = static_cast<size_t>(G) * G;
    WinOut o;
    o.base = planes + static_cast<size_t>(ls) * K * plane_size + static_cast<size_t>(wa) * kWin * G + wb * kWin + n16;
    // Offsets from base fit in 32 bits: k * G^2 + 15 G < 2^31 for K <= 32, G <= 8192.
    o.kstride = static_cast<int>(plane_size);
    o.wa16 = wa * kWin;
    o.wb16 = wb * kWin;
    return o;
}

__device__ __forceinline__ void window_store(const WinOut& o, int G, int K, int a, int k, int n16, float inv, float2 v,
                                             float2* trash, int lane) {
    const int ag = o.wa16 + a, bg = o.wb16 + n16;
    const float sg = ((ag + bg) & 1) ? -inv : inv;
    const bool ok = k < K && ag < G && bg < G;
    float2* dst = ok ? o.base + (k * o.kstride + a * G) : trash + lane;
    *dst = make_float2(v.x * sg, v.y * sg);
}

// One job of the window kernel: one slab batch of one snapshot, binned (records, item lists and
// totals in its call's workspace), with its own planes.  A launch takes up to kMaxJobs of them.
constexpr int kMaxJobs = kMaxWindowJobs;
struct WinJob {
    const WItem* items;
    uint32_t* totals;
    WRecords rec;
    float2* planes;
    float2* partial;
    float2* trash;
    WinGeom wg;
    int K, G;
    int k_lo, k_hi;          // the terms of a dense launch
};
struct WinJobs {
    WinJob job[kMaxJobs];
    int count;
};

// The c scale of a job from the largest |v| of its call: |c| <= 2^14 after scaling by 2^vexp;
// inv undoes it and the ES factors' scale.
struct JobScale {
    int vexp;
    float inv;
};
__device__ __forceinline__ JobScale job_scale(const WinJob& J) {
    const float vmax = __uint_as_float(J.totals[4]);
    int e = 0;
    if (vmax > 0.0f && vmax <= 3.0e38f) (void)frexpf(vmax, &e);
    e = min(max(e, -100), 100);
    return {14 - e, ldexpf(1.0f, e - 14 - kEsScaleLog2Sq)};
}

// The job of global item index g of a queue whose per-job starts are off[0 .. count] (LDS):
// the largest j with off[j] <= g (wave-uniform).
__device__ __forceinline__ int job_of(const int* off, int count, int g) {
    int j = 0;
    while (j + 1 < count && __builtin_amdgcn_readfirstlane(off[j + 1]) <= g) ++j;
    return j;
}

// ---- Dense halves -----------------------------------------------------------------------------
//
// k_win_dense contracts the home records of the dense half windows sorted by footprint column.  In
// the 16 x 16 window contraction a record's 8 x 8 footprint meets on average half of the window's
// rows and all 16 columns are computed for its eight; records that share their footprint's first
// column b0 fit exactly: the 16 columns of an MFMA block are two grid rows times the eight columns
// b0 .. b0 + 7, and records sorted by their first row a0 within b0 need four to six of the eight
// blocks that cover the half's rows.
//
// A workgroup takes one piece (records of one half window): it sorts their indices in LDS by (b0,
// a0), kBatch at a time, and its wavefronts claim runs of 32-record chunks of the sorted list.  A
// wavefront keeps the eight blocks of its current column b0 in registers and adds them to the
// piece's tile in LDS (16 rows x 24 columns x 2K) when the column changes or the run ends; a chunk
// that meets several columns is contracted once per column with c masked.  The tile is FP64
// because its LDS atomics are: ds_add_f32 handles one lane in three cycles on this chip (193 cycles
// per wavefront, measured), ds_add_f64 a wavefront in 9.
//
// Measured (SKA-Low snapshot, 8.4 M samples at 1024^2, 62% of the records in dense halves): 240 us, and
// 139 us for the wavefront items that remain, against 476 us for window contraction of everything;
// eight such snapshots in a batch 5.35 against 6.11 ms.  It issues a quarter of the MFMAs and 0.4 of
// the VALU instructions of the window form (3.5 M and 71 M).  About 110 us of it are the sort, the
// tile's clearing and write-out and the barriers around them, the rest the chunks, which wait for
// their LDS operands as long as they compute (a chunk's chain is about 5000 cycles with three
// wavefronts per SIMD).  Tried and slower: four wavefronts per SIMD at 128 registers (spills; 265 us),
// two workgroups of six wavefronts per CU (490 us, smaller batches), one wavefront sorting a batch
// ahead of the others (260 us), touching the next piece's lines early (255 us), private FP32
// slots with global atomics (27 us per thousand tile updates).
constexpr int kDenseHalf = kWin / 2;
constexpr int kDenseColumns = kWin + 8;                         // first columns -8 .. 15 (copies: -8 .. -1)
constexpr int kDenseGroups = 2 * kDenseColumns;                 // (first rows -8 .. -1 at the grid's top edge, 0 .. 7)
constexpr int kDenseKeys = kDenseHalf * kDenseGroups;
constexpr int kDenseTileStride = kDenseCells + 2;               // doubles per m
constexpr int kDenseURows = 16, kDenseVRows = 9;                // staged rows; columns + the ninth cell
constexpr int kDenseBlocks = kDenseURows / 2;
constexpr int kDStride = 32;                                    // halves or floats per staged ES row (a block's B operand
                                                                // reads two adjacent rows: no padding needed)

template <int P, int MB>
struct DenseTraits {
    using T = WinTraits<P>;
    // The modes of single-f16 ES products stage less and keep within 128 registers (168 with sixteen terms of one f16 each):
    // more wavefronts, and with one f16 per term value a whole default piece sorted at once.  (SKA-Low snapshot, call:
    // single 759 us with twelve wavefronts and 8192 records, 748 so, splitc 772 and 768; single at 16 terms 1130 and 1120.)
    static constexpr int kWaves = MB == 1 ? T::kWaves : P == kPrecSingle ? 12 : 8;
    static constexpr int kBatch = MB > 1 ? 4096 : P == kPrecSingle ? 16384 : 8192;             // records sorted at a time
    static constexpr int kPer = (kBatch + kWaves * 64 - 1) / (kWaves * 64);
    static constexpr int kRows = kDenseURows + kDenseVRows;
    // Per wavefront: the ES rows (ku hi [lo], kv hi [lo] in f16, or ku, kv in FP32), then c[16].
    static constexpr int kEsFloats = T::kBf16 ? kRows * kDStride : kRows * kDStride * (T::kEsLo ? 2 : 1) / 2;
    static constexpr int kStageFloats = kEsFloats + 16 * kStride;
    static constexpr int kTileFloats = 2 * 16 * MB * kDenseTileStride;
    static constexpr size_t kLds = sizeof(float) * (kTileFloats + kWaves * kStageFloats) + sizeof(uint16_t) * kBatch +
                                   sizeof(uint32_t) * (kDenseKeys + 2 * 64 + 2);
    static_assert(kEsFloats % 4 == 0 && kTileFloats % 4 == 0, "16-byte aligned staging rows");
};

// Barrier for data exchanged through LDS: global loads and stores stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A wavefront's staging area and place in the chunk.
template <int P>
struct DenseLane {
    _Float16 *s_kuh, *s_kvh;        // ku rows (hi, then lo), kv rows
    float *s_kuf, *s_kvf;           // FP32 rows (kPrecBf16)
    float* s_c;
    double* tile;
    int lane, rl, axis, g8, n16;
};

// The C operands of a chunk: A (16 x 32): lane holds A[n16][g8 + i], hi and lo, per 16-row block.
template <int P, int MB>
struct DenseC {
    typedef typename std::conditional<WinTraits<P>::kBf16, bf16x8, half8>::type op8;
    op8 hi[MB], lo[MB];
};

template <int P, int MB>
__device__ __forceinline__ void load_c(const DenseLane<P>& L, int mb, DenseC<P, MB>& A) {
    const float* row = L.s_c + L.n16 * kStride + L.g8;
    const float4 x0 = *reinterpret_cast<const float4*>(row), x1 = *reinterpret_cast<const float4*>(row + 4);
    if constexpr (WinTraits<P>::kBf16) {
        const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
        split_bf16(x, A.hi[mb], A.lo[mb]);
    } else if constexpr (WinTraits<P>::kCLo) {
        split_hilo(x0, x1, A.hi[mb], A.lo[mb]);
    } else {
        A.hi[mb] = __builtin_convertvector((floatx8){x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w}, half8);
        A.lo[mb] = A.hi[mb];
    }
}

// The operands of one chunk of a dense piece, staged: `cnt` records (this lane's in q; lanes past
// them hold the last one and contribute c = 0) for the terms kg .. kg + 8 MB - 1.  Returns the
// blocks that the chunk's rows meet, q_lo .. q_hi; row_adj: row of the stored cell 0 in the half.
template <int P, int MB>
__device__ __forceinline__ void dense_stage(const DenseLane<P>& L, int cnt, int kg, int vexp, int row_adj, const uint4& q,
                                            int& q_lo, int& q_hi, DenseC<P, MB>& A) {
    using T = WinTraits<P>;
    const int lane = L.lane, rl = L.rl, axis = L.axis;
    const bool valid = rl < cnt;
    const uint32_t pw = axis ? q.w : q.z;
    const uint32_t fb = rec_frac_bits(pw);
    const bool edge = fb == 0u;
    // First row within the half's eight (row_adj is a multiple of eight).
    const int r0 = rec_cell(pw) & (kDenseHalf - 1);
    {
        const int lo = axis ? kDenseHalf : r0, hi = axis ? 0 : r0 + (edge ? 1 : 0);
        q_lo = __ballot(lo < 2) != 0 ? 0 : __ballot(lo < 4) != 0 ? 1 : __ballot(lo < 6) != 0 ? 2 : 3;
        q_hi = __ballot(hi >= 7) != 0 ? 7 : __ballot(hi >= 5) != 0 ? 6 : __ballot(hi >= 3) != 0 ? 5 : __ballot(hi >= 1) != 0 ? 4 : 3;
    }
    const uint64_t edges = __ballot(axis && valid && edge) >> 32;
    float dith_u = 1.0f, dith_v = 1.0f;
    if constexpr (T::kDither) {                     // (as window_chunk)
        const uint32_t h = (q.x ^ q.y ^ q.z) * 0x9E3779B1u;
        dith_u = 1.0f + static_cast<float>(h >> 24) * (1.0f / 256.0f);
        dith_v = 1.0f + static_cast<float>((h >> 16) & 0xffu) * (1.0f / 256.0f);
    }
    // The rows of ku are cleared, then every lane writes its sample's cells: ku at rows r0 .. r0 + 8 of
    // sixteen, kv at rows 0 .. 7 (and its ninth cell at a row that is not read).
    {
        const uint4 z = make_uint4(0u, 0u, 0u, 0u);
        if constexpr (T::kBf16) {
#pragma unroll
            for (int i = 0; i < kDenseURows * 8; i += 64)
                reinterpret_cast<uint4*>(L.s_kuf + ((lane + i) >> 3) * kDStride)[lane & 7] = z;
        } else {
            constexpr int kRows = kDenseURows * (T::kEsLo ? 2 : 1);
#pragma unroll
            for (int i = 0; i < kRows * 4; i += 64)
                reinterpret_cast<uint4*>(L.s_kuh + ((lane + i) >> 2) * kDStride)[lane & 3] = z;
        }
    }
    wave_lds_sync();
    const int row0 = axis ? 0 : r0;
    {
        const float dith = axis ? dith_v : dith_u;
        float v[8];
        es_cells<T::kDither>(fmaf(static_cast<float>(fb), kRecFracInv, -0.5f), dith, v);
        if constexpr (T::kBf16) {
            float* df = (axis ? L.s_kvf : L.s_kuf) + rl + row0 * kDStride;
#pragma unroll
            for (int j = 0; j < 8; ++j) df[j * kDStride] = v[j];
            df[8 * kDStride] = edge ? kEsPolyEdge : 0.0f;
        } else {
            _Float16* dh = (axis ? L.s_kvh : L.s_kuh) + rl + row0 * kDStride;
            _Float16* dl = dh + (axis ? kDenseVRows : kDenseURows) * kDStride;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const half2v h = __builtin_convertvector((float2v){v[j], v[7 - j]}, half2v);
                dh[j * kDStride] = h[0];
                dh[(7 - j) * kDStride] = h[1];
                if constexpr (T::kEsLo) {
                    const half2v l = residual_f16x2(h, v[j], v[7 - j]);
                    dl[j * kDStride] = l[0];
                    dl[(7 - j) * kDStride] = l[1];
                }
            }
            if constexpr (T::kEsLo) {
                dh[8 * kDStride] = edge ? kEsPolyEdgeHi : static_cast<_Float16>(0.0f);
                dl[8 * kDStride] = edge ? kEsPolyEdgeLo : static_cast<_Float16>(0.0f);
            } else {
                dh[8 * kDStride] = static_cast<_Float16>(edge ? kEsPolyEdge * dith : 0.0f);
            }
        }
    }
    // c rows 2k + axis for the terms kg .. kg + 8 MB - 1 (terms k >= K are dropped at write-out).
    {
        float vs = valid ? rec_v(axis ? q.y : q.x, q.w, vexp) : 0.0f;
        if constexpr (T::kDither) vs *= __builtin_amdgcn_rcpf(dith_u * dith_v);
        const float s = rec_s(q.x, q.y, q.z), s2 = 2.0f * s;
        float t0 = 1.0f, t1 = s;
        for (int k = 0; k < kg; ++k) {
            const float t2 = s2 * t1 - t0;
            t0 = t1;
            t1 = t2;
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            if (mb > 0) wave_lds_sync();
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                L.s_c[(2 * j + axis) * kStride + rl] = t0 * vs;
                const float t2 = s2 * t1 - t0;
                t0 = t1;
                t1 = t2;
            }
            wave_lds_sync();
            if constexpr (MB > 1) load_c<P, MB>(L, mb, A);
            // Footprints of an exactly integer column position have a ninth column, of value ES(1):
            // their contribution to it goes straight to the tile, one record at a time.
            for (uint64_t left = edges; left != 0; left &= left - 1) {
                const int r = __builtin_ctzll(left);
                const int rb = ((__shfl(rec_cell(q.z) + row_adj, r, 64) + kPad) & ~(kDenseHalf - 1)) - kPad;
                const int col = __shfl(rec_cell(q.w), r, 64) + 8;
                const float ev = kEsPolyEdge * __shfl(dith_v, r, 64);
                if (col < 0 || col >= kDenseCols) continue;
                for (int t = lane; t < 16 * kDenseURows; t += 64) {
                    const int m = t / kDenseURows, a = t - m * kDenseURows, ar = rb + a;
                    float ku;
                    if constexpr (T::kBf16) {
                        ku = L.s_kuf[a * kDStride + r];
                    } else {
                        ku = static_cast<float>(L.s_kuh[a * kDStride + r]);
                        if constexpr (T::kEsLo) ku += static_cast<float>(L.s_kuh[(kDenseURows + a) * kDStride + r]);
                    }
                    if (ar >= 0 && ar < kDenseRows)
                        atomicAdd(L.tile + (16 * mb + m) * kDenseTileStride + ar * kDenseCols + col,
                                  static_cast<double>(L.s_c[m * kStride + r]) * (ku * ev));
                }
            }
        }
    }
}

// The staged chunk's records of bits `sel` (bit i = record i) contracted into the blocks d.
// B (32 x 16): lane holds B[g8 + i][n16] = ku of row 2b + n16 / 8 times kv of column n16 % 8;
// D (16 x 16): lane holds D[4 (lane / 16) + i][n16].
template <int P, int MB>
__device__ __forceinline__ void dense_contract(const DenseLane<P>& L, const DenseC<P, MB>& A, uint32_t sel, int q_lo, int q_hi,
                                               floatx4 (&d)[MB][kDenseBlocks]) {
    using T = WinTraits<P>;
    const int g8 = L.g8, n16 = L.n16, par = n16 >> 3, j8 = n16 & 7;
    using op8 = typename DenseC<P, MB>::op8;
    typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
    // (With one block c is still staged: splitting it again costs less than holding it.)
    DenseC<P, MB> C = A;
    if constexpr (MB == 1) load_c<P, MB>(L, 0, C);
    auto& a_hi = C.hi;
    auto& a_lo = C.lo;
    if (sel != 0xffffffffu) {
        const int m8 = static_cast<int>(sel >> g8);
        uint4v mask;
#pragma unroll
        for (int p = 0; p < 4; ++p)
            mask[p] = (static_cast<uint32_t>((m8 << (31 - 2 * p)) >> 31) & 0xffffu) | (static_cast<uint32_t>((m8 << (30 - 2 * p)) >> 31) & 0xffff0000u);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            a_hi[mb] = __builtin_bit_cast(op8, __builtin_bit_cast(uint4v, a_hi[mb]) & mask);
            a_lo[mb] = __builtin_bit_cast(op8, __builtin_bit_cast(uint4v, a_lo[mb]) & mask);
        }
    }
    if constexpr (T::kBf16) {
        const float* vrow = L.s_kvf + j8 * kDStride + g8;
        const float4 v0 = *reinterpret_cast<const float4*>(vrow), v1 = *reinterpret_cast<const float4*>(vrow + 4);
#pragma unroll
        for (int b = 0; b < kDenseBlocks; ++b) {
            if (b < q_lo || b > q_hi) continue;
            const float* ur = L.s_kuf + (2 * b + par) * kDStride + g8;
            const float4 u0 = *reinterpret_cast<const float4*>(ur), u1 = *reinterpret_cast<const float4*>(ur + 4);
            const float p[8] = {u0.x * v0.x, u0.y * v0.y, u0.z * v0.z, u0.w * v0.w,
                                u1.x * v1.x, u1.y * v1.y, u1.z * v1.z, u1.w * v1.w};
            bf16x8 b_hi, b_lo;
            split_bf16(p, b_hi, b_lo);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                d[mb][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_hi[mb], b_hi, d[mb][b], 0, 0, 0);
                d[mb][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_lo[mb], b_hi, d[mb][b], 0, 0, 0);
                d[mb][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_hi[mb], b_lo, d[mb][b], 0, 0, 0);
            }
        }
    } else {
        // Each block's ku values are requested one block ahead, so that their LDS latency overlaps the
        // previous block's products and MFMAs.
        const _Float16* urow = L.s_kuh + (2 * q_lo + par) * kDStride + g8;
        half8 uh_n = *reinterpret_cast<const half8*>(urow);
        half8 ul_n = uh_n;
        if constexpr (T::kEsLo) ul_n = *reinterpret_cast<const half8*>(urow + kDenseURows * kDStride);
        const _Float16* vrow = L.s_kvh + j8 * kDStride + g8;
        const half8 vh = *reinterpret_cast<const half8*>(vrow);
        half8 vl = vh;
        if constexpr (T::kEsLo) vl = *reinterpret_cast<const half8*>(vrow + kDenseVRows * kDStride);
#pragma unroll
        for (int b = 0; b < kDenseBlocks; ++b) {
            if (b < q_lo || b > q_hi) continue;
            const half8 uh = uh_n, ul = ul_n;
            if (b + 1 < kDenseBlocks) {                    // (unused past q_hi)
                const _Float16* ur = L.s_kuh + (2 * b + 2 + par) * kDStride + g8;
                uh_n = *reinterpret_cast<const half8*>(ur);
                if constexpr (T::kEsLo) ul_n = *reinterpret_cast<const half8*>(ur + kDenseURows * kDStride);
            }
            half8 b_hi, b_lo;
            es_product<P>(uh, ul, vh, vl, b_hi, b_lo);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) contract<P>(d[mb][b], a_hi[mb], a_lo[mb], b_hi, b_lo);
        }
    }
}

template <int P, int MB>
__global__ void __launch_bounds__((DenseTraits<P, MB>::kWaves * 64))
k_win_dense(WinJobs jobs) {
    using T = WinTraits<P>;
    using D = DenseTraits<P, MB>;
    constexpr int kThreads = D::kWaves * 64;
    extern __shared__ __align__(16) float dense_lds[];
    __shared__ int s_item, s_chunk;
    __shared__ int s_off[kMaxJobs + 1], s_wave_n[kMaxJobs];
    DenseLane<P> L;
    const int lane = L.lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    L.rl = lane & 31;
    L.axis = lane >> 5;
    L.g8 = 8 * (lane >> 4);
    L.n16 = lane & 15;
    double* const tile = L.tile = reinterpret_cast<double*>(dense_lds);
    float* const stage = dense_lds + D::kTileFloats + wave * D::kStageFloats;
    L.s_c = stage + D::kEsFloats;
    L.s_kuh = reinterpret_cast<_Float16*>(stage);
    L.s_kvh = L.s_kuh + kDenseURows * kDStride * (T::kEsLo ? 2 : 1);
    L.s_kuf = stage;
    L.s_kvf = stage + kDenseURows * kDStride;
    uint16_t* const s_idx = reinterpret_cast<uint16_t*>(dense_lds + D::kTileFloats + D::kWaves * D::kStageFloats);
    uint32_t* const s_hist = reinterpret_cast<uint32_t*>(s_idx + D::kBatch);
    uint32_t* const s_gend = s_hist + kDenseKeys;          // the non-empty columns: end in the sorted list,
    uint32_t* const s_gid = s_gend + 64;                   // and group; [128] their number
    const int njobs = jobs.count;

    // The jobs' pieces as offsets of one queue, whose head is a word of job 0's totals.  The claimed index
    // is read back into a scalar register, so the loop exit is wave-uniform by construction and
    // every wavefront runs the same barriers.
    if (threadIdx.x == 0) {
        int c = 0;
        for (int j = 0; j < njobs; ++j) {
            s_off[j] = c;
            s_wave_n[j] = static_cast<int>(jobs.job[j].totals[1]);
            c += static_cast<int>(jobs.job[j].totals[3]);
        }
        s_off[njobs] = c;
        s_item = static_cast<int>(atomicAdd(&jobs.job[0].totals[kPieceHead + MB - 1], 1u));
    }
    // A piece's job and record range, requested while the piece before it is contracted.
    struct Piece {
        int job, start, count, half_skip, slot;
        const uint4* rec;
    };
    auto fetch = [&](int gi, Piece& p) {
        p.job = job_of(s_off, njobs, gi);
        const WinJob& J = jobs.job[p.job];
        const WItem* it = J.items + (__builtin_amdgcn_readfirstlane(s_wave_n[p.job]) +
                                     (gi - __builtin_amdgcn_readfirstlane(s_off[p.job])));
        p.start = __builtin_amdgcn_readfirstlane(it->start);
        p.count = __builtin_amdgcn_readfirstlane(it->count);
        p.half_skip = __builtin_amdgcn_readfirstlane(it->half | it->skip << 1);
        p.slot = __builtin_amdgcn_readfirstlane(it->slot);
        p.rec = J.rec.r + p.start;
    };
    lds_barrier();
    const int nitems = __builtin_amdgcn_readfirstlane(s_off[njobs]);
    int gi = __builtin_amdgcn_readfirstlane(s_item);
    if (gi >= nitems) return;
    Piece it;
    fetch(gi, it);
    for (;;) {
        lds_barrier();                                   // s_item read; the tile is free
        // The next piece is claimed now and published with this one's sorted indices.
        uint32_t gnext = 0;
        if (threadIdx.x == 0) gnext = atomicAdd(&jobs.job[0].totals[kPieceHead + MB - 1], 1u);
        int gi_next = nitems;
        Piece itn;
        const WinJob& J = jobs.job[it.job];
        const JobScale scale = job_scale(J);
        const int K = J.K, k_lo = J.k_lo, k_hi = J.k_hi;
        // (The upper half's records store their row relative to the window below.)
        const int row_adj = (it.half_skip & 1) ? kDenseHalf : 0;
        const bool skip = (it.half_skip & 2) != 0;
        for (int kg = k_lo; kg < k_hi; kg += 8 * MB) {
            for (int i = threadIdx.x; i < D::kTileFloats / 4; i += kThreads)
                reinterpret_cast<float4*>(dense_lds)[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            for (int b0 = 0; b0 < it.count; b0 += D::kBatch) {
                const uint4* rec = it.rec + b0;
                if (kg == k_lo || it.count > D::kBatch) {
                    // Sort the batch's records by key = (column, first row): counts with each record's
                    // rank, the counts' prefix, then the sorted indices.
                    const int nb = min(D::kBatch, it.count - b0);
                    for (int i = threadIdx.x; i < kDenseKeys; i += kThreads) s_hist[i] = 0;
                    uint2 w[D::kPer];                      // the records' last two words
#pragma unroll
                    for (int u = 0; u < D::kPer; ++u)
                        w[u] = reinterpret_cast<const uint2*>(rec + min(static_cast<int>(threadIdx.x) + u * kThreads, nb - 1))[1];
                    lds_barrier();
                    uint32_t kr[D::kPer];
#pragma unroll
                    for (int u = 0; u < D::kPer; ++u) {
                        const int i = threadIdx.x + u * kThreads;
                        const int row = rec_cell(w[u].x) + row_adj, col = rec_cell(w[u].y);
                        const uint32_t r = static_cast<uint32_t>(min(max(row, -kPad), kDenseHalf - 1) + kPad);
                        const uint32_t c = static_cast<uint32_t>(min(max(col, -kPad), kWin - 1) + kPad);
                        const uint32_t key = ((r >> 3) * kDenseColumns + c) * kDenseHalf + (r & 7u);
                        kr[u] = ~0u;
                        if (i < nb && !(skip && col < 0)) kr[u] = key << 16 | atomicAdd(&s_hist[key], 1u);
                    }
                    lds_barrier();
                    if (wave == 0) {
                        // One group (8 keys) per lane for 48 lanes.
                        uint32_t h[kDenseHalf], tot = 0;
                        const bool on = lane < kDenseGroups;
#pragma unroll
                        for (int i = 0; i < kDenseHalf; ++i) {
                            h[i] = on ? s_hist[lane * kDenseHalf + i] : 0u;
                            tot += h[i];
                        }
                        uint32_t pt = tot;
                        for (int d = 1; d < 64; d <<= 1) {
                            const uint32_t a = __shfl_up(pt, d, 64);
                            if (lane >= d) pt += a;
                        }
                        const uint64_t some = __ballot(tot != 0);
                        if (on) {
                            uint32_t run = pt - tot;
#pragma unroll
                            for (int i = 0; i < kDenseHalf; ++i) {
                                s_hist[lane * kDenseHalf + i] = run;
                                run += h[i];
                            }
                        }
                        if (tot != 0) {
                            const int at = __popcll(some & ((1ull << lane) - 1));
                            s_gend[at] = pt;
                            s_gid[at] = lane;
                        }
                        if (lane == 0) s_gid[64] = static_cast<uint32_t>(__popcll(some));
                    }
                    lds_barrier();
#pragma unroll
                    for (int u = 0; u < D::kPer; ++u)
                        if (kr[u] != ~0u) s_idx[s_hist[kr[u] >> 16] + (kr[u] & 0xffffu)] = static_cast<uint16_t>(threadIdx.x + u * kThreads);
                }
                if (threadIdx.x == 0) {
                    s_chunk = 0;
                    if (b0 == 0 && kg == k_lo) s_item = static_cast<int>(gnext);
                }
                lds_barrier();
                if (b0 == 0 && kg == k_lo) {
                    gi_next = __builtin_amdgcn_readfirstlane(s_item);
                    if (gi_next < nitems) fetch(gi_next, itn);
                }

                // Runs of chunks, claimed from an LDS counter (the SIMDs issue their oldest wavefront
                // first, so an even split would leave the piece waiting for the youngest): one run of
                // r chunks per wavefront, then one of r / 2, then single chunks, r = half an even
                // share.  Lane l holds column l of the list.
                const int ngroups = __builtin_amdgcn_readfirstlane(static_cast<int>(s_gid[64]));
                const uint32_t gend = lane < ngroups ? s_gend[lane] : 0xffffffffu;
                const uint32_t gid = lane < ngroups ? s_gid[lane] : 0u;
                const int n = ngroups > 0 ? __builtin_amdgcn_readlane(static_cast<int>(gend), ngroups - 1) : 0;
                const int nch = (n + kChunk - 1) / kChunk;
                const int run1 = max(1, nch / (2 * D::kWaves)), run2 = max(1, run1 / 2);
                int left = 0;
                auto claim = [&]() -> int {
                    int v = 0;
                    if (lane == 0) v = atomicAdd(&s_chunk, 1);
                    v = __builtin_amdgcn_readfirstlane(v);
                    const int v2 = v - D::kWaves, v3 = v2 - D::kWaves;
                    left = v2 < 0 ? run1 : v3 < 0 ? run2 : 1;
                    return v2 < 0 ? run1 * v : v3 < 0 ? run1 * D::kWaves + run2 * v2 : (run1 + run2) * D::kWaves + v3;
                };
                auto load = [&](int c) { return rec[s_idx[min(c * kChunk + L.rl, n - 1)]]; };
                floatx4 d[MB][kDenseBlocks];
                auto clear = [&]() {
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                        for (int q = 0; q < kDenseBlocks; ++q) d[mb][q] = floatx4{0.f, 0.f, 0.f, 0.f};
                };
                auto flush = [&](int group) {
                    const int rb = group < kDenseColumns ? -kPad : 0;
                    const int col = (group < kDenseColumns ? group : group - kDenseColumns) - kPad + (L.n16 & 7);
                    if (col >= 0) {
                        double* at = tile + (4 * (lane >> 4)) * kDenseTileStride + (rb + (L.n16 >> 3)) * kDenseCols + col;
#pragma unroll
                        for (int q = 0; q < kDenseBlocks; ++q) {
                            const int row = rb + 2 * q + (L.n16 >> 3);
                            if (row >= 0 && row < kDenseRows) {
#pragma unroll
                                for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                                    for (int i = 0; i < 4; ++i)
                                        atomicAdd(at + (16 * mb + i) * kDenseTileStride + 2 * q * kDenseCols, static_cast<double>(d[mb][q][i]));
                            }
                        }
                    }
                    clear();
                };
                int c = claim();
                uint4 q_next = make_uint4(0u, 0u, 0u, 0u);
                if (c < nch) q_next = load(c);
                clear();
                int g = __popcll(__ballot(gend <= static_cast<uint32_t>(c * kChunk)));
                bool held = false;                         // d holds sums of column g
                while (c < nch) {
                    const uint4 q = q_next;
                    const int first = c * kChunk, last = min(first + kChunk, n);
                    int next = c + 1;
                    if (--left == 0) next = claim();
                    if (next < nch) q_next = load(next);
                    int q_lo, q_hi;
                    DenseC<P, MB> A;
                    dense_stage<P, MB>(L, last - first, kg, scale.vexp, row_adj, q, q_lo, q_hi, A);
                    for (int at = first;;) {
                        const int ge = __builtin_amdgcn_readlane(static_cast<int>(gend), g), to = min(ge, last);
                        const uint32_t upto = to - first >= 32 ? 0xffffffffu : (1u << (to - first)) - 1u;
                        const uint32_t sel = at == first && to == last ? 0xffffffffu : upto & ~((1u << (at - first)) - 1u);
                        dense_contract<P, MB>(L, A, sel, q_lo, q_hi, d);
                        held = true;
                        if (ge <= last) {                  // the column ends in this chunk
                            flush(__builtin_amdgcn_readlane(static_cast<int>(gid), g));
                            held = false;
                            ++g;
                        }
                        at = to;
                        if (at >= last) break;
                    }
                    wave_lds_sync();
                    if (next != c + 1) {                   // another run: its column
                        if (held) flush(__builtin_amdgcn_readlane(static_cast<int>(gid), g));
                        held = false;
                        g = __popcll(__ballot(gend <= static_cast<uint32_t>(next * kChunk)));
                    }
                    c = next;
                }
                if (held) flush(__builtin_amdgcn_readlane(static_cast<int>(gid), g));
                lds_barrier();
            }
            // The piece's share: [term][row][column] with the checkerboard sign.
            float2* out = J.partial + (static_cast<size_t>(it.slot) * K + kg) * kDenseCells;
            const int nk = min(8 * MB, k_hi - kg);
            for (int v = threadIdx.x; v < nk * kDenseCells; v += kThreads) {
                const int k = v / kDenseCells, cell = v - k * kDenseCells;
                const float sg = ((cell / kDenseCols + cell) & 1) ? -scale.inv : scale.inv;     // (kDenseCols even)
                out[v] = make_float2(static_cast<float>(tile[2 * k * kDenseTileStride + cell]) * sg,
                                     static_cast<float>(tile[(2 * k + 1) * kDenseTileStride + cell]) * sg);
            }
            if (kg + 8 * MB < k_hi) lds_barrier();
        }
        if (gi_next >= nitems) break;
        it = itn;
    }
}

// Persistent workgroups, one per CU, over the wavefront items of all the launch's jobs: each
// wavefront claims its next item while the current one is contracted and requests its first
// records before the current window is written, so the write-out overlaps the next item's
// loads (vector memory operations complete in order).  The terms are done eight at a time (one
// 16-row block of m = 2k + ri).
template <int P>
__global__ void __launch_bounds__(WinTraits<P>::kWaves * 64)
k_win_grid(WinJobs jobs) {
    using T = WinTraits<P>;
    extern __shared__ __align__(16) float stage_all[];
    __shared__ int s_witem;
    __shared__ int s_wave_off[kMaxJobs + 1];
    WinLane L;
    const int wave = threadIdx.x >> 6;
    L.lane = threadIdx.x & 63;
    L.s_kuh = reinterpret_cast<_Float16*>(stage_all + wave * T::kStageFloats);
    L.s_kuf = L.s_kvf = L.s_kf = nullptr;
    if constexpr (T::kBf16) {
        L.s_kuf = stage_all + wave * T::kStageFloats;
        L.s_kvf = L.s_kuf + kPlaneFloats;
        L.s_c = L.s_kvf + kPlaneFloats;
        L.s_kul = L.s_kvh = L.s_kvl = L.s_kuh;
    } else if constexpr (T::kEsLo) {
        L.s_kul = L.s_kuh + kPlaneHalves;
        L.s_kvh = L.s_kul + kPlaneHalves;
        L.s_kvl = L.s_kvh + kPlaneHalves;
        L.s_c = reinterpret_cast<float*>(L.s_kvl + kPlaneHalves);
    } else {
        L.s_kvh = L.s_kuh + kPlaneHalves;
        L.s_kul = L.s_kuh;
        L.s_kvl = L.s_kvh;
        L.s_c = reinterpret_cast<float*>(L.s_kvh + kPlaneHalves);
    }
    L.rl = L.lane & 31;
    L.axis = L.lane >> 5;
    L.g8 = 8 * (L.lane >> 4);
    L.n16 = L.lane & 15;
    L.s_kh = (L.axis ? L.s_kvh : L.s_kuh) + L.rl;
    L.s_kl = (L.axis ? L.s_kvl : L.s_kul) + L.rl;
    if constexpr (T::kBf16) L.s_kf = (L.axis ? L.s_kvf : L.s_kuf) + L.rl;
    const int lane = L.lane;
    const int njobs = jobs.count;

    // The jobs' item counts as offsets into the one list (each job's items in its largest-first
    // order).
    if (threadIdx.x == 0) {
        int w = 0;
        for (int j = 0; j < njobs; ++j) {
            s_wave_off[j] = w;
            w += static_cast<int>(jobs.job[j].totals[1]);
        }
        s_wave_off[njobs] = w;
        s_witem = 0;
    }
    __syncthreads();

    // Wavefront items of all jobs, one list.  Workgroup g takes items g, g + G, g + 2G, ... of it,
    // G = the number of workgroups, so the CUs get equal shares without a global queue; its
    // wavefronts claim them from an LDS counter, each claiming its next item while it contracts
    // the current one.
    const int nwave = __builtin_amdgcn_readfirstlane(s_wave_off[njobs]);
    const int nwg = static_cast<int>(gridDim.x);
    const int wg_items = nwave > static_cast<int>(blockIdx.x)
                             ? (nwave - static_cast<int>(blockIdx.x) + nwg - 1) / nwg : 0;
    auto claim_item = [&]() -> int {
        int v = 0;
        if (lane == 0) v = atomicAdd(&s_witem, 1);
        return v;
    };
    int ticket = claim_item();
    const int j0 = __builtin_amdgcn_readfirstlane(ticket);
    if (j0 >= wg_items) return;
    int item = static_cast<int>(blockIdx.x) + j0 * nwg;
    int jj = job_of(s_wave_off, njobs, item);
    WItem it = jobs.job[jj].items[item - __builtin_amdgcn_readfirstlane(s_wave_off[jj])];
    // Records of the next chunk, loaded while the current one is contracted.  Every lane loads
    // (lanes past the end re-read the last record and ignore it), so the loads land in place.
    uint4 q_next = jobs.job[jj].rec.get(it.count > 0 ? it.record(min(L.rl, it.count - 1)) : 0);
    for (;;) {
        ticket = claim_item();
        const WinJob& J = jobs.job[jj];
        const JobScale scale = job_scale(J);
        L.vexp = scale.vexp;
        L.inv = scale.inv;
        const int K = J.K, G = J.G;
        int next = nwave, jn = jj;
        WItem it_next = it;
        const WinOut o = window_out(it, J.wg, K, G, J.planes, L.n16);
        for (int kg = 0; kg < K; kg += 8) {
            floatx4 d[kWin];
#pragma unroll
            for (int a = 0; a < kWin; ++a) d[a] = floatx4{0.f, 0.f, 0.f, 0.f};
            for (int c0 = 0; c0 < it.count; c0 += kChunk) {
                const uint4 q = q_next;
                if (c0 + kChunk < it.count) q_next = J.rec.get(it.record(min(c0 + kChunk + L.rl, it.count - 1)));
                window_chunk<P>(L, it, c0, kg, K, J.wg.cls_log2, q, d);
            }
            // What comes next: this item's next term block, or the next item (possibly of
            // another job).  Its first records are requested now, ahead of the stores below.
            {
                int pcount = it.count, pfirst = it.record(min(L.rl, max(it.count - 1, 0)));
                const WRecords* prec = &J.rec;
                if (kg + 8 >= K) {
                    const int tn = __builtin_amdgcn_readfirstlane(ticket);
                    next = tn < wg_items ? static_cast<int>(blockIdx.x) + tn * nwg : nwave;
                    if (next < nwave) {
                        jn = job_of(s_wave_off, njobs, next);
                        it_next = jobs.job[jn].items[next - __builtin_amdgcn_readfirstlane(s_wave_off[jn])];
                        pcount = it_next.count;
                        pfirst = it_next.record(min(L.rl, max(it_next.count - 1, 0)));
                        prec = &jobs.job[jn].rec;
                    } else {
                        pcount = 0;
                    }
                }
                q_next = prec->get(pcount > 0 ? pfirst : 0);
            }
            // Rows m = 4 (lane / 16) + i are (re, im) of terms kg + 2 (lane / 16) and
            // kg + 2 (lane / 16) + 1; column n16.
#pragma unroll
            for (int a = 0; a < kWin; ++a)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    window_store(o, G, K, a, kg + 2 * (lane >> 4) + h, L.n16, L.inv,
                                 make_float2(d[a][2 * h], d[a][2 * h + 1]), J.trash, lane);
        }
        if (next >= nwave) break;
        item = next;
        jj = jn;
        it = it_next;
    }
}

}  // namespace

namespace {
// Row-class height (log2) and bin count of a grid: classes of 4 cells when that histogram fits in
// LDS, else of 8 (half the bins, so half the LDS bands when even those do not fit).
int window_class_log2(const GridParams& gp, int nw) {
    const size_t cols = static_cast<size_t>(gp.nslabs) * nw;
    return cols * ((gp.G + 3) / 4) <= static_cast<size_t>(kLdsBins) ? 2 : 3;
}
size_t window_bins(const GridParams& gp, int nw, int cls_log2) {
    const size_t nh = (static_cast<size_t>(gp.G) + (1u << cls_log2) - 1) >> cls_log2;
    return static_cast<size_t>(gp.nslabs) * nw * nh;
}
}  // namespace

// The class height in use: the tuned one, else by LDS fit.
static int effective_class_log2(const GridParams& gp, int nw) {
    return gp.class_log2 == 2 || gp.class_log2 == 3 ? gp.class_log2 : window_class_log2(gp, nw);
}

// Records at most: one row class and two window columns per sample.
static size_t max_window_records(const SampleInput& in) { return 2 * in.num_samples; }
// Pieces of the coarse bins at most (k_sub_list).
static size_t sub_piece_cap(const WinGeom& wg, size_t max_records) {
    return static_cast<size_t>(wg.nwin_total / wg.nw) * ((wg.nh + kSup - 1) / kSup) + max_records / kSubPiece;
}

bool grid_windows_supported(const SampleInput& in, const GridParams& gp) {
    if (gp.G > 8192 || gp.G < 1) return false;
    const int nw = (gp.G + kWin - 1) / kWin;
    if (window_bins(gp, nw, effective_class_log2(gp, nw)) >= (1ull << 30)) return false;
    return max_window_records(in) < (1ull << 31);
}

// The window geometry of a slab batch, but for what depends on the binning's blocks.
static WinGeom window_geometry(const SampleInput& in, const GridParams& gp) {
    WinGeom wg = {};
    wg.nw = (gp.G + kWin - 1) / kWin;
    wg.cls_log2 = effective_class_log2(gp, wg.nw);
    wg.ncls = 24 >> wg.cls_log2;
    wg.nh = (gp.G + (1 << wg.cls_log2) - 1) >> wg.cls_log2;
    wg.nwin = wg.nw * wg.nw;
    wg.nwin_total = wg.nwin * gp.nslabs;
    wg.nbins = static_cast<int>(window_bins(gp, wg.nw, wg.cls_log2));
    wg.shape = work_shape(in.num_samples, gp.coop_min, gp.coop_cap);
    // Bins that pass the LDS histogram are counted and scattered as coarse bins of eight row classes,
    // whose records k_sub_bins then sorts by class: one pass over the samples where there were up to
    // eight, for one more over the records.  16.7 M samples at 4096^2 (294,912 bins): count, scatter and
    // offsets 1.77 ms, now 0.70; 3.8 M at 2048^2 in three slabs 396 us, now 310.  The records wait in the planes, which
    // nothing has written yet; if these are too small, in LDS bands of the bins themselves.
    const size_t planes_bytes = static_cast<size_t>(gp.nslabs) * gp.K * gp.G * gp.G * sizeof(float2);
    const size_t max_records = max_window_records(in);
    const bool coarse = wg.nbins > kLdsBins &&
                        max_records * sizeof(uint4) + sub_piece_cap(wg, max_records) * sizeof(SubPiece) <= planes_bytes;
    wg.sup_log2 = coarse ? kSupLog2 : 0;
    wg.sup_rows = (wg.nh + (1 << wg.sup_log2) - 1) >> wg.sup_log2;
    wg.lbins = gp.nslabs * wg.nw * wg.sup_rows;
    // (Channels below sixteen would leave most of sixteen groups of threads idle.)
    wg.set_rows = in.num_channels > 8 ? 64 : 256;
    return wg;
}

// A slab batch's buffers in the context's workspace, but for the scratch.
struct WindowBuffers {
    uint32_t *counts, *boff, *cursor, *sums, *icount, *ioff;
    uint4* records;
};
static size_t item_counts(const WinGeom& wg) { return (3 * kItemClasses + 3) * static_cast<size_t>(wg.nwin_total); }
static WindowBuffers window_buffers(svdi_context* ctx, const SampleInput& in, const WinGeom& wg, bool use_lds) {
    const size_t nbins = static_cast<size_t>(wg.nbins), lbins = static_cast<size_t>(wg.lbins), ncounts = item_counts(wg);
    auto words = [&](Workspace::Slot slot, size_t n) { return static_cast<uint32_t*>(ctx->ws.get(slot, n * sizeof(uint32_t))); };
    // (Both forms' sizes where there are two: records that did not fit the planes and then do find room under capture.)
    const size_t sub_lbins = static_cast<size_t>(wg.nwin_total / wg.nw) * ((wg.nh + kSup - 1) / kSup);
    const size_t held = wg.nbins > kLdsBins ? std::max(nbins, (1 + 2 * kSup) * sub_lbins) : lbins;
    WindowBuffers b;
    b.counts = words(Workspace::kBinCounts, held + 14 + kShapeWords);
    b.boff = words(Workspace::kBinOffsets, nbins + 8);
    // Cursors (without LDS histograms); segment sums [kBinSegs][lbins]; the coarse bins' offsets.
    b.cursor = words(Workspace::kBinCursor, lbins + 8 + (use_lds ? kBinSegs * lbins : 0) + (wg.sup_log2 != 0 ? lbins + 8 : 0));
    b.sums = words(Workspace::kScanSums, scan_blocks(std::max(lbins, ncounts)));
    b.icount = words(Workspace::kItemCounts, ncounts + 8);
    b.ioff = words(Workspace::kItemOffsets, ncounts + 8);
    b.records = static_cast<uint4*>(ctx->ws.get(Workspace::kRecPos, max_window_records(in) * sizeof(uint4)));
    return b;
}

// The binning's blocks of a size, and what they keep in memory: per-block record offsets (the counts
// themselves when 32-bit), the (block, band) record totals, then the 16-bit per-block counts when a block has fewer
// than 65536 samples (a bin's count per block is at most its sample count).  LDS bands of at most kLdsBins bins, unless
// the per-block histograms would pass kMaxBlockHistBytes (then one global atomic per record).
struct BinBlocks {
    int size = 0;                                          // rows (snapshot input), samples per thread (preprocessed)
    size_t blocks = 0, bands = 1, nhist = 1, bytes = 0;
    bool use_lds = false, count16 = false;
};
static int most_block_size(const SampleInput& in) { return in.from_snapshot ? kBinRowsMost : kBinPerThreadMost; }
static int least_block_size(const SampleInput& in, const WinGeom& wg) {
    return !in.from_snapshot ? 1 : in.quad_rows ? kBinRowsLeast : wg.set_rows;
}
static BinBlocks bin_blocks(const SampleInput& in, const WinGeom& wg, int size) {
    BinBlocks b;
    b.size = size;
    const size_t units = in.from_snapshot ? in.num_rows : (in.num_samples + kBinThreads - 1) / kBinThreads;
    const size_t lbins = static_cast<size_t>(wg.lbins);
    b.blocks = (units + size - 1) / static_cast<size_t>(size);
    b.use_lds = b.blocks * lbins * sizeof(uint32_t) <= kMaxBlockHistBytes;
    if (b.use_lds) {
        b.bands = (lbins + kLdsBins - 1) / kLdsBins;
        b.nhist = b.blocks * lbins;
        b.count16 = static_cast<size_t>(size) * (in.from_snapshot ? in.num_channels : kBinThreads) < 65536;
    }
    b.bytes = (b.nhist + b.blocks * b.bands) * sizeof(uint32_t) + (b.count16 ? b.nhist * sizeof(uint16_t) : 0);
    return b;
}

// The blocks that a call takes, of those whose memory is at most `room` (the largest size's is given).  A block's time
// goes with its samples
// and, for its histogram, with the bins (about 3.7 ns a sample in the scatter and count passes together
// with 3 ns for ten bins), one block per CU at a time; every block also costs 14 bytes per bin of counts
// and offsets in memory.  So a snapshot that does not fill the chip with the largest blocks takes smaller
// ones (scatter + count of 1.4 M samples in 29,377 rows at 1000^2: 58 blocks 114 us, 230 blocks 56), as long
// as its histograms do not cost more.
static BinBlocks choose_bin_blocks(const svdi_context* ctx, const SampleInput& in, const WinGeom& wg, size_t room) {
    // Samples of a unit, a block's idle groups of threads included.
    auto unit_samples = [&](int size) {
        if (!in.from_snapshot) return static_cast<size_t>(kBinThreads);
        const size_t groups = kBinThreads / static_cast<size_t>(in.quad_rows ? size / 4 : wg.set_rows);
        return (in.num_channels + groups - 1) / groups * groups;
    };
    const int most = most_block_size(in), least = least_block_size(in, wg);
    const int step = in.from_snapshot && in.quad_rows ? 16 : least;
    BinBlocks pick;
    double best = 0.0;
    for (int size = most; size >= least; size -= step) {
        const BinBlocks b = bin_blocks(in, wg, size);
        const size_t rounds = (b.blocks + ctx->cu_count - 1) / ctx->cu_count;
        const double bins = static_cast<double>(wg.lbins);
        const double ns = rounds * (3.7 * static_cast<double>(size * unit_samples(size)) + 0.3 * std::min(bins, 1.0 * kLdsBins)) +
                          b.blocks * bins * 0.0035;
        if (size != most && (ns >= best || !b.use_lds || b.bytes > room)) continue;
        best = ns;
        pick = b;
    }
    return pick;
}

// Bytes of the window gridder's scratch: the binning's blocks first, then work items, partial sums and the scratch line.
constexpr size_t kTrash = 64;                              // float2
static size_t item_bytes(const WinGeom& wg) {
    return static_cast<size_t>(wg.nwin_total) * (sizeof(WItem) + sizeof(WReduce)) + kTrash * sizeof(float2);
}
static size_t slot_bytes(const GridParams& gp) { return static_cast<size_t>(gp.K) * kDenseCells * sizeof(float2) + sizeof(WItem); }

// The scratch is the buffer of the transformed rows (row_bytes), which is idle until the planes are
// done.  It holds a slot for every 576 grid cells, and most snapshots make a piece for every 1,300 to
// 17,000.  Small grids of many samples make more (1,219 at 512^2, one for every 484), so the buffer is larger
// by a slot for every 4,608 samples, or as large as usual_pieces says, where the worst case asks for it.  (With slots for
// the worst case, items and histograms in buffers of their own the context held 1,029 MB after the SKA-Low snapshot and
// 591 after one of 1.4 M samples at 1000^2; so 609 and 345.)
WindowScratch window_scratch(svdi_context* ctx, const SampleInput& in, const GridParams& gp, size_t row_bytes) {
    WindowScratch s = {row_bytes, row_bytes};
    GridParams batch = gp;
    for (int nslabs : {gp.nslabs, gp.total_slabs % gp.nslabs}) {           // whole slab batches and the last one
        if (nslabs == 0) continue;
        batch.nslabs = nslabs;
        const WinGeom wg = window_geometry(in, batch);
        const size_t halves = 2 * static_cast<size_t>(wg.nwin_total), allowance = in.num_samples / 4608 + 16;
        const size_t slots = std::min(most_pieces(wg.shape, max_window_records(in), halves),
                                      std::max((row_bytes - std::min(row_bytes, item_bytes(wg))) / slot_bytes(gp) + allowance,
                                               usual_pieces(wg.shape, in.num_samples, halves)));
        const BinBlocks largest = bin_blocks(in, wg, most_block_size(in));
        s.least = std::max({s.least, item_bytes(wg), largest.bytes});
        s.wanted = std::max({s.wanted, s.least, item_bytes(wg) + slots * slot_bytes(gp)});
        // (The choice is made only where it can matter: it is host time of every call.)
        if (bin_blocks(in, wg, least_block_size(in, wg)).bytes > s.wanted)
            s.wanted = std::max(s.wanted, choose_bin_blocks(ctx, in, wg, kMaxBlockHistBytes / 8).bytes);
        if (ctx->ws.in_arena()) (void)window_buffers(ctx, in, wg, largest.use_lds);
    }
    return s;
}

WindowJob bin_windows(svdi_context* ctx, const SampleInput& in, const GridParams& gp, float2* planes, void* scratch,
                      size_t scratch_bytes) {
    if (gp.K < 1 || gp.K > kMaxTerms) throw std::logic_error("term count out of range");
    if (!grid_windows_supported(in, gp)) throw UnsupportedError("grid or sample count too large for the window gridder");
    WinGeom wg = window_geometry(in, gp);
    const size_t max_records = max_window_records(in);
    const size_t nbins = static_cast<size_t>(wg.nbins), lbins = static_cast<size_t>(wg.lbins);
    const size_t nwt = static_cast<size_t>(wg.nwin_total);
    const bool coarse = wg.sup_log2 != 0;
    const uint32_t sub_cap = static_cast<uint32_t>(sub_piece_cap(wg, max_records));
    const BinBlocks bb = choose_bin_blocks(ctx, in, wg, std::min(scratch_bytes, kMaxBlockHistBytes / 8));
    if (std::max(bb.bytes, item_bytes(wg)) > scratch_bytes) throw std::logic_error("the window gridder's scratch is too small");
    const unsigned blocks = static_cast<unsigned>(bb.blocks);
    wg.block_size = bb.size;
    wg.use_lds = bb.use_lds ? 1 : 0;
    const bool count16 = bb.count16;
    const size_t nbands = (lbins + kLdsBins - 1) / kLdsBins;
    wg.band_bins = static_cast<int>((lbins + nbands - 1) / nbands);
    const size_t bin_lds = wg.use_lds ? static_cast<size_t>(wg.band_bins) * sizeof(uint32_t) : 0;
    const dim3 bin_grid(blocks, static_cast<unsigned>(bb.bands));

    // counts[0, lbins) | counts[lbins + 2, +12) = totals | the coarse bins' class counts and the slots handed out, kSup lbins
    // each | the halves' sizes (fit_shape).
    const size_t nsub = coarse ? kSup * lbins : 0;
    const size_t ncleared = lbins + 14 + 2 * nsub + kShapeWords;
    const WindowBuffers buf = window_buffers(ctx, in, wg, bb.use_lds);
    uint32_t *const counts = buf.counts, *const boff = buf.boff, *const cursor = buf.cursor, *const sums = buf.sums;
    uint32_t *const icount = buf.icount, *const ioff = buf.ioff;
    uint32_t* sub_counts = counts + lbins + 14;
    uint32_t* half_sizes = sub_counts + 2 * nsub;
    uint32_t* blockhist = static_cast<uint32_t*>(scratch);
    uint32_t* blocktot = blockhist + bb.nhist;
    uint16_t* blockcount16 = count16 ? reinterpret_cast<uint16_t*>(blocktot + bb.blocks * bb.bands) : nullptr;
    uint32_t* segsum = cursor + lbins + 8;
    uint32_t* coff = coarse ? segsum + (wg.use_lds ? kBinSegs * lbins : 0) : boff;
    const size_t ncounts = item_counts(wg);
    uint32_t* totals = counts + lbins + 2;
    const WRecords rec = {buf.records};

    // Wavefront items: one per window at most.  Pieces, and partial slots: as many as any sizes of the halves could
    // need, or as many as the scratch holds: then fit_shape sees to it that they suffice.
    const size_t most = most_pieces(wg.shape, max_records, 2 * nwt);
    const size_t room = std::min((scratch_bytes - item_bytes(wg)) / slot_bytes(gp), static_cast<size_t>(kAllSlotsFit - 1));
    const size_t max_slots = std::min(most, room);
    wg.slots = most <= room ? kAllSlotsFit : static_cast<uint32_t>(room);
    const size_t max_items = nwt + max_slots;
    float2* partial = static_cast<float2*>(scratch);
    float2* trash = partial + max_slots * static_cast<size_t>(gp.K) * kDenseCells;
    WReduce* red = reinterpret_cast<WReduce*>(trash + kTrash);
    WItem* items = reinterpret_cast<WItem*>(red + nwt);

    launch_fill(ctx, reinterpret_cast<float*>(counts), ncleared, 0.0f);
    // 16-bit LDS histograms (two bins per word) when there are also more blocks than CUs, so that
    // two can share a CU.  With one block per CU the halved LDS gains nothing and the packing
    // costs a little (snapshot rows at 64 channels: 35.9 against 33.9 us; preprocessed samples:
    // 50 against 64).
    const bool hist16 = count16 && blocks > static_cast<unsigned>(ctx->cu_count);
    const size_t count_lds = hist16 ? static_cast<size_t>((wg.band_bins + 1) / 2) * sizeof(uint32_t) : bin_lds;
    auto count = [&](auto kernel, auto* out) {
        allow_dynamic_lds(reinterpret_cast<const void*>(kernel), count_lds);
        kernel<<<bin_grid, kBinThreads, count_lds, ctx->stream>>>(in, gp, wg, counts, out, blocktot);
    };
    if (in.from_snapshot) {
        if (hist16) count(&k_win_count<true, true, uint16_t>, blockcount16);
        else if (count16) count(&k_win_count<true, false, uint16_t>, blockcount16);
        else count(&k_win_count<true, false, uint32_t>, blockhist);
    } else {
        if (hist16) count(&k_win_count<false, true, uint16_t>, blockcount16);
        else if (count16) count(&k_win_count<false, false, uint16_t>, blockcount16);
        else count(&k_win_count<false, false, uint32_t>, blockhist);
    }
    SVDI_LAUNCH_CHECK();
    const unsigned seg_grid = static_cast<unsigned>((kBinSegs * lbins + 255) / 256);
    if (wg.use_lds) {
        if (count16)
            k_bin_seg_sums<uint16_t><<<seg_grid, 256, 0, ctx->stream>>>(blockcount16, static_cast<int>(blocks),
                                                                       wg.lbins, segsum, counts);
        else
            k_bin_seg_sums<uint32_t><<<seg_grid, 256, 0, ctx->stream>>>(blockhist, static_cast<int>(blocks), wg.lbins,
                                                                       segsum, counts);
        SVDI_LAUNCH_CHECK();
    }
    launch_exclusive_scan(ctx, counts, coff, wg.use_lds ? nullptr : cursor, sums, lbins);
    // The halves' sizes, where they are needed, are counted on the way if the bins' offsets are there by now.
    const bool sizes = wg.slots != kAllSlotsFit;
    const unsigned size_blocks = sizes && wg.use_lds && !coarse ? half_size_blocks(wg) : 0u;
    if (wg.use_lds) {
        if (count16)
            k_bin_block_offsets<uint16_t><<<seg_grid + size_blocks, 256, 0, ctx->stream>>>(
                blockcount16, blockhist, static_cast<int>(blocks), wg.lbins, segsum, coff, size_blocks, wg, half_sizes);
        else
            k_bin_block_offsets<uint32_t><<<seg_grid + size_blocks, 256, 0, ctx->stream>>>(
                blockhist, blockhist, static_cast<int>(blocks), wg.lbins, segsum, coff, size_blocks, wg, half_sizes);
        SVDI_LAUNCH_CHECK();
    }
    const uint32_t limit = static_cast<uint32_t>(max_records);
    const WRecords scattered = coarse ? WRecords{reinterpret_cast<uint4*>(planes)} : rec;
    SubPiece* sub_list = reinterpret_cast<SubPiece*>(reinterpret_cast<uint4*>(planes) + max_records);
    if (in.from_snapshot) {
        allow_dynamic_lds(reinterpret_cast<const void*>(&k_win_scatter<true>), bin_lds);
        k_win_scatter<true><<<bin_grid, kBinThreads, bin_lds, ctx->stream>>>(in, gp, wg, blockhist, blocktot, cursor,
                                                                         scattered, limit, totals + 4, ctx->dev_err);
    } else {
        allow_dynamic_lds(reinterpret_cast<const void*>(&k_win_scatter<false>), bin_lds);
        k_win_scatter<false><<<bin_grid, kBinThreads, bin_lds, ctx->stream>>>(in, gp, wg, blockhist, blocktot, cursor,
                                                                          scattered, limit, totals + 4, ctx->dev_err);
    }
    SVDI_LAUNCH_CHECK();
    if (coarse) {
        k_sub_list<<<static_cast<unsigned>((lbins + 255) / 256), 256, 0, ctx->stream>>>(coff, wg, limit, sub_list, sub_cap,
                                                                                       totals + 8, boff);
        SVDI_LAUNCH_CHECK();
        const unsigned sub_grid = static_cast<unsigned>(std::min<size_t>(ctx->cu_count * kSubGroupsPerCu,
                                                                         (sub_cap + kSubWaves - 1) / kSubWaves));
        k_sub_bins<true><<<sub_grid, kSubWaves * 64, 0, ctx->stream>>>(sub_list, sub_cap, totals + 8, wg, scattered.r,
                                                                       sub_counts, sub_counts + nsub, boff, rec, limit);
        SVDI_LAUNCH_CHECK();
        k_sub_bins<false><<<sub_grid, kSubWaves * 64, 0, ctx->stream>>>(sub_list, sub_cap, totals + 8, wg, scattered.r,
                                                                        sub_counts, sub_counts + nsub, boff, rec, limit);
        SVDI_LAUNCH_CHECK();
    }
    if (sizes && size_blocks == 0) {
        k_win_half_sizes<<<half_size_blocks(wg), 256, 0, ctx->stream>>>(boff, wg, half_sizes);
        SVDI_LAUNCH_CHECK();
    }
    k_win_item_counts<<<static_cast<unsigned>((nwt + 255) / 256), 256, 0, ctx->stream>>>(boff, wg, icount, totals, half_sizes);
    SVDI_LAUNCH_CHECK();
    launch_exclusive_scan(ctx, icount, ioff, nullptr, sums, ncounts);
    k_win_item_write<<<static_cast<unsigned>((kItemLanes * nwt + 255) / 256), 256, 0, ctx->stream>>>(
        boff, ioff, wg, items, static_cast<uint32_t>(max_items), red, totals);
    SVDI_LAUNCH_CHECK();

    WindowJob job;
    static_assert(sizeof(WinGeom) <= sizeof(job.geom), "window geometry does not fit the job");
    std::memcpy(job.geom, &wg, sizeof wg);
    job.items = items;
    job.totals = totals;
    job.records = rec.r;
    job.planes = planes;
    job.partial = partial;
    job.trash = trash;
    job.reduce = red;
    job.max_slots = static_cast<uint32_t>(max_slots);
    job.K = gp.K;
    job.G = gp.G;
    job.prec = gp.prec;
    return job;
}

void contract_windows(svdi_context* ctx, const WindowJob* jobs, int count) {
    if (count < 1 || count > kMaxJobs) throw std::logic_error("window job count out of range");
    // The dense halves' blocks of sixteen terms and of eight go in launches of their own.  Sixteen have eight wavefronts and half
    // the batch, and multiply zeros for terms that a job does not have, so a job's last terms go with the eights where they are
    // no more (eight SKA-Low snapshots, one of them of 16 terms, as one planned batch: all in one launch of sixteens 6.9 to
    // 7.2 ms, 6.0 to 6.1 so; one of 24 terms: contraction by sixteens alone 1207 us, 1068 so).
    WinJobs wj = {}, by_terms[2] = {};
    wj.count = count;
    for (int j = 0; j < count; ++j) {
        if (jobs[j].prec != jobs[0].prec) throw std::logic_error("window jobs of one launch differ in precision");
        WinJob& d = wj.job[j];
        d.items = static_cast<const WItem*>(jobs[j].items);
        d.totals = jobs[j].totals;
        d.rec.r = static_cast<uint4*>(jobs[j].records);
        d.planes = jobs[j].planes;
        d.partial = jobs[j].partial;
        d.trash = jobs[j].trash;
        std::memcpy(&d.wg, jobs[j].geom, sizeof d.wg);
        d.K = jobs[j].K;
        d.G = jobs[j].G;
        auto add = [&](WinJobs& t, int k_lo, int k_hi) {
            if (k_lo >= k_hi) return;
            WinJob& part = t.job[t.count++] = d;
            part.k_lo = k_lo;
            part.k_hi = k_hi;
        };
        const int sixteens = d.K % 16 <= 8 ? d.K - d.K % 16 : d.K;
        add(by_terms[0], sixteens, d.K);
        add(by_terms[1], 0, sixteens);
    }
    const size_t tok = stage_begin(ctx, 5);
    const unsigned grid = static_cast<unsigned>(std::max(1, ctx->cu_count - ctx->grid_reserve));
    auto launch = [&](auto prec) {
        constexpr int P = decltype(prec)::value;
        using T = WinTraits<P>;
        auto dense = [&](auto mb) {
            constexpr int MB = decltype(mb)::value;
            using D = DenseTraits<P, MB>;
            allow_dynamic_lds(reinterpret_cast<const void*>(&k_win_dense<P, MB>), D::kLds);
            k_win_dense<P, MB><<<grid, D::kWaves * 64, D::kLds, ctx->stream>>>(by_terms[MB - 1]);
            SVDI_LAUNCH_CHECK();
        };
        if (by_terms[0].count != 0) dense(std::integral_constant<int, 1>());
        if (by_terms[1].count != 0) dense(std::integral_constant<int, 2>());
        constexpr size_t lds = sizeof(float) * T::kStageFloats * T::kWaves;
        allow_dynamic_lds(reinterpret_cast<const void*>(&k_win_grid<P>), lds);
        k_win_grid<P><<<grid, T::kWaves * 64, lds, ctx->stream>>>(wj);
    };
    const int prec = jobs[0].prec;
    if (prec == kPrecBf16) launch(std::integral_constant<int, kPrecBf16>());
    else if (prec == kPrecSingle) launch(std::integral_constant<int, kPrecSingle>());
    else if (prec == kPrecSplitC) launch(std::integral_constant<int, kPrecSplitC>());
    else launch(std::integral_constant<int, kPrecSplit3>());
    SVDI_LAUNCH_CHECK();
    stage_end(ctx, tok);
}

void reduce_windows(svdi_context* ctx, const WindowJob& job) {
    WinGeom wg;
    std::memcpy(&wg, job.geom, sizeof wg);
    k_win_reduce<<<4096, 256, 0, ctx->stream>>>(static_cast<const WReduce*>(job.reduce), job.totals, wg, job.G, job.K,
                                               job.max_slots, job.partial, job.planes);
    SVDI_LAUNCH_CHECK();
}

const uint32_t* launch_grid_windows(svdi_context* ctx, const SampleInput& in, const GridParams& gp,
                                    float2* planes, void* scratch, size_t scratch_bytes) {
    const WindowJob job = bin_windows(ctx, in, gp, planes, scratch, scratch_bytes);
    contract_windows(ctx, &job, 1);
    reduce_windows(ctx, job);
    return job.totals;
}

}  // namespace svdi
