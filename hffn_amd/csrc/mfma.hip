// Tile-densified MFMA path of the HFFN forward (gfx950, v_mfma_f32_32x32x16_f16).
//
// At high density and large token counts a tile of neurons has a nearly dense union support, so the layer is two
// contractions: Z[N, d_ff] = X[N, d_model] W_up^T, A = gelu(Z + b_up), Y[N, d_model] = A W_down^T + b_down.
// Every operand enters the MFMA units as a pair of fp16 "planes" (hi and lo parts) scaled by powers of two: the
// weights are densified once at load (one power of two per row, so that its largest entry lies in [1, 2)); the input
// X is split by a small kernel before the up GEMM (one power of two per token); the activations are split by the up
// GEMM's epilogue (one power of two per token and 128-neuron block). Each product is  a_hi b_hi + a_hi b_lo +
// a_lo b_hi  accumulated in fp32 (the lo*lo term, ~2^-22 relative, is dropped; bf16 weights take the first and last
// terms on the hi plane only, which holds them exactly down to 2^-14 of their row's largest magnitude; below that
// fp16 subnormals keep fewer bits, at most ~2^-25 of that magnitude per weight). The powers of two are undone
// exactly: the down GEMM rescales its accumulators at each 128-wide k block by the ratio of the blocks' powers of
// two, and the epilogues apply the last.
//
// Plane layout (K-chunk-major): k is cut into 32-wide k-tiles and each k-tile into four 16-byte chunks of 8 halves;
// for k-tile kt, part p (0 hi, 1 lo) and chunk c, the chunks of all rows follow one another:
//   planes[((((kt * 2 + p) * 4 + c) * rows + n) * 8 + k % 8]   with c = (k % 32) / 8.
// A block's tile of B rows is 8 runs of B * 16 contiguous bytes, and LDS keeps the same order, so the MFMA operand
// reads (32 lanes on 32 consecutive rows of one chunk) and the staging writes touch consecutive 16-byte blocks: no
// LDS bank conflicts, no padding. Token planes have a row count padded to kRowPad (rows past N are zeros in X and
// hold gelu(b_up) in A; their outputs are never stored); a call of at most 64 or 128 tokens writes and reads only
// the first 64 or 128 rows (rows_live).
//
// Two GEMM kernels: the streamed one (gemm_dma_kernel: 256 x 128 tiles whose k-tiles go from global memory straight
// into LDS, K split 2-32 ways by an estimate of the rounds of blocks and the partials' cost, partials added by
// separate passes; a down GEMM may take its first column tiles over all of K and split only the others) takes every
// shape whose tiles and splits give enough blocks; the register-staged one below (gemm_planes_kernel) remains for
// narrower layers at small N.
//
// Register-staged GEMM blocks: 4 waves in 2 x 2, each wave a (32 MI) x (32 NI) tile of 32x32 MFMA accumulators; the k loop stages
// 32-wide k-tiles of both planes through double-buffered LDS with plain 16-byte copies (one barrier per k-tile, the
// next tile's global loads in flight during the current tile's MFMAs). The grid is one-dimensional and remapped so
// that each of the 8 XCDs works on one compact group of output tiles (its L2 then holds the A rows and B columns
// those tiles share). A down projection with very few output tiles splits K over 2 blocks per tile; the block that
// finishes a tile last (an integer counter per tile) adds the partials in split order, so the result does not depend
// on which block ends first.
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"

namespace hffn {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // 16 bytes of plane: 8 halves

constexpr int kThreads = 256;
constexpr int kBK = 32;          // k per staged step, one plane k-tile
constexpr int kRuns = 8;         // (part, chunk) runs of a k-tile
constexpr uint32_t kXcds = 8;    // MI355X: 8 XCDs, workgroups dispatched round-robin over them
constexpr uint32_t kGroupM = 4;  // output-tile rows per group of the tile order
constexpr uint32_t kRowPad = 256;  // token planes hold a multiple of this many rows
constexpr uint32_t kActBlock = 128;  // neurons per activation power of two (the up GEMM's column tile)
constexpr uint32_t kKtPerActBlock = kActBlock / kBK;

// Every plane row (a token's inputs, a weight row, a token's activation block) is stored as hi + lo = v * 2^-e, e
// its power of two. e puts the row's largest |v| at 2^kPlaneLift .. 2^(kPlaneLift + 1) (below fp16's 65504 with room
// to spare), far above fp16's smallest normal 2^-14: lo, the residual of hi (at most 2^-11 of |hi|), is then a
// normal fp16 for every entry down to 2^-(kPlaneLift + 3) of the row's largest, and below that its absolute error
// (2^-25 after scaling) is 2^-(25 + kPlaneLift) of the largest. Scaled products stay below 2^26 per term, so fp32
// accumulation has no overflow at any K. Whoever reads a plane undoes e exactly (ldexp), so the lift is invisible
// outside the planes.
constexpr int kPlaneLift = 12;
// binades are clamped to +-kBinadeClamp before the lift: 2^(kBinadeClamp + kPlaneLift) is a finite float scale, and an
// activation block's binade fits an int8 (a row of only tiny entries, below 2^-100, keeps less than fp32's precision)
constexpr int kBinadeClamp = 100;

// floor(log2(m)) - kPlaneLift of a non-negative float given by its bits (clamped); -kPlaneLift for zero (any scale is
// exact for zeros). inf and NaN give the clamp's top, which scales them to themselves.
__device__ __forceinline__ int binade_of_bits(uint32_t bits) {
    const int e = bits == 0 ? 0 : static_cast<int>((bits >> 23) & 0xff) - 127;
    return min(max(e, -kBinadeClamp), kBinadeClamp) - kPlaneLift;
}

// Power of two of an activation block (a token's kActBlock neurons): binade_of_bits of its largest |v| rounded up to a
// multiple of kActBinadeStep (kPlaneLift is one, so the rounding is that of the true binade). The block's largest
// value scaled lies in 2^(kPlaneLift - 3) .. 2^(kPlaneLift + 1); neighbouring blocks of a token then mostly share their
// power of two, and the down GEMM has nothing to rescale between them. Range: -112 .. 88, an int8.
constexpr int kActBinadeStep = 4;
static_assert(kPlaneLift % kActBinadeStep == 0, "the lift keeps activation binades on their grid");
static_assert(kBinadeClamp + kPlaneLift + kActBinadeStep < 128, "activation binades fit an int8");
__device__ __forceinline__ int act_binade(uint32_t bits) {
    const int e = binade_of_bits(bits);
    return e >= 0 ? (e + kActBinadeStep - 1) / kActBinadeStep * kActBinadeStep : -(-e / kActBinadeStep * kActBinadeStep);
}

// Activation block binades are int8 (multiples of kActBinadeStep, -112 .. 88), block-major [d_ff / kActBlock][rows_pad]:
// the down GEMM transfers each activation block's binades of its 256 rows, one contiguous 256-byte run, straight into
// LDS. They travel through the GEMMs' int32 binade pointers (Up: out_exp; Down: a_exp), read and written as bytes.
__device__ __forceinline__ size_t act_exp_at(uint32_t rows_pad, uint32_t m, uint32_t block) {
    return static_cast<size_t>(block) * rows_pad + m;
}
__device__ __forceinline__ const int8_t* act_exps(const int32_t* p) { return reinterpret_cast<const int8_t*>(p); }
__device__ __forceinline__ int8_t* act_exps(int32_t* p) { return reinterpret_cast<int8_t*>(p); }

__device__ __forceinline__ uint32_t abs_bits(float v) { return __float_as_uint(v) & 0x7fffffffu; }

__device__ __forceinline__ void split(float v, _Float16& hi, _Float16& lo) {
    hi = static_cast<_Float16>(v);
    lo = static_cast<_Float16>(v - static_cast<float>(hi));
}

// Whether column k of a B plane lies in an odd chain of 2^bits columns (the chained GEMMs; kNoChains: never).
constexpr uint32_t kNoChains = 31;
constexpr uint32_t chain_bits(uint32_t ktiles) { return ktiles == 1 ? 5 : 1 + chain_bits(ktiles / 2); }  // 32 k per k-tile
__device__ __forceinline__ bool chain_odd(uint32_t k, uint32_t bits) { return (k >> bits) & 1u; }

// Index of element (row, k) of part p (0 hi, 1 lo) in planes of `rows` rows.
__device__ __forceinline__ size_t plane_at(uint32_t rows, uint32_t row, uint32_t k, uint32_t p) {
    return ((static_cast<size_t>(k / kBK) * kRuns + p * 4 + (k % kBK) / 8) * rows + row) * 8 + k % 8;
}

// ------------------------------------------------------------------------------------------ input planes
// X [M, K] fp32 (row stride ld; entries at k >= k_real read as zeros) -> planes of X [rows_pad, K] and e[row] =
// binade of max |x[row, :]| (rows M .. 8 * gridDim.x: zeros, e = -kPlaneLift; K a multiple of 256). A block takes 8 rows; its wave w takes k in [w K/4, (w + 1) K/4) in steps of 64,
// up to 4 steps (a chunk) at a time: in a step, lane l holds 8 consecutive k (piece l / 8) of row l % 8, so that the
// 8 lanes of a row read 256 contiguous bytes of it and the 8 lanes of a piece write the 8 rows' 16 bytes of one
// 128-byte run of the planes. First the row maxima (lanes, then the 4 waves through LDS), then the split; a wave
// whose range is one chunk keeps its values in registers, longer ranges are read again (from L2).
constexpr uint32_t kSplitBlockRows = 8;
constexpr uint32_t kSplitChunk = 256;  // k per chunk: 4 steps of 64
constexpr uint32_t kSplitWaves = kThreads / kWave;
constexpr uint32_t kTinyRow = static_cast<uint32_t>(127 - kBinadeClamp) << 23;  // bits of 2^-kBinadeClamp
// The work of kThreads threads (tid) on row group `group`; part: their maxima in LDS. Every thread of the block calls it.
__device__ __forceinline__ void split_rows(uint32_t (&part)[kSplitWaves][kSplitBlockRows], uint32_t tid, uint32_t group,
                                           const float* __restrict__ x, uint32_t M, uint32_t rows_pad, uint32_t K, uint32_t ld,
                                           uint32_t k_real, _Float16* __restrict__ planes, int32_t* __restrict__ e,
                                           bool mark = false) {
    constexpr uint32_t kWaves = kSplitWaves;
    const uint32_t lane = tid % kWave, wave = uniform(tid / kWave);
    const uint32_t r = lane % kSplitBlockRows, piece = lane / kSplitBlockRows;
    const uint32_t row = group * kSplitBlockRows + r;
    const uint32_t span = K / kWaves, k_begin = wave * span, k_end = k_begin + span;
    const float* src = x + static_cast<size_t>(row) * ld;
    const bool real = row < M;
    float v[4][8];
    const auto load_chunk = [&](uint32_t k0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
            const uint32_t k = k0 + 64 * i + 8 * piece;
            if (real && k0 + 64 * i < k_end && k < k_real) {
                const float* q = src + k;
                if (k + 8 <= k_real) {
                    a = *reinterpret_cast<const float4*>(q);
                    b = *reinterpret_cast<const float4*>(q + 4);
                } else {  // a piece across the end of the real columns: only those are read (the row may end there)
                    const uint32_t valid = k_real - k;
                    a.x = q[0];
                    if (valid > 1) a.y = q[1];
                    if (valid > 2) a.z = q[2];
                    if (valid > 3) a.w = q[3];
                    if (valid > 4) b.x = q[4];
                    if (valid > 5) b.y = q[5];
                    if (valid > 6) b.z = q[6];
                }
            }
            v[i][0] = a.x; v[i][1] = a.y; v[i][2] = a.z; v[i][3] = a.w;
            v[i][4] = b.x; v[i][5] = b.y; v[i][6] = b.z; v[i][7] = b.w;
        }
    };
    uint32_t m = 0;
    for (uint32_t k0 = k_begin; k0 < k_end; k0 += kSplitChunk) {
        load_chunk(k0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int q = 0; q < 8; ++q) m = max(m, abs_bits(v[i][q]));
    }
#pragma unroll
    for (int s = kSplitBlockRows; s < kWave; s <<= 1) m = max(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), s, kWave)));
    if (piece == 0) part[wave][r] = m;
    __syncthreads();
    uint32_t mx = part[0][r];
#pragma unroll
    for (uint32_t w = 1; w < kWaves; ++w) mx = max(mx, part[w][r]);
    const int be = binade_of_bits(mx);
    if (wave == 0 && piece == 0) e[row] = be;
    // mark: a row of only tiny entries, which the planes hold with fewer bits, becomes NaN (irregular_row takes it)
    const float scale = mark && mx != 0 && mx < kTinyRow ? __uint_as_float(0x7fc00000u) : ldexpf(1.0f, -be);
    for (uint32_t k0 = k_begin; k0 < k_end; k0 += kSplitChunk) {
        if (span > kSplitChunk) load_chunk(k0);  // one chunk: still in registers
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (k0 + 64 * i >= k_end) break;
            half8 h, l;
            const uint32_t k = k0 + 64 * i + 8 * piece;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                _Float16 hh, ll;
                split(v[i][q] * scale, hh, ll);
                h[q] = hh;
                l[q] = ll;
            }
            *reinterpret_cast<half8*>(planes + plane_at(rows_pad, row, k, 0)) = h;
            *reinterpret_cast<half8*>(planes + plane_at(rows_pad, row, k, 1)) = l;
        }
    }
}
__global__ __launch_bounds__(kThreads) void split_rows_kernel(const float* __restrict__ x, uint32_t M, uint32_t rows_pad,
                                                             uint32_t K, uint32_t ld, uint32_t k_real, _Float16* __restrict__ planes,
                                                             int32_t* __restrict__ e) {
    __shared__ uint32_t part[kSplitWaves][kSplitBlockRows];
    split_rows(part, threadIdx.x, blockIdx.x, x, M, rows_pad, K, ld, k_real, planes, e);
}

// Two matrices of the same columns in one launch (the operands of a sampled product).
__global__ __launch_bounds__(kThreads) void split_pair_kernel(const float* __restrict__ a, uint32_t a_rows, _Float16* __restrict__ a_planes,
                                                             int32_t* __restrict__ a_e, const float* __restrict__ b, uint32_t b_rows,
                                                             _Float16* __restrict__ b_planes, int32_t* __restrict__ b_e, uint32_t K,
                                                             uint32_t ld, uint32_t k_real) {
    __shared__ uint32_t part[kSplitWaves][kSplitBlockRows];
    const uint32_t a_blocks = a_rows / kSplitBlockRows;
    if (blockIdx.x < a_blocks) split_rows(part, threadIdx.x, blockIdx.x, a, a_rows, a_rows, K, ld, k_real, a_planes, a_e);
    else split_rows(part, threadIdx.x, blockIdx.x - a_blocks, b, b_rows, b_rows, K, ld, k_real, b_planes, b_e);
}

// --------------------------------------------------------------------------------------------- densify
// Row n of the dense matrix (a neuron of W_up, or an output of W_down^T) has its slots [off[n], off[n+1]) at columns
// idx[] (distinct within a row; the host checks it); densifying writes the whole row of both planes (zeros outside
// the support) and its binade. A block takes kDensRows consecutive rows and dens_chunk columns: the rows'
// maxima (a wave per row, over all its slots), then their hi/lo parts in its columns assembled in LDS (zeroed
// meanwhile, then each slot of the chunk in its column) and written out whole: for every 16-byte chunk run the block's rows are
// kDensRows consecutive 16-byte pieces, one 128-byte line per (run, row group). The rows are padded by 16 bytes in
// LDS so that the eight rows of a chunk fall in different banks; the tile (33 KB) leaves room for four blocks per CU.
constexpr uint32_t kDensRows = 8, kDensThreads = 512, kDensPad = 8;
constexpr uint32_t dens_chunk(uint32_t parts) { return parts == 2 ? 1024 : 2048; }  // columns of a block's tile (33 KB)
// Slots [8 q, 8 q + 8) of the compact rows: one 16-byte load of their indices, one (float32: two) of their values. vec:
// idx and val start on 16-byte boundaries.
template <typename V>
struct SlotPiece {
    static constexpr int kVals = 2 * static_cast<int>(sizeof(V));
    uint32_t ids[4], vals[kVals];
    // pos (float32, null for none): slot s holds val[pos[s]], one more load of the 8 positions, then 8 gathered values
    __device__ __forceinline__ void load(const int16_t* __restrict__ idx, const V* __restrict__ val, const int32_t* __restrict__ pos,
                                         int32_t q, int32_t nnz, bool vec) {
        const int32_t s = 8 * q;
        if (vec && s + 8 <= nnz) {
            const uint4 i4 = *reinterpret_cast<const uint4*>(idx + s);
            ids[0] = i4.x; ids[1] = i4.y; ids[2] = i4.z; ids[3] = i4.w;
            if constexpr (sizeof(V) == 4) {
                if (pos != nullptr) {
                    const int4 a = *reinterpret_cast<const int4*>(pos + s), b = *reinterpret_cast<const int4*>(pos + s + 4);
                    const int32_t at[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
                    for (int u = 0; u < 8; ++u) vals[u] = __float_as_uint(val[at[u]]);
                    return;
                }
            }
#pragma unroll
            for (int p = 0; p < kVals; p += 4) {
                const uint4 v4 = reinterpret_cast<const uint4*>(val + s)[p / 4];
                vals[p] = v4.x; vals[p + 1] = v4.y; vals[p + 2] = v4.z; vals[p + 3] = v4.w;
            }
            return;
        }
        // unaligned arrays, or the piece across the end of the arrays: slot by slot, those past nnz zero
#pragma unroll
        for (int i = 0; i < 4; ++i) ids[i] = 0;
#pragma unroll
        for (int i = 0; i < kVals; ++i) vals[i] = 0;
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (s + u < nnz) {
                ids[u / 2] |= static_cast<uint32_t>(static_cast<uint16_t>(idx[s + u])) << (16 * (u % 2));
                if constexpr (sizeof(V) == 2) vals[u / 2] |= static_cast<uint32_t>(val[s + u]) << (16 * (u % 2));
                else vals[u] = __float_as_uint(val[pos != nullptr ? pos[s + u] : s + u]);
            }
    }
    __device__ __forceinline__ uint32_t index(int u) const { return u % 2 ? ids[u / 2] >> 16 : ids[u / 2] & 0xffffu; }
    __device__ __forceinline__ float value(int u) const {
        if constexpr (sizeof(V) == 2) return __uint_as_float(u % 2 ? vals[u / 2] & 0xffff0000u : vals[u / 2] << 16);
        else return __uint_as_float(vals[u]);
    }
};

// The slots [begin, end) of one row on a wave, in pieces of 8 on 8-slot boundaries, 64 at a time (lane l: pieces first + 64
// q). The first piece of a lane is requested at construction and held; the further ones of rows of more than 504 slots are
// read at each pass.
template <typename V>
struct RowSlots {
    static constexpr int32_t kStride = kWave;
    const int16_t* idx;
    const V* val;
    const int32_t* pos;
    int32_t begin, end, first, last, nnz;
    bool vec;
    SlotPiece<V> held;
    __device__ __forceinline__ RowSlots(const int16_t* __restrict__ i, const V* __restrict__ v, const int32_t* __restrict__ positions, int32_t b,
                                        int32_t e, int32_t slots, bool aligned, uint32_t lane)
        : idx(i), val(v), pos(positions), begin(b), end(e), first((b >> 3) + static_cast<int32_t>(lane)), last(e > b ? (e + 7) >> 3 : 0),
          nnz(slots), vec(aligned) {
        if (first < last) held.load(idx, val, pos, first, nnz, vec);
    }
    // f(index, value, inside the row) of every slot of the lane's pieces
    template <typename F>
    __device__ __forceinline__ void each(const F& f) const {
        if (first >= last) return;
        piece(held, first, f);
        for (int32_t q = first + kStride; q < last; q += kStride) {
            SlotPiece<V> p;
            p.load(idx, val, pos, q, nnz, vec);
            piece(p, q, f);
        }
    }
    template <typename F>
    __device__ __forceinline__ void piece(const SlotPiece<V>& p, int32_t q, const F& f) const {
#pragma unroll
        for (int u = 0; u < 8; ++u)
            f(p.index(u), p.value(u), static_cast<uint32_t>(8 * q + u - begin) < static_cast<uint32_t>(end - begin));
    }
};
template <uint32_t PARTS>
struct DensTile {
    _Float16 tile[PARTS][kDensRows][dens_chunk(PARTS) + kDensPad];
};
struct DensSide {
    const int32_t* off;
    const int16_t* idx;
    const void* val;
    const int32_t* pos;          // null, or (float32) the slots' places in val
    uint32_t rows, rows_pad, k;  // real rows; rows and columns of the planes
    uint32_t bits;               // chain_odd
    bool vec;
    _Float16* planes;
    int32_t* exps;
};
// A side's blocks: (row group, column chunk), chunk-major.
constexpr uint32_t dens_blocks(uint32_t rows_pad, uint32_t k, uint32_t parts) {
    return (rows_pad + kDensRows - 1) / kDensRows * ((k + dens_chunk(parts) - 1) / dens_chunk(parts));
}
constexpr uint32_t kDensOccupancy = 8;  // waves per SIMD of four blocks: at most 64 VGPRs

// PARTS 1 (bfloat16 planes of one call): the hi plane alone, the only one its GEMMs read. Rows `rows` .. rows_pad - 1 and
// columns past the indices are zeros.
template <typename V, uint32_t PARTS>
__device__ __forceinline__ void densify(DensTile<PARTS>& lds, const DensSide& side, uint32_t block) {
    static_assert(kDensRows * 16 == 128, "a row group's pieces of one chunk run fill one 128-byte line");
    auto& tile = lds.tile;
    constexpr uint32_t kDensChunk = dens_chunk(PARTS);
    static_assert(kDensThreads / kWave == kDensRows, "a wave per row");
    const uint32_t tid = threadIdx.x, lane = tid % kWave, row = uniform(tid / kWave);
    const uint32_t groups = (side.rows_pad + kDensRows - 1) / kDensRows, chunk = block / groups;
    const uint32_t group = side.pos != nullptr ? xcd_order(block % groups, groups) : block % groups;  // values by position: neighbours share lines
    const uint32_t r0 = group * kDensRows, n = r0 + row, c0 = chunk * kDensChunk;
    const uint32_t width = min(kDensChunk, side.k - c0), pieces = width / 8;  // width: a multiple of 32
    const bool real = n < side.rows;
    RowSlots<V> slots(side.idx, static_cast<const V*>(side.val), side.pos, real ? side.off[n] : 0, real ? side.off[n + 1] : 0, side.off[side.rows],
                      side.vec, lane);
    // the tile zeroed while the slots are in flight
    for (uint32_t i = tid; i < PARTS * sizeof(tile[0]) / 16; i += kDensThreads) reinterpret_cast<uint4*>(tile)[i] = make_uint4(0, 0, 0, 0);
    uint32_t m = 0;
    slots.each([&](uint32_t, float v, bool inside) { m = max(m, inside ? abs_bits(v) : 0u); });
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = max(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), o, kWave)));
    const int e = binade_of_bits(m);
    __syncthreads();  // the tile is zeroed
    slots.each([&](uint32_t column, float v, bool inside) {
        // a slot of another row or column block goes to the row's padding, which nothing reads: no branch per slot
        const uint32_t c = column - c0, at = inside && c < width ? c : kDensChunk;
        _Float16 hi, lo;
        split(ldexpf(chain_odd(column, side.bits) ? -v : v, -e), hi, lo);
        tile[0][row][at] = hi;
        if constexpr (PARTS == 2) tile[1][row][at] = lo;
    });
    __syncthreads();
    // thread t: row t % 8, pieces t / 8, t / 8 + 64, ... of every part (no division by the width: two per 16 bytes moved
    // cost more than the moves)
    const uint32_t rr = tid % kDensRows;
    if (r0 + rr < side.rows_pad)
        for (uint32_t j = tid / kDensRows; j < pieces; j += kDensThreads / kDensRows)
#pragma unroll
            for (uint32_t part = 0; part < PARTS; ++part)
                *reinterpret_cast<uint4*>(side.planes + plane_at(side.rows_pad, r0 + rr, c0 + j * 8, part)) =
                    *reinterpret_cast<const uint4*>(&tile[part][rr][j * 8]);
    if (chunk == 0 && lane == 0 && n < side.rows_pad) side.exps[n] = e;
}
template <typename V>
__global__ __launch_bounds__(kDensThreads, kDensOccupancy) void densify_kernel(DensSide side) {
    __shared__ __attribute__((aligned(16))) DensTile<2> lds;
    densify<V, 2>(lds, side, blockIdx.x);
}

// What a call that densifies its own planes (launch_prefill) needs before its first GEMM, in one launch: the planes of
// both sides from the compact rows and the input planes of x. The first split_blocks split x, kSplitGroups groups of 8
// rows a block, the next trans_blocks transpose it (training), the next up_blocks densify W_up, the others W_down (the
// split, a block's longest work, first: last it was the launch's tail, 46 us instead of 34.5 at 1999 tokens on 2048 x 8192).
// MI355X: 7.8 us on 512 x 2048 at 20 % (float32, 128 tokens), 17 on 1024 x 4096 at 10 % with uneven rows, 28 on 2048 x
// 8192 at 20 % (bfloat16, 128 tokens; 72 with single slots a lane in place of 8, 38 in blocks of 1024 threads, two per CU).
// A block is a chain of four round trips (offsets, slots, LDS, stores): many small blocks cover one another.
constexpr uint32_t kSplitGroups = kDensThreads / kThreads;
template <typename V>
__global__ __launch_bounds__(kDensThreads, kDensOccupancy) void prefill_prep_kernel(DensSide up, DensSide down, uint32_t up_blocks,
                                                                                   uint32_t split_blocks, uint32_t trans_blocks,
                                                                                   const float* __restrict__ x, uint32_t M,
                                                                                   uint32_t rows_pad, uint32_t K, uint32_t ld,
                                                                                   _Float16* __restrict__ planes, int32_t* __restrict__ e,
                                                                                   float* __restrict__ x_t, uint32_t t_ld, uint32_t tiles_c,
                                                                                   bool vectors) {
    constexpr uint32_t kParts = sizeof(V) == 2 ? 1 : 2;
    __shared__ __attribute__((aligned(16))) DensTile<kParts> lds;
    const uint32_t g = uniform(threadIdx.x / kThreads);
    uint32_t block = blockIdx.x;
    if (block < split_blocks) {
        using Parts = uint32_t[kSplitGroups][kSplitWaves][kSplitBlockRows];
        split_rows(reinterpret_cast<Parts&>(lds)[g], threadIdx.x % kThreads, block * kSplitGroups + g, x, M, rows_pad, K, ld, ld, planes, e, x_t == nullptr);
        return;
    }
    block -= split_blocks;
    if (block < trans_blocks) {
        // training: x [M, ld] transposed too, a tile per group (a tile past the rows moves nothing)
        static_assert(kThreads == kTransThreads && sizeof(TransposeTile) * kSplitGroups <= sizeof(lds), "a tile per group of threads");
        const uint32_t tile = block * kSplitGroups + g;
        transpose_tile(reinterpret_cast<TransposeTile*>(&lds)[g], threadIdx.x % kThreads, tile / tiles_c * kTransRows,
                       tile % tiles_c * kTransCols, x, x_t, M, ld, ld, t_ld, vectors);
        return;
    }
    block -= trans_blocks;
    if (block < up_blocks) densify<V, kParts>(lds, up, block);
    else densify<V, kParts>(lds, down, block - up_blocks);
}

// ------------------------------------------------------------------------------------ irregular results
// What the planes of a call cannot hold is computed again as the lane-per-token kernels compute it: from the float32
// operands in stored slot order, the same bits. A token's planes turn an infinity, a NaN, a magnitude beyond fp16's range
// past the clamp of its power of two (2^104) and (mark above) a row of only tiny entries into NaN, and the zeros of the
// dense planes carry that to every output of the token; a weight beyond the clamp does so to its output or, through its
// neuron's activation, to the token's every output. So the kernel that writes y sees it: an output that is not finite. Its
// wave then walks that token's outputs in its columns. Calls whose outputs are finite take
// the same time as without it where K is split (512 x 2048 at 20 %, 128 tokens: 26.6 us; 2048 x 8192 at 20 % bfloat16, 1999
// tokens: 304.5) and on row tiles of 64 (512 x 2048, 3000 tokens: 69.2 and 69.0), 2 us more on row tiles of 128 in one split
// (6000 tokens: 109.5 -> 112.4); a launch of its own that looked at the tokens cost 2.2-5.6 us, a check by the whole block 1-2.
struct Walk {
    const float* x;  // [M, d]
    const int32_t* up_off;
    const int16_t* up_idx;
    const void* up_val;
    const float* b_up;
    const int32_t* down_off;
    const int16_t* down_idx;
    const void* down_val;
    const float* b_down;
    uint32_t d, h;
};
__device__ __forceinline__ bool finite(float v) { return abs_bits(v) < 0x7f800000u; }
__device__ __forceinline__ bool finite(const float4& v) { return finite(v.x) && finite(v.y) && finite(v.z) && finite(v.w); }
// y[row, o] for o in [o0, o_end), at most THREADS of them, by THREADS threads (a block, or a wave): the token's activations
// CHUNK neurons at a time in `act` (LDS, free for it), thread i the slots of output o0 + i among them (ascending within a
// row, so the chunks in turn are the stored order). Every one of the threads calls it.
template <typename V, uint32_t THREADS, uint32_t CHUNK>
__device__ __forceinline__ void irregular_row(const Walk& a, float* act, uint32_t row, uint32_t o0, uint32_t o_end, float* y) {
    const auto meet = [] {
        if constexpr (THREADS == kWave) {  // a wave's LDS accesses keep their order: only the compiler has to
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            __builtin_amdgcn_wave_barrier();
        } else {
            __syncthreads();
        }
    };
    const float* x = a.x + static_cast<size_t>(row) * a.d;
    const V *up_val = static_cast<const V*>(a.up_val), *down_val = static_cast<const V*>(a.down_val);
    const uint32_t thread = threadIdx.x % THREADS, o = o0 + thread;
    const bool mine = o < o_end;
    int32_t slot = mine ? a.down_off[o] : 0;
    const int32_t end = mine ? a.down_off[o + 1] : 0;
    float out = 0.0f;
    for (uint32_t c0 = 0; c0 < a.h; c0 += CHUNK) {
        for (uint32_t r = c0 + thread; r < min(c0 + CHUNK, a.h); r += THREADS) {
            float z = 0.0f;
            const int32_t last = a.up_off[r + 1];
#pragma unroll 4
            for (int32_t s = a.up_off[r]; s < last; ++s) z = fmaf(widen(up_val[s]), x[static_cast<uint16_t>(a.up_idx[s])], z);
            act[r - c0] = gelu(a.b_up[r] + z);
        }
        meet();
        for (; slot < end; ++slot) {
            const uint32_t at = static_cast<uint16_t>(a.down_idx[slot]) - c0;
            if (at >= CHUNK) break;
            out = fmaf(widen(down_val[slot]), act[at], out);
        }
        meet();
    }
    if (mine) y[static_cast<size_t>(row) * a.d + o] = out + a.b_down[o];
}

// ------------------------------------------------------------------------------------------------ GEMM
// Up: the up GEMM with the GELU epilogue writing activation planes. Down: the down GEMM writing y or split partials.
// UpSplit: the up GEMM over a k split, writing fp32 partial sums (no bias, no GELU) for act_planes_kernel.
enum class Epi { Up, Down, UpSplit };

struct Tile {
    uint32_t m, n, split;
};

// Workgroup id -> (row tile, column tile, k split). The first 8 * floor(T / 8) ids are dealt so that XCD j (ids
// j, j + 8, ...) takes the j-th contiguous run of the tile order; the tile order walks groups of kGroupM tile rows
// column by column, so a run is a compact block of tiles.
__device__ __forceinline__ Tile tile_of(uint32_t id, uint32_t tiles_m, uint32_t tiles_n, uint32_t splits) {
    const uint32_t total = tiles_m * tiles_n * splits;
    const uint32_t per = total / kXcds;
    uint32_t t = id < kXcds * per ? (id % kXcds) * per + id / kXcds : id;
    const uint32_t per_split = tiles_m * tiles_n;
    Tile tile;
    tile.split = t / per_split;
    t %= per_split;
    const uint32_t group = t / (kGroupM * tiles_n);
    const uint32_t first = group * kGroupM;
    const uint32_t rows = min(tiles_m - first, kGroupM);
    const uint32_t within = t % (kGroupM * tiles_n);
    tile.m = first + within % rows;
    tile.n = within / rows;
    return tile;
}

// One k-tile of a block's operands in flight: ARPT 16-byte chunks of the A planes and BRPT of the B planes per thread.
template <int ARPT, int BRPT>
struct StageRegs {
    u32x4 a[ARPT];
    u32x4 b[BRPT];
};

// Global loads of k-tile kt: thread t copies run t / 32 (part, chunk) of rows t % 32 + 32 j of each operand.
template <int ARPT, int BRPT>
__device__ __forceinline__ void load_stage(StageRegs<ARPT, BRPT>& r, const _Float16* a_src, size_t a_stride, const _Float16* b_src,
                                           size_t b_stride, uint32_t kt) {
#pragma unroll
    for (int j = 0; j < ARPT; ++j) r.a[j] = *reinterpret_cast<const u32x4*>(a_src + kt * a_stride + 32 * j * 8);
#pragma unroll
    for (int j = 0; j < BRPT; ++j) r.b[j] = *reinterpret_cast<const u32x4*>(b_src + kt * b_stride + 32 * j * 8);
}

template <int BM, int BN, int ARPT, int BRPT>
__device__ __forceinline__ void store_stage(const StageRegs<ARPT, BRPT>& r, _Float16* s_a, _Float16* s_b, uint32_t run,
                                            uint32_t row) {
#pragma unroll
    for (int j = 0; j < ARPT; ++j) *reinterpret_cast<u32x4*>(s_a + (run * BM + row + 32 * j) * 8) = r.a[j];
#pragma unroll
    for (int j = 0; j < BRPT; ++j) *reinterpret_cast<u32x4*>(s_b + (run * BN + row + 32 * j) * 8) = r.b[j];
}

// Row m (within the block tile) of accumulator register r of tile row i of wave row wm, lane `lane`: accumulator r
// of a 32x32 tile holds row 8 (r / 4) + 4 (lane / 32) + r % 4 and column lane % 32.
template <int BM>
__device__ __forceinline__ uint32_t acc_row(uint32_t wm, int i, int r, uint32_t lane) {
    return wm * (BM / 2) + i * 32 + 8 * (r / 4) + 4 * (lane / 32) + r % 4;
}

// The same for waves of WR rows each (the streamed GEMM's 4- or 8-wave blocks).
template <uint32_t WR>
__device__ __forceinline__ uint32_t wave_row(uint32_t wm, int i, int r, uint32_t lane) {
    return wm * WR + i * 32 + 8 * (r / 4) + 4 * (lane / 32) + r % 4;
}

// C[M, Ncol] = A[M, K] B[Ncol, K]^T from planes. Up: A = X planes (power of two per row), epilogue bias + GELU,
// writes the activation planes (K-chunk-major over the d_ff neurons) and one power of two per (row, BN block).
// Down: A = activation planes (power of two per row and kActBlock-wide k block), epilogue bias, writes Y fp32.
template <Epi EPI, int MI, int NI, bool LO_B, int SPLITS>
__global__ __launch_bounds__(kThreads) void gemm_planes_kernel(
    const _Float16* __restrict__ a_planes,  // [K / 32][8][rows_pad][8]
    const int32_t* __restrict__ a_exp,      // Up: [rows_pad]; Down: [K / kActBlock, rows_pad] (act_exp_at)
    const _Float16* __restrict__ b_planes,  // [K / 32][8][Ncol][8]
    const int32_t* __restrict__ b_exp,      // [Ncol]
    const float* __restrict__ bias,         // [Ncol]
    float* __restrict__ out,                // Down: [M, Ncol] fp32 row-major
    _Float16* __restrict__ out_planes,      // Up: activation planes [Ncol / 32][8][rows_pad][8]
    int32_t* __restrict__ out_exp,          // Up: [Ncol / BN, rows_pad] activation block binades (act_exp_at)
    float* __restrict__ partials,           // SPLITS > 1: [SPLITS, M, Ncol] partial sums
    int32_t* __restrict__ counters,         // SPLITS > 1: [tiles], zero between calls
    uint32_t M, uint32_t rows_pad, uint32_t Ncol, uint32_t K) {
    constexpr int BM = 64 * MI, BN = 64 * NI;
    constexpr int ARPT = BM / 32, BRPT = BN / 32;  // chunks per thread and k-tile (8 runs x 32 rows per block pass)

    // staged k-tiles, [buffer][part][chunk][row][8 halves] of A then of B; the up epilogue reuses it for its output
    __shared__ __attribute__((aligned(16))) _Float16 smem[2 * kRuns * (BM + BN) * 8];
    const auto s_a = [&](uint32_t buffer) { return smem + buffer * (kRuns * BM * 8); };
    const auto s_b = [&](uint32_t buffer) { return smem + 2 * kRuns * BM * 8 + buffer * (kRuns * BN * 8); };
    __shared__ int32_t row_e[2][BM];  // Up: [0] the row binades; Down: the row binades of the current / next k block
    __shared__ uint32_t row_max[2][BM];
    __shared__ int32_t last;

    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const uint32_t wm = wave / 2, wn = wave % 2;
    const uint32_t tiles_m = rows_pad / BM, tiles_n = Ncol / BN;
    const Tile tile = tile_of(blockIdx.x, tiles_m, tiles_n, SPLITS);
    const uint32_t m0 = tile.m * BM, n0 = tile.n * BN;
    const uint32_t ktiles = K / kBK;
    const uint32_t k_begin = tile.split * ktiles / SPLITS, k_end = (tile.split + 1) * ktiles / SPLITS;

    if (tid < BM) {
        if constexpr (EPI == Epi::Up) row_e[0][tid] = a_exp[m0 + tid];
        else row_e[(k_begin / kKtPerActBlock) & 1][tid] = act_exps(a_exp)[act_exp_at(rows_pad, m0 + tid, k_begin / kKtPerActBlock)];
    }

    const uint32_t run = tid / 32, row = tid % 32;
    const _Float16* a_src = a_planes + (static_cast<size_t>(run) * rows_pad + m0 + row) * 8;
    const _Float16* b_src = b_planes + (static_cast<size_t>(run) * Ncol + n0 + row) * 8;
    const size_t a_stride = static_cast<size_t>(kRuns) * rows_pad * 8, b_stride = static_cast<size_t>(kRuns) * Ncol * 8;
    StageRegs<ARPT, BRPT> regs;

    floatx16 acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    int32_t next_e = 0;  // Down: binades of the activation block of the k-tile in flight, when it starts one
    if (k_begin < k_end) {
        load_stage<ARPT, BRPT>(regs, a_src, a_stride, b_src, b_stride, k_begin);
        store_stage<BM, BN, ARPT, BRPT>(regs, s_a(0), s_b(0), run, row);
        if (k_begin + 1 < k_end) {
            load_stage<ARPT, BRPT>(regs, a_src, a_stride, b_src, b_stride, k_begin + 1);
            if constexpr (EPI == Epi::Down) {
                if ((k_begin + 1) % kKtPerActBlock == 0 && tid < BM)
                    next_e = act_exps(a_exp)[act_exp_at(rows_pad, m0 + tid, (k_begin + 1) / kKtPerActBlock)];
            }
        }
    }
    __syncthreads();
    for (uint32_t kt = k_begin; kt < k_end; ++kt) {
        const int buf = (kt - k_begin) & 1;
        if constexpr (EPI == Epi::Down) {
            // a new activation block: bring the accumulators to its power of two (exact), and fetch the next one's
            if (kt % kKtPerActBlock == 0 && kt != k_begin) {
                const uint32_t kb = kt / kKtPerActBlock;
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const uint32_t m = acc_row<BM>(wm, i, r, lane);
                        const float f = ldexpf(1.0f, row_e[(kb - 1) & 1][m] - row_e[kb & 1][m]);
#pragma unroll
                        for (int j = 0; j < NI; ++j) acc[i][j][r] *= f;
                    }
            }
        }
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const uint32_t chunk = kk * 2 + lane / 32;
            half8 ah[MI], al[MI], bh[NI], bl[NI];
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const uint32_t r = wm * (BM / 2) + i * 32 + lane % 32;
                ah[i] = *reinterpret_cast<const half8*>(s_a(buf) + (chunk * BM + r) * 8);
                al[i] = *reinterpret_cast<const half8*>(s_a(buf) + ((4 + chunk) * BM + r) * 8);
            }
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                const uint32_t r = wn * (BN / 2) + j * 32 + lane % 32;
                bh[j] = *reinterpret_cast<const half8*>(s_b(buf) + (chunk * BN + r) * 8);
                if constexpr (LO_B) bl[j] = *reinterpret_cast<const half8*>(s_b(buf) + ((4 + chunk) * BN + r) * 8);
            }
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[i], bh[j], acc[i][j], 0, 0, 0);
                    if constexpr (LO_B) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[i], bl[j], acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[i], bh[j], acc[i][j], 0, 0, 0);
                }
        }
        if (kt + 1 < k_end) {
            store_stage<BM, BN, ARPT, BRPT>(regs, s_a(buf ^ 1), s_b(buf ^ 1), run, row);
            if constexpr (EPI == Epi::Down) {
                // the next activation block's binades travel with the stage loads: requested with k-tile 4 kb, they
                // reach LDS with its store, one barrier before the rescale at k-tile 4 kb reads them
                if ((kt + 1) % kKtPerActBlock == 0 && tid < BM) row_e[((kt + 1) / kKtPerActBlock) & 1][tid] = next_e;
            }
            if (kt + 2 < k_end) {
                load_stage<ARPT, BRPT>(regs, a_src, a_stride, b_src, b_stride, kt + 2);
                if constexpr (EPI == Epi::Down) {
                    if ((kt + 2) % kKtPerActBlock == 0 && tid < BM)
                        next_e = act_exps(a_exp)[act_exp_at(rows_pad, m0 + tid, (kt + 2) / kKtPerActBlock)];
                }
            }
        }
        __syncthreads();
    }
    const int e_last = EPI == Epi::Up ? 0 : static_cast<int>(((k_end - 1) / kKtPerActBlock) & 1);

    if constexpr (EPI == Epi::Up) {
        // v = gelu(z + b): first its largest |v| per row over the tile's BN neurons (one tile row at a time, to keep
        // few registers live), then v again, split with that row's power of two into the activation planes
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            uint32_t lane_max[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) lane_max[r] = 0;
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                const uint32_t col = n0 + wn * (BN / 2) + j * 32 + lane % 32;
                const int ce = b_exp[col];
                const float cb = bias[col];
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    lane_max[r] = max(lane_max[r],
                                      abs_bits(gelu(ldexpf(acc[i][j][r], row_e[0][acc_row<BM>(wm, i, r, lane)] + ce) + cb)));
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                uint32_t v = lane_max[r];
#pragma unroll
                for (int s = 16; s >= 1; s >>= 1) v = max(v, static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), s, kWave)));
                if (lane % 32 == 0) row_max[wn][acc_row<BM>(wm, i, r, lane)] = v;
            }
        }
        __syncthreads();
        if (tid < BM) {
            const int e = act_binade(max(row_max[0][tid], row_max[1][tid]));
            row_e[1][tid] = e;
            act_exps(out_exp)[act_exp_at(rows_pad, m0 + tid, tile.n)] = static_cast<int8_t>(e);
        }
        // the planes go out through LDS, half the block's rows (one wave row) at a time: the waves of that row store
        // v as fp32 [row][col], then every thread splits 8 consecutive columns of one row and writes 16 bytes per
        // part, 64 consecutive rows of one chunk per wave (1 KB contiguous)
        constexpr uint32_t R = BM / 2, kLd = BN + 8;
        static_assert(R * kLd * sizeof(float) <= sizeof(smem), "the epilogue tile fits the staging LDS");
        float* tile_v = reinterpret_cast<float*>(smem);
#pragma unroll
        for (uint32_t half = 0; half < 2; ++half) {
            __syncthreads();
            if (wm == half) {
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const uint32_t c = wn * (BN / 2) + j * 32 + lane % 32;
                    const int ce = b_exp[n0 + c];
                    const float cb = bias[n0 + c];
#pragma unroll
                    for (int i = 0; i < MI; ++i)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const uint32_t m = acc_row<BM>(wm, i, r, lane);
                            tile_v[(m - half * R) * kLd + c] = gelu(ldexpf(acc[i][j][r], row_e[0][m] + ce) + cb);
                        }
                }
            }
            __syncthreads();
            for (uint32_t q = tid; q < R * (BN / 8); q += kThreads) {
                const uint32_t m = q % R, chunk = q / R, k = n0 + chunk * 8;
                const float scale = ldexpf(1.0f, -row_e[1][half * R + m]);
                const float* src = tile_v + m * kLd + chunk * 8;
                half8 h, l;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    _Float16 hh, ll;
                    split(src[e] * scale, hh, ll);
                    h[e] = hh;
                    l[e] = ll;
                }
                *reinterpret_cast<half8*>(out_planes + plane_at(rows_pad, m0 + half * R + m, k, 0)) = h;
                *reinterpret_cast<half8*>(out_planes + plane_at(rows_pad, m0 + half * R + m, k, 1)) = l;
            }
        }
    } else if constexpr (SPLITS == 1) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            const uint32_t col = n0 + wn * (BN / 2) + j * 32 + lane % 32;
            const int ce = b_exp[col];
            const float cb = bias[col];
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t m = acc_row<BM>(wm, i, r, lane);
                    if (m0 + m < M) out[static_cast<size_t>(m0 + m) * Ncol + col] = ldexpf(acc[i][j][r], row_e[e_last][m] + ce) + cb;
                }
        }
    } else {
        // every split writes its partial (powers of two undone), then the block that completes the tile adds them in
        // split order
        const size_t plane_size = static_cast<size_t>(M) * Ncol;
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            const uint32_t col = n0 + wn * (BN / 2) + j * 32 + lane % 32;
            const int ce = b_exp[col];
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t m = acc_row<BM>(wm, i, r, lane);
                    acc[i][j][r] = ldexpf(acc[i][j][r], row_e[e_last][m] + ce);
                    if (m0 + m < M) partials[tile.split * plane_size + static_cast<size_t>(m0 + m) * Ncol + col] = acc[i][j][r];
                }
        }
        __threadfence();
        __syncthreads();
        if (tid == 0) {
            const uint32_t counter = tile.m * tiles_n + tile.n;
            const int32_t arrived = atomicAdd(&counters[counter], 1);
            last = arrived == SPLITS - 1;
            if (last) counters[counter] = 0;  // every split of this tile has arrived: ready for the next call
        }
        __syncthreads();
        if (!last) return;
        __threadfence();
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            const uint32_t col = n0 + wn * (BN / 2) + j * 32 + lane % 32;
            const float cb = bias[col];
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t m = acc_row<BM>(wm, i, r, lane);
                    if (m0 + m >= M) continue;
                    const size_t at = static_cast<size_t>(m0 + m) * Ncol + col;
                    float total = 0.0f;
#pragma unroll
                    for (int s = 0; s < SPLITS; ++s) {
                        const float p = s == static_cast<int>(tile.split)
                                            ? acc[i][j][r]
                                            : __hip_atomic_load(partials + s * plane_size + at, __ATOMIC_RELAXED,
                                                                __HIP_MEMORY_SCOPE_AGENT);
                        total = s == 0 ? p : total + p;
                    }
                    out[at] = total + cb;
                }
        }
    }
}

// ------------------------------------------------------------------------------- streamed GEMM (LDS DMA)
// The large-N GEMM: 256 x 128 block tiles of 8 waves (4 x 2, 64 x 64 outputs each: two waves per SIMD, so that one
// wave's barrier and transfer waits are covered by the other's MFMAs), one block per CU, and k-tiles streamed
// straight from global memory into a ring of kDmaStages LDS stages by global_load_lds (16 bytes per lane, no
// registers on the way). In the middle of k-tile kt (its first 16-wide step multiplied, its second read into
// registers) the block waits for stage kt + 1, meets at a barrier and requests stage kt + kDmaStages into the slot of
// kt; each stage is thus requested kDmaStages - 1 k-tiles before its wait, and the MFMAs never wait for LDS reads.
// Before the first k-tile the lower half of the waves requests the first stages while the upper half loads the
// activation binades of the tile's rows and k range (the down GEMM). Same products and order as gemm_planes_kernel.
constexpr int kDmaStages = 3;
constexpr int kDmaBM = 256, kDmaBN = 128;
constexpr int kDmaWaves = 8;  // waves per block: two per SIMD, 64 x 64 outputs each
constexpr uint32_t kDmaMaxActBlocks = 40;  // activation blocks of one down split held in LDS (int8 binades)
constexpr uint32_t kDmaLoRuns = 32;        // activation blocks more per ring slot with bfloat16 weights (its B lo plane)

// Workgroup barrier without the memory fence of __syncthreads (whose release would also wait for every LDS DMA in
// flight); LDS visibility is ensured by the wait_loads before it.
__device__ __forceinline__ void block_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Waits until at most min(R, later) stages of L transfers each are in flight: the wave's oldest have landed.
template <int R, int L>
__device__ __forceinline__ void wait_stages(uint32_t later) {
    if constexpr (R == 0) wait_loads<0>();
    else if (later >= static_cast<uint32_t>(R)) wait_loads<R * L>();
    else wait_stages<R - 1, L>(later);
}

// LIVE < BM (one row tile of up to LIVE tokens): only the first LIVE rows of A are transferred and multiplied; the
// waves whose rows are all padding only transfer and meet at the barriers. The live rows get the same
// products in the same order as with LIVE = BM, and the padding rows' accumulators stay zero, as zero A rows leave
// them, so the results are bitwise those of the full tile.
//
// CHAIN > 0 (the calls whose planes are densified per call, which stand in for the compact store's paths): the MFMA
// accumulators run over CHAIN k-tiles only, then are added to a second set of float32 sums (Down: brought from the
// activation block's power of two to 1 on the way, exact, in place of the rescale) and start from zero again. One
// chain of MFMAs over all of K loses 6.5e-7 of the result (2048 x 8192 at 20 %, bfloat16, 1999 tokens, against 64 bits),
// three times as much as the tiles path it stands in for (2.05e-7); in chains of one activation block it keeps 2.0e-7, for
// ~4 % of the GEMMs' time.
//
// The MFMAs' own sums are biased downwards (mean error -1.3e-8 of a pre-activation's deviation, whatever its sign). So the
// B planes of these calls hold -w in every odd chain's columns (chain_odd), whose sums are subtracted: the bias cancels
// (4e-10).
//
// BM < 256 (those calls too): row tiles of 128 (waves of 32 x 64) or 64 (32 x 32), where 256 rows by 128 columns leave
// CUs idle or would have to be split over K, with the partials' round trip and another launch. A k-tile of such a tile
// is multiplied faster than its transfer arrives, so the ring holds as many stages as LDS takes. 768 x 3072 (float32) at
// 512 tokens: up projection 18.2 + 6.4 us in 3 splits of 256 rows and their activation pass, 17.6 us with 64 rows (no
// split); down 18.7 -> 14.6 us.
constexpr int dma_stages(int bm) { return bm == 64 ? 6 : bm == 128 ? 4 : kDmaStages; }
//
// WALK (a chained down GEMM of one split, which writes y): irregular outputs are walked (irregular_row). An instance of its
// own: in the one that writes partials the code costs 1-3 us of 127 without being reached.
template <Epi EPI, bool LO_B, int LIVE, int CHAIN, int BM = kDmaBM, bool WALK = false>
__global__ __launch_bounds__(64 * kDmaWaves) void gemm_dma_kernel(
    const _Float16* __restrict__ a_planes,  // [K / 32][8][rows_pad][8]
    const int32_t* __restrict__ a_exp,      // Up: [rows_pad]; Down: [K / kActBlock, rows_pad] (act_exp_at)
    const _Float16* __restrict__ b_planes,  // [K / 32][8][Ncol][8]
    const int32_t* __restrict__ b_exp,      // [Ncol]
    const float* __restrict__ bias,         // [Ncol]
    float* __restrict__ out,                // Down: y [M, Ncol] (splits == 1) or partials [splits, M, Ncol]; UpSplit: partials
    _Float16* __restrict__ out_planes,      // Up: activation planes [Ncol / 32][8][rows_pad][8]
    int32_t* __restrict__ out_exp,          // Up: [Ncol / BN, rows_pad] activation block binades (act_exp_at)
    uint32_t M, uint32_t rows_pad, uint32_t Ncol, uint32_t K, uint32_t splits,
    uint32_t whole_n,                       // Down: column tiles below whole_n take all of K and write y into `out`
    float* __restrict__ part,               // Down, whole_n > 0: the other column tiles' partials [splits, M, Ncol - whole_n BN]
    uint32_t cols,                          // real columns (<= Ncol, a multiple of 4): biases and y end there
    Walk walk) {                            // WALK: what irregular outputs are computed again from
    // 256 rows: 8 waves in 4 x 2, 64 x 64 outputs each (two waves per SIMD)
    constexpr int W = kDmaWaves, MI = BM == kDmaBM ? 2 : 1, NI = BM == 64 ? 1 : 2, BN = kDmaBN, S = dma_stages(BM);
    constexpr uint32_t kT = 64 * W, kWaveRows = 32 * MI, kWaveCols = 32 * NI, kWavesN = BN / kWaveCols;
    static_assert(kWaveRows * (W / kWavesN) == BM, "the waves cover the block's rows");
    static_assert(BM == kDmaBM || (LIVE == BM && (CHAIN > 0 || EPI == Epi::UpSplit)), "narrower row tiles: whole ones, in chains or split products");
    constexpr bool FOLD = CHAIN > 0;
    static_assert(!FOLD || EPI != Epi::Down || CHAIN == static_cast<int>(kKtPerActBlock), "a down chain has one power of two per row");
    static_assert(LIVE == BM || LIVE == 128 || LIVE == 64, "live rows: the whole tile, its first half or first quarter");
    constexpr uint32_t kStage = kRuns * (BM + BN) * 8;  // halves per stage
    // Down: the activation binades of up to kDmaMaxActBlocks blocks sit in e_tab; with bfloat16 weights the B lo plane of
    // every ring slot (8 KB, never transferred) holds 32 blocks more, so that a tile can take all of a wide K
    constexpr uint32_t kLoRegion = kRuns * BM * 8 + kRuns / 2 * BN * 8, kLoRuns = kRuns / 2 * BN * 8 * 2 / BM;
    constexpr uint32_t kMaxActBlocks = LO_B || BM != kDmaBM ? kDmaMaxActBlocks : kDmaMaxActBlocks + S * kLoRuns;
    static_assert(BM != kDmaBM || kLoRuns == kDmaLoRuns, "the host's plan counts the ring's spare runs alike");
    constexpr int kRowRuns = LIVE / 64;                  // 64-row runs of A transferred per (part, chunk)
    // runs of B transferred per k-tile: both planes, or the hi plane alone when the lo plane is not read (LO_B false)
    constexpr int kRunsB = LO_B ? kRuns : kRuns / 2;
    constexpr int kLoadsA = kRowRuns * kRuns / W, kLoadsB = BN * kRunsB / kWave / W;  // DMA instructions per wave
    static_assert(kLoadsA * W == kRowRuns * kRuns && kLoadsB * W == BN * kRunsB / kWave, "the transfers divide over the waves");
    constexpr int kLoads = kLoadsA + kLoadsB;
    static_assert(kLoads * S + (kMaxActBlocks + W - 1) / W < 64, "the prologue's transfers of a wave fit vmcnt");
    // multiplied 32-row tiles of a live wave (its rows start at wm * kWaveRows; LIVE is a multiple of kWaveRows)
    constexpr int MIL = LIVE >= static_cast<int>(kWaveRows) ? MI : LIVE / 32;

    __shared__ __attribute__((aligned(16))) _Float16 smem[S * kStage];
    __shared__ __attribute__((aligned(16))) int32_t e_row[1][BM];  // Up: x binades
    __shared__ __attribute__((aligned(16))) int8_t e_tab[EPI == Epi::Down ? kDmaMaxActBlocks : 1][EPI == Epi::Down ? BM : 1];  // Down: [block][row]
    // Down: the BM binades of the k range's activation block c (c < kMaxActBlocks): a row of e_tab, or a 256-byte run in
    // the unused B lo plane of ring slot (c - kDmaMaxActBlocks) / kLoRuns
    const auto etab = [&](uint32_t c) -> int8_t* {
        if (LO_B || BM != kDmaBM || c < kDmaMaxActBlocks) return &e_tab[c][0];
        const uint32_t o = c - kDmaMaxActBlocks;
        return reinterpret_cast<int8_t*>(smem + (o / kLoRuns) * kStage + kLoRegion) + (o % kLoRuns) * BM;
    };

    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = uniform(tid / kWave);
    const uint32_t wm = wave / kWavesN, wn = wave % kWavesN;
    // wave-uniform: this wave's rows hold tokens (a constant for a full tile)
    const bool live = LIVE == BM || wm * kWaveRows < static_cast<uint32_t>(LIVE);
    const uint32_t tiles_m = BM == kDmaBM ? rows_pad / BM : (M + BM - 1) / BM, tiles_n = Ncol / BN;
    // the first tiles_m * whole_n blocks: column tiles 0 .. whole_n - 1 over all of K (one round of long blocks first);
    // the others: the remaining column tiles, K split `splits` ways (whole_n 0: every tile split alike)
    const uint32_t whole_blocks = tiles_m * whole_n;
    const bool whole = blockIdx.x < whole_blocks;
    Tile tile = whole ? tile_of(blockIdx.x, tiles_m, whole_n, 1) : tile_of(blockIdx.x - whole_blocks, tiles_m, tiles_n - whole_n, splits);
    if (!whole) tile.n += whole_n;
    const uint32_t nsplit = whole ? 1 : splits;
    const uint32_t m0 = tile.m * BM, n0 = tile.n * BN;
    const uint32_t ktiles = K / kBK;
    // K split on k-tiles (Down: on activation blocks)
    constexpr uint32_t kUnit = EPI == Epi::Down ? kKtPerActBlock : 1;
    const uint32_t k_begin = tile.split * (ktiles / kUnit) / nsplit * kUnit, k_end = (tile.split + 1) * (ktiles / kUnit) / nsplit * kUnit;
    const uint32_t kb0 = k_begin / kKtPerActBlock;

    // piece q of wave w's share of a stage: a run of 64 rows (1 KB) of A (pieces below kLoadsA), then of B; its
    // element offsets within a k-tile's planes and within a ring slot
    const auto piece = [&](uint32_t w, int q, uint32_t& src, uint32_t& dst) {
        if (q < kLoadsA) {
            const uint32_t at = w * kLoadsA + q, run = at / kRowRuns, rb = at % kRowRuns;
            src = (run * rows_pad + m0 + rb * 64) * 8;
            dst = (run * BM + rb * 64) * 8;
        } else {
            const uint32_t at = w * kLoadsB + (q - kLoadsA), run = at / (BN / 64), rb = at % (BN / 64);
            src = (run * Ncol + n0 + rb * 64) * 8;
            dst = kRuns * BM * 8 + (run * BN + rb * 64) * 8;
        }
    };
    // this wave's pieces, computed once: the lanes' byte offsets from the k-tile's base (vector registers) and the
    // LDS offsets (wave-uniform), so that a transfer in the k loop takes the k-tile's base pointer of its operand
    const size_t a_kt = static_cast<size_t>(kRuns) * rows_pad * 8, b_kt = static_cast<size_t>(kRuns) * Ncol * 8;
    uint32_t src_lane[kLoads], dst_off[kLoads];
#pragma unroll
    for (int q = 0; q < kLoads; ++q) {
        uint32_t src;
        piece(wave, q, src, dst_off[q]);
        src_lane[q] = src * 2 + lane * 16;
    }
    const auto issue_piece = [&](uint32_t kt, uint32_t slot, int q) {
        const _Float16* base = q < kLoadsA ? a_planes + kt * a_kt : b_planes + kt * b_kt;
        dma16(base, src_lane[q], smem + slot * kStage + dst_off[q]);
    };
    const auto issue = [&](uint32_t kt, uint32_t slot) {
#pragma unroll
        for (int q = 0; q < kLoads; ++q) issue_piece(kt, slot, q);
    };

    // Prologue: every wave requests its pieces of the first stages, after the binades of the tile's rows, which go
    // straight into LDS as well (Up: the x binades, one 1 KB run; Down: the split's activation blocks, one 256-byte run
    // of int8 each, block c from wave c % W). vmcnt retires in order within a wave, so once the first stage has landed
    // so have they: the block meets once, and no wave holds a register for them. (Loaded into registers by half of the
    // waves and reduced to change masks there, the down GEMM's binades kept the block 6.5 us in its prologue, where
    // the first stage lands in 2.5-3 us.)
    const uint32_t steps = k_end - k_begin;  // at least 1
    if constexpr (EPI == Epi::Down) {
        const uint32_t blocks = (k_end - k_begin) / kKtPerActBlock;  // at least one: K is split on activation blocks
        const int8_t* tab = act_exps(a_exp);
        for (uint32_t c = wave; c < blocks; c += W)
            if (lane < BM / 4) dma4(tab + act_exp_at(rows_pad, m0, kb0 + c), lane * 4, etab(c));
    } else {
        if (wave == 0 && lane < BM / 4) dma16(a_exp + m0, lane * 16, &e_row[0][0]);
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (static_cast<uint32_t>(s) < steps) issue(k_begin + s, s);
    // stage k_begin has landed (later stages may be in flight), and with it the binades; then the block meets
    if constexpr (S == 3) {
        if (steps >= 3) wait_loads<2 * kLoads>();
        else if (steps == 2) wait_loads<kLoads>();
        else wait_loads<0>();
    } else {
        wait_stages<S - 1, kLoads>(steps - 1);
    }
    block_barrier();

    floatx16 acc[MI][NI], sum[FOLD ? MI : 1][FOLD ? NI : 1];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[i][j][r] = 0.0f;
                if constexpr (FOLD) sum[i][j][r] = 0.0f;
            }

    // operand fragments of one 16-wide k step (chunk pair kk of a k-tile)
    struct Frags {
        half8 ah[MI], al[MI], bh[NI], bl[NI];
    };
    const auto load = [&](Frags& f, uint32_t slot, int kk) {
        if (!live) return;
        const _Float16* s_a = smem + slot * kStage;
        const _Float16* s_b = s_a + kRuns * BM * 8;
        const uint32_t chunk = kk * 2 + lane / 32;
#pragma unroll
        for (int i = 0; i < MIL; ++i) {
            const uint32_t r = wm * kWaveRows + i * 32 + lane % 32;
            f.ah[i] = *reinterpret_cast<const half8*>(s_a + (chunk * BM + r) * 8);
            f.al[i] = *reinterpret_cast<const half8*>(s_a + ((4 + chunk) * BM + r) * 8);
        }
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            const uint32_t r = wn * kWaveCols + j * 32 + lane % 32;
            f.bh[j] = *reinterpret_cast<const half8*>(s_b + (chunk * BN + r) * 8);
            if constexpr (LO_B) f.bl[j] = *reinterpret_cast<const half8*>(s_b + ((4 + chunk) * BN + r) * 8);
        }
    };
    const auto multiply = [&](const Frags& f) {
        if (!live) return;
#pragma unroll
        for (int i = 0; i < MIL; ++i)
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.ah[i], f.bh[j], acc[i][j], 0, 0, 0);
                if constexpr (LO_B) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.ah[i], f.bl[j], acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.al[i], f.bh[j], acc[i][j], 0, 0, 0);
            }
    };
    // The same products with stage kt's transfers spread among them, one after every few MFMAs: a transfer's issue
    // holds the wave while the CU's address unit takes the other waves' transfers, and in-order issue would
    // otherwise keep the MFMA unit idle behind a burst of them. sched_barrier pins the order.
    constexpr int kProducts = LO_B ? 3 : 2, kMfmas = MI * NI * kProducts;
    static_assert(kMfmas >= kLoads, "at most one transfer per MFMA");
    const auto multiply_issuing = [&](const Frags& f, uint32_t kt, uint32_t slot, bool transfer) {
        if constexpr (LIVE < BM) {  // few MFMAs: the stage's transfers go out first, in one burst
            if (transfer) issue(kt, slot);
            __builtin_amdgcn_sched_barrier(0);
            multiply(f);
            return;
        }
#pragma unroll
        for (int p = 0; p < kProducts; ++p)  // product-major: consecutive MFMAs accumulate into different tiles
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const half8& a = p == kProducts - 1 ? f.al[i] : f.ah[i];
                    const half8& b = (LO_B && p == 1) ? f.bl[j] : f.bh[j];
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, acc[i][j], 0, 0, 0);
                    const int m = (p * MI + i) * NI + j;  // MFMAs issued so far, less one
                    if ((m + 1) * kLoads % kMfmas < kLoads) {   // kLoads transfers evenly over kMfmas MFMAs
                        __builtin_amdgcn_sched_barrier(0);
                        if (transfer) issue_piece(kt, slot, (m + 1) * kLoads / kMfmas - 1);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
    };

    // Software pipeline over half k-tiles: the fragments of the next 16-wide step are read from LDS while the MFMAs
    // of the current one run, and the block meets once per k-tile, between its two steps (after every wave has read
    // all of k-tile kt and before anyone reads k-tile kt + 1), where the slot of kt is refilled with kt + kDmaStages.
    // The first stages went out in the prologue.
    // a new activation block at k-tile kt: bring the accumulators to its power of two (exact), when some row of the
    // wave changes it (lane l checks the wave's row l; binades are multiples of kActBinadeStep, so changes are rare;
    // checked here rather than for all blocks after the prologue, which measured 0.5 % slower); accumulator registers
    // 4g .. 4g + 3 hold 4 consecutive rows, so one 4-byte read per block and group
    // the chain that ends before k-tile kt, into the float32 sums
    const auto fold = [&](uint32_t kt) {
        if constexpr (FOLD) {
            if (!live) return;
            const float sign = ((kt - 1) / CHAIN) & 1u ? -1.0f : 1.0f;  // odd chains: the B planes hold -w
            const uint32_t kb = (kt - 1) / kKtPerActBlock - kb0;
#pragma unroll
            for (int i = 0; i < MIL; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    uint32_t e = 0;
                    if constexpr (EPI == Epi::Down)
                        e = *reinterpret_cast<const uint32_t*>(etab(kb) + wave_row<kWaveRows>(wm, i, 4 * g, lane));
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        const float f = EPI == Epi::Down ? ldexpf(sign, static_cast<int8_t>(e >> (8 * b))) : sign;
#pragma unroll
                        for (int j = 0; j < NI; ++j) {
                            const int r = 4 * g + b;
                            sum[i][j][r] = fmaf(acc[i][j][r], f, sum[i][j][r]);
                            acc[i][j][r] = 0.0f;
                        }
                    }
                }
        }
    };
    const auto rescale = [&](uint32_t kt) {
        if constexpr (FOLD) {
            if (kt % CHAIN == 0 && kt != k_begin) fold(kt);
        } else if constexpr (EPI == Epi::Down) {
            const uint32_t kb = kt / kKtPerActBlock - kb0;
            if (kt % kKtPerActBlock != 0 || kt == k_begin || !live) return;
            const uint32_t own = wm * kWaveRows + lane;
            if (__builtin_amdgcn_ballot_w64(etab(kb - 1)[own] != etab(kb)[own]) != 0) {
#pragma unroll
                for (int i = 0; i < MIL; ++i)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const uint32_t m = wave_row<kWaveRows>(wm, i, 4 * g, lane);
                        const uint32_t before = *reinterpret_cast<const uint32_t*>(etab(kb - 1) + m);
                        const uint32_t now = *reinterpret_cast<const uint32_t*>(etab(kb) + m);
#pragma unroll
                        for (int b = 0; b < 4; ++b) {
                            const int d = static_cast<int8_t>(before >> (8 * b)) - static_cast<int8_t>(now >> (8 * b));
                            const float f = ldexpf(1.0f, d);
#pragma unroll
                            for (int j = 0; j < NI; ++j) acc[i][j][4 * g + b] *= f;
                        }
                    }
            }
        }
    };
    // A wave raises its issue priority (s_setprio) for the MFMA run that carries the stage's transfers, so that of the two
    // waves of a SIMD the one with products ready issues ahead of the other's LDS reads (same box, alternating builds:
    // the 2.8B layer's up GEMM 415-427 -> 401-402 us and down GEMM 466-468 -> 444-458 us, the 410M layer's up GEMM
    // ~56 -> 54.5 us; the raised priority around the other MFMA run gave nothing on the down GEMM and lost ~2 % on the
    // up GEMM).
    const auto raise_priority = [] { __builtin_amdgcn_s_setprio(1); };
    const auto lower_priority = [] {
        __builtin_amdgcn_sched_barrier(0);  // the MFMA run ends here
        __builtin_amdgcn_s_setprio(0);
    };
    Frags f0, f1;
    load(f0, 0, 0);
    // every k-tile but the last (peeled, so that no path reaches the second step's MFMAs without the barrier's wait
    // for the first step's reads: the compiler's own LDS waits then never hold them for the reads just issued)
    // (sched_barrier keeps each step's LDS reads ahead of the MFMAs they overlap)
    for (uint32_t kt = k_begin; kt + 1 < k_end; ++kt) {
        const uint32_t it = kt - k_begin, slot = it % S;
        rescale(kt);
        wait_loads<63>();  // this step's reads, issued a step ago, are in: the next reads do not hold its MFMAs
        load(f1, slot, 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(f0);
        // stage kt + 1 has landed, the S - 2 after it may be in flight
        if constexpr (S == 3) {
            if (kt + 2 < k_end) wait_loads<kLoads>();
            else wait_loads<0>();
        } else {
            wait_stages<S - 2, kLoads>(k_end - kt - 2);
        }
        wait_loads<63>();  // the same LDS wait on every path, where the compiler's wait tracking sees it
        block_barrier();
        load(f0, (it + 1) % S, 0);
        __builtin_amdgcn_sched_barrier(0);
        raise_priority();
        multiply_issuing(f1, kt + S, slot, kt + S < k_end);  // straight-line MFMAs: one set of accumulators
        lower_priority();
    }
    rescale(k_end - 1);
    wait_loads<63>();
    load(f1, (steps - 1) % S, 1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(f0);
    multiply(f1);
    fold(k_end);
    __syncthreads();
    const auto result = [&](int i, int j, int r) -> float {
        if constexpr (FOLD) return sum[i][j][r];
        else return acc[i][j][r];
    };

    if constexpr (EPI == Epi::Up) {
        // v = gelu(z + b) once per element into an fp32 [BM][BN] tile in LDS; then thread t takes block row t: the
        // largest |v| of the row over the tile's BN neurons gives its power of two, and the row goes out split, 16
        // bytes per part and chunk (the 256 threads write 256 consecutive rows of one chunk: 4 KB contiguous)
        constexpr uint32_t kLd = BN + 4;
        static_assert(BM * kLd * sizeof(float) <= sizeof(smem), "the epilogue tile fits the staging LDS");
        float* tile_v = reinterpret_cast<float*>(smem);
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            const uint32_t c = wn * kWaveCols + j * 32 + lane % 32;
            const int ce = b_exp[n0 + c];
            const float cb = FOLD && n0 + c >= cols ? 0.0f : bias[n0 + c];  // a padding neuron (chained calls only): gelu(0) = 0
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t m = wave_row<kWaveRows>(wm, i, r, lane);
                    const float z = ldexpf(result(i, j, r), e_row[0][m] + ce) + cb;
                    tile_v[m * kLd + c] = FOLD ? gelu_near(z) : gelu(z);
                }
        }
        __syncthreads();
        // H threads per block row (2, 4 or 8 with 256, 128 or 64 rows: lanes h of a row are adjacent), each a BN / H-wide part
        constexpr uint32_t H = kT / BM;
        const uint32_t row = tid / H, part = tid % H;
        const float* row_v = tile_v + row * kLd;
        uint32_t largest = 0;
#pragma unroll 8
        for (uint32_t c = part * (BN / H); c < (part + 1) * (BN / H); c += 4) {
            const float4 v = *reinterpret_cast<const float4*>(row_v + c);
            largest = max(largest, max(max(abs_bits(v.x), abs_bits(v.y)), max(abs_bits(v.z), abs_bits(v.w))));
        }
#pragma unroll
        for (uint32_t off = 1; off < H; off <<= 1)
            largest = max(largest, static_cast<uint32_t>(__shfl_xor(static_cast<int>(largest), static_cast<int>(off), kWave)));
        const int e = act_binade(largest);
        if (part == 0) act_exps(out_exp)[act_exp_at(rows_pad, m0 + row, tile.n)] = static_cast<int8_t>(e);
        const float scale = ldexpf(1.0f, -e);
#pragma unroll 4
        for (uint32_t chunk = part * (BN / 8 / H); chunk < (part + 1) * (BN / 8 / H); ++chunk) {
            const float4 u = *reinterpret_cast<const float4*>(row_v + chunk * 8);
            const float4 w = *reinterpret_cast<const float4*>(row_v + chunk * 8 + 4);
            const float v[8] = {u.x, u.y, u.z, u.w, w.x, w.y, w.z, w.w};
            half8 h, l;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                _Float16 hh, ll;
                split(v[q] * scale, hh, ll);
                h[q] = hh;
                l[q] = ll;
            }
            *reinterpret_cast<half8*>(out_planes + plane_at(rows_pad, m0 + row, n0 + chunk * 8, 0)) = h;
            *reinterpret_cast<half8*>(out_planes + plane_at(rows_pad, m0 + row, n0 + chunk * 8, 1)) = l;
        }
    } else {
        // y (Down, one split) or this split's partial, powers of two undone: through an fp32 [BM][BN] tile in LDS, so
        // that every thread writes 16 bytes (a wave: two rows of BN columns)
        constexpr uint32_t kLd = BN + 4;
        static_assert(BM * kLd * sizeof(float) <= sizeof(smem), "the epilogue tile fits the staging LDS");
        float* tile_v = reinterpret_cast<float*>(smem);
        const uint32_t kb_last = (k_end - 1) / kKtPerActBlock - kb0;
        // the last activation block's binades held in a ring slot (a wide k range), which the tile below overwrites,
        // are first copied to e_row (block-uniform condition)
        const bool last_in_ring = EPI == Epi::Down && !FOLD && kb_last >= kDmaMaxActBlocks;
        if (last_in_ring) {
            if (tid < BM) e_row[0][tid] = etab(kb_last)[tid];
            __syncthreads();
        }
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            const uint32_t c = wn * kWaveCols + j * 32 + lane % 32;
            const int ce = b_exp[n0 + c];
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t m = wave_row<kWaveRows>(wm, i, r, lane);
                    // (a folded down sum is in units of 1 already)
                    const int ea = EPI != Epi::Down || last_in_ring ? e_row[0][m] : FOLD ? 0 : static_cast<int>(e_tab[kb_last][m]);
                    tile_v[m * kLd + c] = ldexpf(result(i, j, r), ea + ce);
                }
        }
        __syncthreads();
        // y (whole k range) or this split's partial: [splits, M, Ncol], or with whole_n > 0 [splits, M, Ncol - whole_n BN]
        // over the split column tiles only
        // (y: the real columns only; partials: the padded ones as well)
        const bool apart = nsplit > 1 && whole_n > 0, is_y = FOLD && EPI == Epi::Down && nsplit == 1;  // (padded: chained calls only)
        const uint32_t ld = apart ? Ncol - whole_n * BN : is_y ? cols : Ncol, c0 = n0 - (apart ? whole_n * BN : 0);
        float* target = nsplit == 1 ? out : (whole_n > 0 ? part : out) + static_cast<size_t>(tile.split) * M * ld;
        const uint32_t c_end = is_y ? cols - min(cols, n0) : BN;
        const bool add_bias = EPI == Epi::Down && nsplit == 1 && bias != nullptr;  // no bias: the training gx product
        float irregular = 0.0f;  // WALK: 0 while every output of the thread is finite, else NaN
        for (uint32_t q = tid; q < BM * (BN / 4); q += kT) {
            const uint32_t m = q / (BN / 4), c = (q % (BN / 4)) * 4;
            if (m0 + m >= M) break;  // rows ascend with q
            if (FOLD && c >= c_end) continue;
            float4 v = *reinterpret_cast<const float4*>(tile_v + m * kLd + c);
            if (add_bias) {
                const float4 b = *reinterpret_cast<const float4*>(bias + n0 + c);
                v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w;
            }
            if constexpr (WALK) irregular = fmaf(v.x, 0.0f, fmaf(v.y, 0.0f, fmaf(v.z, 0.0f, fmaf(v.w, 0.0f, irregular))));
            *reinterpret_cast<float4*>(target + static_cast<size_t>(m0 + m) * ld + c0 + c) = v;
        }
        if constexpr (WALK) {
            // by the wave that stored them, beside the tile (other waves may still read it)
            constexpr uint32_t kWalkChunk = 256, kBeside = BM * kLd, kPassRows = kT / (BN / 4), kWaveRowsStored = kWave / (BN / 4);
            static_assert(FOLD && EPI == Epi::Down && (kBeside + W * kWalkChunk) * 4 <= S * kStage * 2, "the activations fit the ring");
            if (__builtin_amdgcn_ballot_w64(irregular != 0.0f) == 0) return;
            for (uint32_t i = 0; i < BM / kPassRows; ++i) {
                const uint32_t m = m0 + i * kPassRows + tid / (BN / 4), c = tid % (BN / 4) * 4;
                const bool odd = m < M && c < c_end && !finite(*reinterpret_cast<const float4*>(out + static_cast<size_t>(m) * cols + n0 + c));
                for (uint32_t r = 0; r < kWaveRowsStored; ++r) {
                    if (__builtin_amdgcn_ballot_w64(odd && lane / (BN / 4) == r) == 0) continue;
                    for (uint32_t o = n0; o < min(n0 + BN, cols); o += kWave)
                        irregular_row<std::conditional_t<LO_B, float, uint16_t>, kWave, kWalkChunk>(
                            walk, tile_v + kBeside + wave * kWalkChunk, m0 + i * kPassRows + wave * kWaveRowsStored + r, o,
                            min(min(o + kWave, n0 + BN), cols), out);
                }
            }
        }
    }
}

// One thread's four columns; whether they are finite.
__device__ __forceinline__ bool reduce_quad(const float* __restrict__ partials, const float* __restrict__ bias, float* __restrict__ y,
                                            uint32_t M, uint32_t splits, uint32_t width, uint32_t cols, uint32_t m, uint32_t quad,
                                            uint32_t c) {
    const size_t quads = static_cast<size_t>(M) * (width / 4), i = static_cast<size_t>(m) * (width / 4) + quad;
    const float4* p = reinterpret_cast<const float4*>(partials);
    float4 t = p[i];
    for (uint32_t s0 = 1; s0 < splits; s0 += 8) {  // 8 loads in flight, added in split order
        float4 u[8];
#pragma unroll
        for (uint32_t q = 0; q < 8; ++q)
            if (s0 + q < splits) u[q] = p[(s0 + q) * quads + i];
#pragma unroll
        for (uint32_t q = 0; q < 8; ++q)
            if (s0 + q < splits) {
                t.x += u[q].x; t.y += u[q].y; t.z += u[q].z; t.w += u[q].w;
            }
    }
    if (bias != nullptr) {  // none for the training gx product
        const float4 b = *reinterpret_cast<const float4*>(bias + c);
        t.x += b.x; t.y += b.y; t.z += b.z; t.w += b.w;
    }
    *reinterpret_cast<float4*>(y + static_cast<size_t>(m) * cols + c) = t;
    return finite(t);
}
// y[m, c0 + c] = sum over splits (in split order) of partials[s, m, c] + bias[c0 + c] for the partials' width columns
// below cols (y rows of cols); 4 columns per thread, kReduceRows rows x 256 columns per block.
// V: float or uint16_t, the walk's values (irregular_row; the calls whose planes are densified per call), or void: none.
constexpr uint32_t kReduceRows = 4;
template <typename V>
__global__ __launch_bounds__(kThreads) void reduce_splits_kernel(const float* __restrict__ partials, const float* __restrict__ bias,
                                                                float* __restrict__ y, uint32_t M, uint32_t splits, uint32_t width,
                                                                uint32_t c0, uint32_t cols, Walk walk) {
    const uint32_t m = blockIdx.x * kReduceRows + threadIdx.x / 64, quad = blockIdx.y * 64 + threadIdx.x % 64, c = c0 + quad * 4;
    const bool live = m < M && quad * 4 < width && c < cols;
    const bool odd = live && !reduce_quad(partials, bias, y, M, splits, width, cols, m, quad, c);
    if constexpr (!std::is_void_v<V>) {
        constexpr uint32_t kChunk = 512;
        __shared__ float act[kReduceRows][kChunk];
        static_assert(kReduceRows * kWave == kThreads, "a wave per row");
        if (__builtin_amdgcn_ballot_w64(odd) == 0) return;
        const uint32_t o_end = min(c0 + blockIdx.y * 256 + 256, cols);
        for (uint32_t o = c0 + blockIdx.y * 256; o < o_end; o += kWave)
            irregular_row<V, kWave, kChunk>(walk, act[threadIdx.x / kWave], m, o, min(o + kWave, o_end), y);
    }
}

// Activation planes from the up GEMM's k-split partial sums (Epi::UpSplit): v = gelu(sum over the splits, in split
// order, of partials[s, m, n] + b_up[n]); rows m >= M hold gelu(b_up[n]), as the zero rows of x give in the fused
// epilogue. Then, per token and 128-neuron block, the binade of the largest |v| and the hi/lo planes, as
// gemm_dma_kernel<Up> writes them. A wave takes 4 rows of one 128-neuron block: 16 lanes per row, 8 consecutive
// neurons per lane (one 16-byte chunk per part); the block's maximum is a 16-lane xor butterfly.
constexpr uint32_t kActRowsPerBlock = kThreads / 16;
template <bool NEAR>  // gelu_near
__global__ __launch_bounds__(kThreads) void act_planes_kernel(const float* __restrict__ partials, uint32_t splits,
                                                             const float* __restrict__ b_up, _Float16* __restrict__ planes,
                                                             int8_t* __restrict__ exps, uint32_t M, uint32_t rows_pad, uint32_t H,
                                                             uint32_t cols) {
    const uint32_t m = blockIdx.x * kActRowsPerBlock + threadIdx.x / 16, sub = threadIdx.x % 16;
    const uint32_t nb = blockIdx.y, n = nb * kActBlock + sub * 8;
    float4 b0 = make_float4(0.f, 0.f, 0.f, 0.f), b1 = b0;
    if (n < cols) {  // a multiple of 8: whole pieces
        b0 = *reinterpret_cast<const float4*>(b_up + n);
        b1 = *reinterpret_cast<const float4*>(b_up + n + 4);
    }
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (m < M) {
        for (uint32_t s0 = 0; s0 < splits; s0 += 4) {  // 8 loads in flight, added in split order
            float4 u[4], w[4];
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q)
                if (s0 + q < splits) {
                    const float* p = partials + (static_cast<size_t>(s0 + q) * M + m) * H + n;
                    u[q] = *reinterpret_cast<const float4*>(p);
                    w[q] = *reinterpret_cast<const float4*>(p + 4);
                }
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q)
                if (s0 + q < splits) {
                    v[0] += u[q].x; v[1] += u[q].y; v[2] += u[q].z; v[3] += u[q].w;
                    v[4] += w[q].x; v[5] += w[q].y; v[6] += w[q].z; v[7] += w[q].w;
                }
        }
    }
    const float b[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
    uint32_t largest = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        v[q] = NEAR ? gelu_near(v[q] + b[q]) : gelu(v[q] + b[q]);
        largest = max(largest, abs_bits(v[q]));
    }
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) largest = max(largest, static_cast<uint32_t>(__shfl_xor(static_cast<int>(largest), off, kWave)));
    const int e = act_binade(largest);
    if (sub == 0) exps[act_exp_at(rows_pad, m, nb)] = static_cast<int8_t>(e);
    const float scale = ldexpf(1.0f, -e);
    half8 hi, lo;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        _Float16 hh, ll;
        split(v[q] * scale, hh, ll);
        hi[q] = hh;
        lo[q] = ll;
    }
    *reinterpret_cast<half8*>(planes + plane_at(rows_pad, m, n, 0)) = hi;
    *reinterpret_cast<half8*>(planes + plane_at(rows_pad, m, n, 1)) = lo;
}

// Training epilogues of the split up-shaped products [tokens, d_ff] (the sums of the split partials, in split order):
//   Forward: z = b_up + sum, act = gelu(z): z and act hidden-major [d_ff, ld], act also as planes with its block
//            binades (read by the down GEMM);
//   GradZ:   gz = sum * gelu'(z), z read hidden-major: gz hidden-major and as planes with block binades (read by the gx
//            GEMM).
// Threads as act_planes_kernel (16 per token, 8 neurons each), 32 tokens x one 128-neuron block. The hidden-major rows go
// through LDS tiles [128 neurons][32 tokens]: thread i takes neuron i / 8 and tokens 4 (i % 8) .. + 3, 16 bytes at a time
// (ld and the block's first token are multiples of 4, so a vector that starts below ld ends below it), a 128-byte line per
// neuron; only tokens below M are written. Bound by memory (4 bytes a split read, 12
// or 16 read or written per entry): MI355X, 2048 tokens x 4096 neurons, Forward / GradZ: 49 / 39 us in blocks of 16 tokens
// (half lines, 4-byte stores), 27.6 / 26.3 us now.
constexpr uint32_t kTrainRows = 32, kTrainThreads = kTrainRows * 16;
enum class TrainPost { Forward, GradZ };
template <TrainPost MODE>
__global__ __launch_bounds__(kTrainThreads) void train_planes_kernel(const float* __restrict__ partials, uint32_t splits,
                                                               const float* __restrict__ b_up, const float* __restrict__ z_in,
                                                               float* __restrict__ out_a, float* __restrict__ out_b,
                                                               _Float16* __restrict__ planes, int8_t* __restrict__ exps, uint32_t M,
                                                               uint32_t rows_pad, uint32_t H, uint32_t ld) {
    constexpr uint32_t R = kTrainRows, kQuads = R / 4;
    static_assert(kActBlock * kQuads % kTrainThreads == 0, "the tile rows divide over the threads");
    __shared__ float ta[kActBlock][R + 1], tb[kActBlock][R + 1];  // Forward: z, act; GradZ: z, gz
    __shared__ float scales[R];
    const uint32_t ml = threadIdx.x / 16, sub = threadIdx.x % 16;
    const uint32_t m0 = blockIdx.x * R, m = m0 + ml;
    const uint32_t nb = blockIdx.y, n0 = nb * kActBlock, n = n0 + sub * 8;
    if constexpr (MODE == TrainPost::GradZ) {
#pragma unroll
        for (uint32_t i = threadIdx.x; i < kActBlock * kQuads; i += kTrainThreads) {
            const uint32_t r = i / kQuads, c = (i % kQuads) * 4;
            float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
            if (m0 + c < ld) q = *reinterpret_cast<const float4*>(z_in + static_cast<size_t>(n0 + r) * ld + m0 + c);
            ta[r][c] = q.x, ta[r][c + 1] = q.y, ta[r][c + 2] = q.z, ta[r][c + 3] = q.w;
        }
        __syncthreads();
    }
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (m < M) {
        for (uint32_t s0 = 0; s0 < splits; s0 += 4) {  // 8 loads in flight, added in split order
            float4 u[4], w[4];
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q)
                if (s0 + q < splits) {
                    const float* p = partials + (static_cast<size_t>(s0 + q) * M + m) * H + n;
                    u[q] = *reinterpret_cast<const float4*>(p);
                    w[q] = *reinterpret_cast<const float4*>(p + 4);
                }
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q)
                if (s0 + q < splits) {
                    v[0] += u[q].x; v[1] += u[q].y; v[2] += u[q].z; v[3] += u[q].w;
                    v[4] += w[q].x; v[5] += w[q].y; v[6] += w[q].z; v[7] += w[q].w;
                }
        }
    }
    uint32_t largest = 0;
    if constexpr (MODE == TrainPost::Forward) {
        const float4 b0 = *reinterpret_cast<const float4*>(b_up + n), b1 = *reinterpret_cast<const float4*>(b_up + n + 4);
        const float b[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float z = v[q] + b[q];
            ta[sub * 8 + q][ml] = z;
            v[q] = gelu(z);
            tb[sub * 8 + q][ml] = v[q];
            largest = max(largest, abs_bits(v[q]));
        }
    } else {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            v[q] *= gelu_grad(ta[sub * 8 + q][ml]);
            tb[sub * 8 + q][ml] = v[q];
            largest = max(largest, abs_bits(v[q]));
        }
    }
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) largest = max(largest, static_cast<uint32_t>(__shfl_xor(static_cast<int>(largest), off, kWave)));
    if (sub == 0) {
        const int e = act_binade(largest);
        exps[act_exp_at(rows_pad, m, nb)] = static_cast<int8_t>(e);
        scales[ml] = ldexpf(1.0f, -e);
    }
    __syncthreads();
    {  // the planes from the tile, token by token: 32 tokens' 16 bytes of a chunk follow one another
        const uint32_t t = threadIdx.x % R, chunk = threadIdx.x / R;
        const float scale = scales[t];
        half8 hi, lo;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            _Float16 hh, ll;
            split(tb[chunk * 8 + q][t] * scale, hh, ll);
            hi[q] = hh;
            lo[q] = ll;
        }
        *reinterpret_cast<half8*>(planes + plane_at(rows_pad, m0 + t, n0 + chunk * 8, 0)) = hi;
        *reinterpret_cast<half8*>(planes + plane_at(rows_pad, m0 + t, n0 + chunk * 8, 1)) = lo;
    }
#pragma unroll
    for (uint32_t i = threadIdx.x; i < kActBlock * kQuads; i += kTrainThreads) {
        const uint32_t r = i / kQuads, c = (i % kQuads) * 4;
        const size_t at = static_cast<size_t>(n0 + r) * ld + m0 + c;
        const auto row = [&](float* __restrict__ to, const float (&from)[R + 1]) {
            if (m0 + c + 4 <= M) {
                *reinterpret_cast<float4*>(to + at) = make_float4(from[c], from[c + 1], from[c + 2], from[c + 3]);
            } else {
#pragma unroll
                for (uint32_t q = 0; q < 3; ++q)
                    if (m0 + c + q < M) to[at + q] = from[c + q];
            }
        };
        if constexpr (MODE == TrainPost::Forward) {
            row(out_a, ta[r]);
            row(out_b, tb[r]);
        } else {
            row(out_a, tb[r]);
        }
    }
}

uint32_t ceil_div(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

struct Shape {
    int mi, ni, splits;  // wave tile (32 mi) x (32 ni), block tile (64 mi) x (64 ni), k splits
};

constexpr int kMaxSplits = 4;

uint32_t rows_padded(uint32_t m) { return ceil_div(m, kRowPad) * kRowPad; }

// Rows of the token and activation planes that a call of m tokens reads: one row tile of at most 64 or 128 tokens
// runs the live-row GEMMs (gemm_dma_kernel<..., 64 or 128>), which read only its first 64 or 128 rows; otherwise every
// padded row. The split and activation-plane passes write these rows only.
uint32_t rows_live(uint32_t m) { return m <= 64 ? 64 : m <= 128 ? 128 : rows_padded(m); }

// Up: 128 x 128 blocks (the column tile is the activation block). Down: 64 x 128 blocks without a k split; K is
// split only when a down projection has fewer than 64 blocks (the fixup's device-scope fences write back the L2).
Shape up_shape(uint32_t, uint32_t) { return {2, 2, 1}; }

Shape down_shape(uint32_t m, uint32_t ncol, uint32_t k) {
    const uint32_t tiles = rows_padded(m) / 64 * (ncol / 128);
    return {1, 2, tiles < 64 && k >= 2048 ? 2 : 1};
}

template <Epi EPI, bool LO_B, int MI, int NI, int SPLITS>
hipError_t launch_gemm(const _Float16* a_planes, const int32_t* a_exp, const _Float16* b_planes, const int32_t* b_exp,
                       const float* bias, float* out, _Float16* out_planes, int32_t* out_exp, float* partials, int32_t* counters,
                       uint32_t M, uint32_t Ncol, uint32_t K, hipStream_t stream) {
    static_assert(EPI == Epi::Down || 64 * NI == kActBlock, "the up GEMM's column tile is the activation block");
    const uint32_t rows_pad = rows_padded(M);
    const uint32_t tiles = rows_pad / (64 * MI) * (Ncol / (64 * NI));
    hipLaunchKernelGGL((gemm_planes_kernel<EPI, MI, NI, LO_B, SPLITS>), dim3(tiles * SPLITS), dim3(kThreads), 0, stream, a_planes,
                       a_exp, b_planes, b_exp, bias, out, out_planes, out_exp, partials, counters, M, rows_pad, Ncol, K);
    return hipGetLastError();
}

// The instantiated shapes: up (mi, ni) in {(2,2), (4,2), (1,2)} without splits; down (2,2) and (1,2) with 1, 2 or 4
// splits and (2,4) with 1 or 2.
template <Epi EPI, bool LO_B>
hipError_t gemm(Shape shape, const _Float16* a_planes, const int32_t* a_exp, const _Float16* b_planes, const int32_t* b_exp,
                const float* bias, float* out, _Float16* out_planes, int32_t* out_exp, float* partials, int32_t* counters,
                uint32_t M, uint32_t Ncol, uint32_t K, hipStream_t stream) {
#define HFFN_GEMM(MI, NI, S)                                                                                                   \
    if (shape.mi == MI && shape.ni == NI && shape.splits == S)                                                                 \
        return launch_gemm<EPI, LO_B, MI, NI, S>(a_planes, a_exp, b_planes, b_exp, bias, out, out_planes, out_exp, partials,   \
                                                 counters, M, Ncol, K, stream);
    if constexpr (EPI == Epi::Up) {
        HFFN_GEMM(2, 2, 1)
        HFFN_GEMM(4, 2, 1)
        HFFN_GEMM(1, 2, 1)
    } else {
        HFFN_GEMM(2, 2, 1)
        HFFN_GEMM(2, 2, 2)
        HFFN_GEMM(2, 2, 4)
        HFFN_GEMM(1, 2, 1)
        HFFN_GEMM(1, 2, 2)
        HFFN_GEMM(1, 2, 4)
        HFFN_GEMM(2, 4, 1)
        HFFN_GEMM(2, 4, 2)
    }
#undef HFFN_GEMM
    return hipErrorInvalidValue;
}

// The streamed kernel takes a GEMM when its 256 x 128 tiles times its k splits give at least kDmaMinBlocks blocks
// (an up projection) or kDmaMinDownBlocks (a down projection, whose split count is bounded by the activation blocks
// of narrow layers); the split partials are added by reduce_splits_kernel (down) or act_planes_kernel (up).
constexpr uint32_t kDmaMinBlocks = 128;
constexpr uint32_t kDmaMinDownBlocks = 64;

uint32_t dma_tiles(uint32_t m, uint32_t ncol) { return rows_padded(m) / kDmaBM * (ncol / kDmaBN); }

// Splits of the streamed down GEMM by estimated time, over the split counts (powers of two up to kDmaMaxSplits) that
// cut K on activation blocks, hold a split's binades in LDS and give at least kDmaMinDownBlocks blocks: the blocks
// run in rounds of one per CU (the LDS ring takes a CU), each block kDmaKtileUs per k-tile plus kDmaBlockUs of
// prologue and epilogue; a split count above 1 adds its partials' round trip (written, then read by
// reduce_splits_kernel) and that kernel's launch. The partials are priced on the padded rows, so every token count
// of one padded row count takes the same splits and a token's sums do not depend on the call's other tokens.
// Constants measured on MI355X (256 x 128 blocks of 8 waves: a k-tile 1.29-1.46 us, prologue + epilogue 7-9 us,
// partials at ~4 TB/s). 0: not streamed.
constexpr uint32_t kDmaMaxSplits = 32;
constexpr uint32_t kCus = 256;
constexpr double kDmaKtileUs = 1.35, kDmaBlockUs = 8.0, kPartialBytesPerUs = 4.0e6, kReduceUs = 4.0;
uint32_t dma_down_splits(uint32_t m, uint32_t ncol, uint32_t k) {
    const uint32_t tiles = dma_tiles(m, ncol), ktiles = k / kBK;
    uint32_t best = 0;
    double best_us = 0.0;
    for (uint32_t splits = 1; splits <= kDmaMaxSplits; splits *= 2) {
        if (k % (kActBlock * splits) != 0 || k / kActBlock / splits > kDmaMaxActBlocks || tiles * splits < kDmaMinDownBlocks)
            continue;
        const double rounds = ceil_div(tiles * splits, kCus);
        double us = rounds * (static_cast<double>(ktiles) / splits * kDmaKtileUs + kDmaBlockUs);
        if (splits > 1) us += 8.0 * splits * rows_padded(m) * ncol / kPartialBytesPerUs + kReduceUs;
        if (best == 0 || us < best_us) best = splits, best_us = us;
    }
    return best;
}

// The streamed down GEMM's plan: `splits` k splits of every column tile (whole_n 0), or, where that is estimated faster,
// the first whole_n column tiles over all of K (one round of long blocks, writing y) and the others in `splits` k
// splits, whose partials cover only their columns. A wide K takes the whole-K tiles only where a tile holds all of its
// activation blocks' binades in LDS (bfloat16 weights leave the ring's B lo plane free for them). Priced as
// dma_down_splits: the split blocks that the CUs without a whole tile finish meanwhile, then whole rounds of the rest.
// MI355X, 2.8B shape at 4096 tokens (16 x 20 tiles, 320 k-tiles): 16 whole column tiles and 4 column tiles in 4 splits
// (256 + 256 blocks) against 4 splits of all 20 (1280 blocks), a fifth of the partials.
struct DownPlan {
    uint32_t splits, whole_n;
};
DownPlan dma_down_plan(uint32_t m, uint32_t ncol, uint32_t k, bool bf16) {
    const uint32_t uniform = dma_down_splits(m, ncol, k);
    DownPlan plan{uniform, 0};
    const uint32_t tiles_m = rows_padded(m) / kDmaBM, tiles_n = ncol / kDmaBN, ktiles = k / kBK;
    const uint32_t max_blocks = bf16 ? kDmaMaxActBlocks + kDmaStages * kDmaLoRuns : kDmaMaxActBlocks;
    if (uniform == 0 || k % kActBlock != 0 || k / kActBlock > max_blocks) return plan;
    const double partial_us = 8.0 * rows_padded(m) / kPartialBytesPerUs;  // per split and column
    double best_us = ceil_div(tiles_m * tiles_n * uniform, kCus) * (static_cast<double>(ktiles) / uniform * kDmaKtileUs + kDmaBlockUs) +
                     (uniform > 1 ? partial_us * uniform * ncol + kReduceUs : 0.0);
    const double whole_us = ktiles * kDmaKtileUs + kDmaBlockUs;
    for (uint32_t whole_n = 1; whole_n < tiles_n && tiles_m * whole_n <= kCus; ++whole_n)
        for (uint32_t splits = 2; splits <= kDmaMaxSplits; splits *= 2) {
            if (k % (kActBlock * splits) != 0 || k / kActBlock / splits > kDmaMaxActBlocks) continue;
            const double split_us = static_cast<double>(ktiles) / splits * kDmaKtileUs + kDmaBlockUs;
            const uint32_t free_cus = kCus - tiles_m * whole_n, pieces = tiles_m * (tiles_n - whole_n) * splits;
            const uint32_t meanwhile = free_cus * static_cast<uint32_t>(whole_us / split_us);
            const double span = pieces <= meanwhile ? max(whole_us, ceil_div(pieces, free_cus) * split_us)
                                                    : whole_us + ceil_div(pieces - meanwhile, kCus) * split_us;
            const double us = span + partial_us * splits * (tiles_n - whole_n) * kDmaBN + kReduceUs;
            if (us < best_us) plan = {splits, whole_n}, best_us = us;
        }
    return plan;
}

// Splits of the streamed up GEMM: 1 when its tiles alone fill the chip, else doubled (up to 8, each split at least
// one k-tile) until ~192 blocks; the partial sums then go through act_planes_kernel. 0: not streamed.
constexpr uint32_t kDmaMaxUpSplits = 8;
uint32_t dma_up_splits(uint32_t m, uint32_t ncol, uint32_t k) {
    const uint32_t tiles = dma_tiles(m, ncol);
    if (tiles >= kDmaMinBlocks) return 1;
    uint32_t splits = 1;
    while (splits < kDmaMaxUpSplits && tiles * splits < 192 && k % (kBK * splits * 2) == 0) splits *= 2;
    return tiles * splits >= kDmaMinBlocks ? splits : 0;
}

// Sampled products of the training backward from a dense product: G[rows, cols] = A[rows, n] B[cols, n]^T by the
// streamed GEMM (Epi::UpSplit partials [splits, rows, cols], powers of two undone), then one wave per owner row o:
// g[q] = sum over the splits (in split order) of G[o, idx[q]] for the row's slots q, and gb[o] = sum_t A[o, t]
// (lanes over the tokens, then the fixed xor butterfly).
__global__ __launch_bounds__(kThreads) void gather_dense_kernel(const float* __restrict__ partials, uint32_t splits,
                                                               const float* __restrict__ a, uint32_t ld, uint32_t n,
                                                               const int32_t* __restrict__ off, const int16_t* __restrict__ idx,
                                                               float* __restrict__ g, float* __restrict__ gb, uint32_t rows,
                                                               uint32_t cols) {
    const uint32_t o = blockIdx.x * (kThreads / kWave) + uniform(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    if (o >= rows) return;
    // (kBatch loads per lane in flight; each lane's sums in the order of its tokens and splits)
    constexpr int kBatch = 16;
    float s = 0.0f;
    const float* arow = a + static_cast<size_t>(o) * ld;
    for (uint32_t t0 = lane; t0 < n; t0 += kBatch * kWave) {
        float v[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) v[j] = t0 + j * kWave < n ? arow[t0 + j * kWave] : 0.0f;
#pragma unroll
        for (int j = 0; j < kBatch; ++j)
            if (t0 + j * kWave < n) s += v[j];
    }
    s = wave_sum(s);
    if (lane == 0) gb[o] = s;
    const size_t plane = static_cast<size_t>(rows) * cols;
    const float* row = partials + static_cast<size_t>(o) * cols;
    const int32_t end = off[o + 1];
    // a batch's loads all issued before the first is used (no branch between them): a slot past the row reads the
    // row's last slot again, and its sum is not written
    for (int32_t q0 = off[o] + static_cast<int32_t>(lane); q0 < end; q0 += kBatch * kWave) {
        uint32_t c[kBatch];
        float v[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) c[j] = static_cast<uint16_t>(idx[min(q0 + j * static_cast<int32_t>(kWave), end - 1)]);
#pragma unroll
        for (int j = 0; j < kBatch; ++j) v[j] = row[c[j]];
        for (uint32_t sp = 1; sp < splits; ++sp) {
            float u[kBatch];
#pragma unroll
            for (int j = 0; j < kBatch; ++j) u[j] = row[sp * plane + c[j]];
#pragma unroll
            for (int j = 0; j < kBatch; ++j) v[j] += u[j];
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j)
            if (q0 + j * static_cast<int32_t>(kWave) < end) g[q0 + j * kWave] = v[j];
    }
}

// One row tile of at most 64 or 128 tokens takes the kernel that transfers and multiplies only those rows.
template <Epi EPI, bool LO_B>
hipError_t launch_dma(const _Float16* a_planes, const int32_t* a_exp, const _Float16* b_planes, const int32_t* b_exp,
                      const float* bias, float* out, _Float16* out_planes, int32_t* out_exp, uint32_t M, uint32_t Ncol, uint32_t K,
                      uint32_t splits, hipStream_t stream, uint32_t whole_n = 0, float* part = nullptr) {
    const uint32_t tiles_m = rows_padded(M) / kDmaBM, tiles_n = Ncol / kDmaBN;
    const dim3 grid(tiles_m * whole_n + tiles_m * (tiles_n - whole_n) * splits), block(64 * kDmaWaves);
    const uint32_t rows_pad = rows_padded(M), live = rows_live(M);
    if (live == 64)
        hipLaunchKernelGGL((gemm_dma_kernel<EPI, LO_B, 64, 0>), grid, block, 0, stream, a_planes, a_exp, b_planes, b_exp, bias, out,
                           out_planes, out_exp, M, rows_pad, Ncol, K, splits, whole_n, part, Ncol, Walk{});
    else if (live == 128)
        hipLaunchKernelGGL((gemm_dma_kernel<EPI, LO_B, 128, 0>), grid, block, 0, stream, a_planes, a_exp, b_planes, b_exp, bias, out,
                           out_planes, out_exp, M, rows_pad, Ncol, K, splits, whole_n, part, Ncol, Walk{});
    else
        hipLaunchKernelGGL((gemm_dma_kernel<EPI, LO_B, kDmaBM, 0>), grid, block, 0, stream, a_planes, a_exp, b_planes, b_exp, bias, out,
                           out_planes, out_exp, M, rows_pad, Ncol, K, splits, whole_n, part, Ncol, Walk{});
    return hipGetLastError();
}

// The chained GEMMs: row tiles of bm (64, 128 or 256) tokens, K split `splits` ways (CHAIN 0: one chain, bm 128; WALK: one
// split).
template <Epi EPI, bool LO_B, int CHAIN, bool WALK = false>
hipError_t launch_chained(uint32_t bm, const _Float16* a_planes, const int32_t* a_exp, const _Float16* b_planes, const int32_t* b_exp,
                          const float* bias, float* out, _Float16* out_planes, int32_t* out_exp, uint32_t M, uint32_t Ncol, uint32_t K,
                          uint32_t splits, uint32_t cols, hipStream_t stream, const Walk& walk = {}) {
    const dim3 grid(ceil_div(M, bm) * (Ncol / kDmaBN) * splits);
    const uint32_t rows_pad = rows_padded(M);
#define HFFN_CHAINED(BM)                                                                                                          \
    hipLaunchKernelGGL((gemm_dma_kernel<EPI, LO_B, BM, CHAIN, BM, WALK>), grid, dim3(64 * kDmaWaves), 0, stream, a_planes, a_exp, b_planes, \
                       b_exp, bias, out, out_planes, out_exp, M, rows_pad, Ncol, K, splits, 0u, static_cast<float*>(nullptr), cols, walk)
    if constexpr (CHAIN == 0) HFFN_CHAINED(128);
    else if (bm == 64) HFFN_CHAINED(64);
    else if (bm == 128) HFFN_CHAINED(128);
    else HFFN_CHAINED(256);
#undef HFFN_CHAINED
    return hipGetLastError();
}

// y = the split partials [splits, M, width] of columns c0 .. c0 + width - 1, added in split order, plus the bias.
template <typename V = void>
hipError_t launch_reduce_splits(const float* partials, const float* bias, float* y, uint32_t M, uint32_t splits, uint32_t width, uint32_t c0,
                                uint32_t cols, hipStream_t stream, const Walk& walk = {}) {
    hipLaunchKernelGGL(reduce_splits_kernel<V>, dim3(ceil_div(M, kReduceRows), ceil_div(width, 256)), dim3(kThreads), 0, stream, partials, bias, y,
                       M, splits, width, c0, cols, walk);
    return hipGetLastError();
}

template <bool LO_B>
hipError_t dma_down(DownPlan plan, const _Float16* a_planes, const int32_t* a_exp, const _Float16* b_planes, const int32_t* b_exp,
                    const float* bias, float* y, float* partials, uint32_t M, uint32_t Ncol, uint32_t K, hipStream_t stream) {
    if (plan.splits == 1)
        return launch_dma<Epi::Down, LO_B>(a_planes, a_exp, b_planes, b_exp, bias, y, nullptr, nullptr, M, Ncol, K, 1, stream);
    const hipError_t status =
        plan.whole_n > 0 ? launch_dma<Epi::Down, LO_B>(a_planes, a_exp, b_planes, b_exp, bias, y, nullptr, nullptr, M, Ncol, K,
                                                       plan.splits, stream, plan.whole_n, partials)
                         : launch_dma<Epi::Down, LO_B>(a_planes, a_exp, b_planes, b_exp, bias, partials, nullptr, nullptr, M, Ncol, K,
                                                       plan.splits, stream);
    if (status != hipSuccess) return status;
    const uint32_t c0 = plan.whole_n * kDmaBN;
    return launch_reduce_splits(partials, bias, y, M, plan.splits, Ncol - c0, c0, Ncol, stream);
}

// Workspace layout (int32 words unless stated; rows = M padded to kRowPad): split counters [down tiles of the
// largest token count, 64 x 64 tiles] | x binades [rows] | activation block binades [rows, d_ff / kActBlock] |
// (256-byte aligned, bytes) x planes [rows * d_model * 2 halves] | activation planes [rows * d_ff * 2 halves] |
// float partials (partial_floats: the largest [splits, M, d_model] or [splits, M, d_ff] of any N up to M). The counters
// come first and are sized for every M and tile shape, so a call at
// any M finds them where the previous call, at any other M, left them (at zero).
struct Workspace {
    size_t counters, x_binades, act_binades, x_planes, act_planes, partials, bytes;
};

// Floats of split partial sums any call of up to m tokens may need (the register-staged down GEMM's kMaxSplits, or
// the streamed GEMMs' splits for every padded row count up to m's): a workspace sized for m serves every smaller n.
size_t partial_floats(uint32_t m, uint32_t d, uint32_t h) {
    size_t most = static_cast<size_t>(kMaxSplits) * m * d;
    for (uint32_t rows = kRowPad; rows <= rows_padded(m); rows += kRowPad) {
        const size_t tokens = min(m, rows);
        most = max(most, static_cast<size_t>(dma_down_splits(rows, d, h)) * tokens * d);
        for (const bool bf16 : {false, true}) {
            const DownPlan plan = dma_down_plan(rows, d, h, bf16);
            most = max(most, static_cast<size_t>(plan.splits) * tokens * (d - plan.whole_n * kDmaBN));
        }
        const uint32_t up = dma_up_splits(rows, h, d);
        if (up > 1) most = max(most, static_cast<size_t>(up) * tokens * h);
    }
    return most;
}

// The training products run the up-shaped GEMMs (the forward's up projection, gz) as split products with partials at
// every split count, one included: their partials need the largest [max(1, splits), M, d_ff] of any N up to M too.
size_t train_partial_floats(uint32_t m, uint32_t d, uint32_t h) {
    size_t most = partial_floats(m, d, h);
    for (uint32_t rows = kRowPad; rows <= rows_padded(m); rows += kRowPad)
        most = max(most, static_cast<size_t>(max(1u, dma_up_splits(rows, h, d))) * min(m, rows) * h);
    return most;
}

Workspace workspace_layout(uint32_t m, uint32_t d, uint32_t h, bool training = false) {
    const size_t rows = rows_padded(m);
    Workspace w{};
    w.counters = 0;
    const size_t counter_words = static_cast<size_t>(ceil_div(kMaxTokens, 64)) * (d / 64);
    // both binade tables start on 256-byte boundaries: the streamed GEMM transfers them into LDS 16 or 4 bytes a lane
    w.x_binades = (w.counters + counter_words + 63) / 64 * 64;
    w.act_binades = (w.x_binades + rows + 63) / 64 * 64;
    const size_t words_end = (w.act_binades + rows * (h / kActBlock) / 4) * 4;  // int8 activation binades
    w.x_planes = (words_end + 255) / 256 * 256;  // bytes from here on
    w.act_planes = w.x_planes + rows * d * 4;
    w.partials = w.act_planes + rows * h * 4;
    w.bytes = w.partials + (training ? train_partial_floats(m, d, h) : partial_floats(m, d, h)) * 4;
    return w;
}

}  // namespace

namespace {
size_t align256(size_t v) { return (v + 255) / 256 * 256; }
}  // namespace

size_t dense_plane_halves(uint32_t rows, uint32_t k) { return static_cast<size_t>(rows) * k * 2; }

bool mfma_shape_supported(uint32_t d, uint32_t h) { return d % 256 == 0 && h % 256 == 0; }

bool mfma_streamed(uint32_t n, uint32_t d, uint32_t h) { return dma_up_splits(n, h, d) != 0 && dma_down_splits(n, d, h) != 0; }

size_t mfma_workspace_bytes(uint32_t n, uint32_t d, uint32_t h) { return workspace_layout(n, d, h).bytes; }

namespace {
bool slots_aligned(const void* idx, const void* val) {
    return reinterpret_cast<uintptr_t>(idx) % 16 == 0 && reinterpret_cast<uintptr_t>(val) % 16 == 0;
}
}  // namespace

hipError_t launch_densify(int vt, const int32_t* off, const int16_t* idx, const void* val, uint32_t rows, uint32_t k,
                          void* planes, int32_t* exps, hipStream_t stream) {
    const dim3 grid(dens_blocks(rows, k, 2)), block(kDensThreads);
    const DensSide side{off, idx, val, nullptr, rows, rows, k, kNoChains, slots_aligned(idx, val), static_cast<_Float16*>(planes), exps};
    if (vt == kBF16) hipLaunchKernelGGL((densify_kernel<uint16_t>), grid, block, 0, stream, side);
    else hipLaunchKernelGGL((densify_kernel<float>), grid, block, 0, stream, side);
    return hipGetLastError();
}

hipError_t launch_mfma_split(const float* x, void* workspace, uint32_t n, uint32_t d, uint32_t h, hipStream_t stream) {
    const Workspace w = workspace_layout(n, d, h);
    int32_t* words = static_cast<int32_t*>(workspace);
    auto* x_planes = reinterpret_cast<_Float16*>(static_cast<char*>(workspace) + w.x_planes);
    hipLaunchKernelGGL(split_rows_kernel, dim3(rows_live(n) / kSplitBlockRows), dim3(kThreads), 0, stream, x, n, rows_padded(n), d, d,
                       d, x_planes, words + w.x_binades);  // 8 rows per block
    return hipGetLastError();
}

hipError_t launch_mfma_up(int vt, const float* x, const void* planes, const int32_t* w_exp, const float* b_up, void* workspace,
                          uint32_t n, uint32_t d, uint32_t h, hipStream_t stream) {
    if (hipError_t status = launch_mfma_split(x, workspace, n, d, h, stream); status != hipSuccess) return status;
    return launch_mfma_up_planes(vt, planes, w_exp, b_up, workspace, n, d, h, stream);
}

hipError_t launch_mfma_up_planes(int vt, const void* planes, const int32_t* w_exp, const float* b_up, void* workspace, uint32_t n,
                                 uint32_t d, uint32_t h, hipStream_t stream) {
    const Workspace w = workspace_layout(n, d, h);
    int32_t* words = static_cast<int32_t*>(workspace);
    char* bytes = static_cast<char*>(workspace);
    auto* x_planes = reinterpret_cast<_Float16*>(bytes + w.x_planes);
    auto* act_planes = reinterpret_cast<_Float16*>(bytes + w.act_planes);
    const auto* p = static_cast<const _Float16*>(planes);
    if (const uint32_t splits = dma_up_splits(n, h, d); splits > 1) {
        float* partials = reinterpret_cast<float*>(bytes + w.partials);
        const hipError_t status =
            vt == kBF16 ? launch_dma<Epi::UpSplit, false>(x_planes, words + w.x_binades, p, w_exp, nullptr, partials, nullptr, nullptr, n,
                                                          h, d, splits, stream)
                        : launch_dma<Epi::UpSplit, true>(x_planes, words + w.x_binades, p, w_exp, nullptr, partials, nullptr, nullptr, n,
                                                         h, d, splits, stream);
        if (status != hipSuccess) return status;
        hipLaunchKernelGGL(act_planes_kernel<false>, dim3(rows_live(n) / kActRowsPerBlock, h / kActBlock), dim3(kThreads), 0, stream, partials,
                           splits, b_up, act_planes, reinterpret_cast<int8_t*>(words + w.act_binades), n, rows_padded(n), h, h);
        return hipGetLastError();
    }
    if (dma_tiles(n, h) >= kDmaMinBlocks) {
        if (vt == kBF16)
            return launch_dma<Epi::Up, false>(x_planes, words + w.x_binades, p, w_exp, b_up, nullptr, act_planes, words + w.act_binades,
                                              n, h, d, 1, stream);
        return launch_dma<Epi::Up, true>(x_planes, words + w.x_binades, p, w_exp, b_up, nullptr, act_planes, words + w.act_binades, n,
                                         h, d, 1, stream);
    }
    const Shape shape = up_shape(n, h);
    if (vt == kBF16)
        return gemm<Epi::Up, false>(shape, x_planes, words + w.x_binades, p, w_exp, b_up, nullptr, act_planes, words + w.act_binades,
                                    nullptr, nullptr, n, h, d, stream);
    return gemm<Epi::Up, true>(shape, x_planes, words + w.x_binades, p, w_exp, b_up, nullptr, act_planes, words + w.act_binades,
                               nullptr, nullptr, n, h, d, stream);
}

hipError_t launch_mfma_down(int vt, const void* planes, const int32_t* v_exp, const float* b_down, float* y, void* workspace,
                            uint32_t n, uint32_t d, uint32_t h, hipStream_t stream) {
    const Workspace w = workspace_layout(n, d, h);
    int32_t* words = static_cast<int32_t*>(workspace);
    char* bytes = static_cast<char*>(workspace);
    const auto* act_planes = reinterpret_cast<const _Float16*>(bytes + w.act_planes);
    float* partials = reinterpret_cast<float*>(bytes + w.partials);
    const auto* p = static_cast<const _Float16*>(planes);
    if (const DownPlan plan = dma_down_plan(n, d, h, vt == kBF16); plan.splits != 0) {
        if (vt == kBF16)
            return dma_down<false>(plan, act_planes, words + w.act_binades, p, v_exp, b_down, y, partials, n, d, h, stream);
        return dma_down<true>(plan, act_planes, words + w.act_binades, p, v_exp, b_down, y, partials, n, d, h, stream);
    }
    const Shape shape = down_shape(n, d, h);
    if (vt == kBF16)
        return gemm<Epi::Down, false>(shape, act_planes, words + w.act_binades, p, v_exp, b_down, y, nullptr, nullptr, partials,
                                      words + w.counters, n, d, h, stream);
    return gemm<Epi::Down, true>(shape, act_planes, words + w.act_binades, p, v_exp, b_down, y, nullptr, nullptr, partials,
                                 words + w.counters, n, d, h, stream);
}

// ------------------------------------------------------------------------------ planes densified per call
// A call above the decode sizes on a layer without planes of its own: the planes of both sides are densified from the
// compact rows into the call's workspace (one launch, with the split of x), then the streamed GEMMs run on them as on a
// layer's own. Widths are padded to multiples of 256 (zero rows and columns; biases and y end at the real ones). The
// GEMMs run in chains of one activation block, the float32 up projection in half of one: its three MFMAs per step make
// chains of 128 k as long as the sums over them (error against 64 bits, 1024 x 4096 shape at 2048 tokens: 2.48e-7 ->
// 2.38e-7; the bfloat16 1.4B shape the other way, 2.16e-7 -> 2.23e-7). Calls above kPrefillPiece tokens run in pieces over the
// same planes, which bounds the workspace.
constexpr uint32_t kPrefillPiece = 16384;
constexpr int kPrefillDownChain = kKtPerActBlock, kUpChainF32 = kKtPerActBlock / 2, kUpChainBf16 = kKtPerActBlock;
constexpr uint32_t kPrefillDownBlocks = 16;  // activation blocks of a down split: longer sums lose more than the tiles path
constexpr uint32_t pad256(uint32_t v) { return (v + 255) / 256 * 256; }

// Row tile and k splits by estimated time: the blocks run in rounds of one per CU, each ktile_us per k-tile plus its
// prologue and epilogue; a count above 1 adds its partials' round trip and a launch. `unit`: k-tiles a split may not
// cut (1: the up projection). Constants measured on MI355X at 8-64 k-tiles and 40-2048 blocks.
struct ChainTile {
    uint32_t bm;
    double ktile_us[2], up_us, down_us;  // a k-tile with float32, bfloat16 weights; prologue and epilogue
};
constexpr ChainTile kChainTiles[] = {{64, {0.45, 0.36}, 6.4, 4.5}, {128, {0.66, 0.56}, 8.5, 6.0}, {256, {1.36, 0.97}, 9.0, 8.0}};
constexpr uint32_t kPrefillMaxSplits = 24;
struct ChainPlan {
    uint32_t bm, splits;
};
ChainPlan chain_plan(uint32_t m, uint32_t ncol, uint32_t k, bool bf16, uint32_t unit, uint32_t min_splits) {
    const uint32_t units = k / kBK / unit;
    ChainPlan best{0, 0};
    double best_us = 0.0;
    for (const ChainTile& tile : kChainTiles)
        for (uint32_t splits = min_splits; splits <= min(units, kPrefillMaxSplits); ++splits) {
            const uint32_t rounds = ceil_div(ceil_div(m, tile.bm) * (ncol / kDmaBN) * splits, kCus);
            double us = rounds * (ceil_div(units, splits) * unit * tile.ktile_us[bf16] + (unit == 1 ? tile.up_us : tile.down_us));
            if (splits > 1) us += 8.0 * splits * m * ncol / kPartialBytesPerUs + kReduceUs;
            if (best.bm == 0 || us < best_us) best = {tile.bm, splits}, best_us = us;
        }
    return best;
}
struct PrefillPlan {
    ChainPlan up, down;
};
// m: the real tokens; planned for the end of their block of kRowPad (128 below it), so that a workspace sized for n
// serves every smaller call
uint32_t prefill_class(uint32_t m) { return m <= 128 ? 128 : rows_padded(m); }
PrefillPlan prefill_plan(uint32_t m, uint32_t d, uint32_t h, bool bf16) {
    static_assert(kPrefillDownBlocks <= kDmaMaxActBlocks, "a split's binades fit LDS");
    const uint32_t rows = prefill_class(m);
    return {chain_plan(rows, h, d, bf16, 1, 1), chain_plan(rows, d, h, bf16, kKtPerActBlock, ceil_div(h / kActBlock, kPrefillDownBlocks))};
}

struct PrefillLayout {
    uint32_t d, h;  // padded widths
    size_t up_planes, up_exp, down_planes, down_exp, x_exp, act_exp, x_planes, act_planes, partials, bytes;
};
// Byte offsets (256-byte aligned) for calls of up to n tokens; the partials hold the largest of any smaller call's.
PrefillLayout plan_layout(bool bf16, uint32_t n, uint32_t d, uint32_t h) {
    PrefillLayout l{};
    l.d = pad256(d);
    l.h = pad256(h);
    n = min(n, kPrefillPiece);
    const size_t rows = rows_padded(n);
    size_t at = 0;
    const auto take = [&at](size_t bytes) {
        const size_t from = at;
        at = align256(at + bytes);
        return from;
    };
    l.up_planes = take(dense_plane_halves(l.h, l.d) * 2);
    l.up_exp = take(static_cast<size_t>(l.h) * 4);
    l.down_planes = take(dense_plane_halves(l.d, l.h) * 2);
    l.down_exp = take(static_cast<size_t>(l.d) * 4);
    l.x_exp = take(rows * 4);
    l.act_exp = take(rows * (l.h / kActBlock));
    l.x_planes = take(dense_plane_halves(rows, l.d) * 2);
    l.act_planes = take(dense_plane_halves(rows, l.h) * 2);
    size_t most = 0;
    for (uint32_t m = 128; m <= max(rows, size_t{128}); m += m == 128 ? 128 : kRowPad) {
        const PrefillPlan plan = prefill_plan(m, l.d, l.h, bf16);
        if (plan.up.splits > 1) most = max(most, static_cast<size_t>(plan.up.splits) * min(m, n) * l.h);
        if (plan.down.splits > 1) most = max(most, static_cast<size_t>(plan.down.splits) * min(m, n) * l.d);
    }
    l.partials = take(most * 4);
    l.bytes = at;
    return l;
}

// The last layouts of the thread by their arguments (each plans every row count up to n: ~10 us of host time at 2048).
PrefillLayout prefill_layout(bool bf16, uint32_t n, uint32_t d, uint32_t h) {
    struct Entry {
        bool bf16;
        uint32_t n, d, h;
        PrefillLayout layout;
    };
    thread_local Entry entries[8] = {};
    thread_local uint32_t next = 0;
    for (const Entry& e : entries)
        if (e.n == n && e.d == d && e.h == h && e.bf16 == bf16) return e.layout;
    Entry& e = entries[next++ % 8];
    e = {bf16, n, d, h, plan_layout(bf16, n, d, h)};
    return e.layout;
}

uint64_t prefill_workspace_bytes(int vt, uint32_t n, uint32_t d, uint32_t h) { return prefill_layout(vt == kBF16, n, d, h).bytes; }

namespace {
__global__ __launch_bounds__(kThreads) void copy_kernel(const float4* __restrict__ from, float4* __restrict__ to, uint32_t quads) {
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    if (i < quads) to[i] = from[i];
}
template <typename V>
hipError_t prefill(const PrefillCall& c, hipStream_t stream) {
    constexpr bool kLoB = sizeof(V) == 4;
    constexpr uint32_t kParts = kLoB ? 2 : 1;
    constexpr int kUpChain = kLoB ? kUpChainF32 : kUpChainBf16;
    const PrefillLayout l = prefill_layout(!kLoB, c.n, c.d, c.h);
    char* w = static_cast<char*>(c.workspace);
    const auto halves = [&](size_t at) { return reinterpret_cast<_Float16*>(w + at); };
    const auto words = [&](size_t at) { return reinterpret_cast<int32_t*>(w + at); };
    float* partials = reinterpret_cast<float*>(w + l.partials);
    const DensSide up{c.up_off, c.up_idx, c.up_val, nullptr, c.h, l.h, l.d, chain_bits(kUpChain), slots_aligned(c.up_idx, c.up_val), halves(l.up_planes), words(l.up_exp)};
    const DensSide down{c.down_off, c.down_idx, c.down_val, nullptr, c.d, l.d, l.h, chain_bits(kPrefillDownChain), slots_aligned(c.down_idx, c.down_val), halves(l.down_planes), words(l.down_exp)};
    for (uint32_t t0 = 0; t0 < c.n; t0 += kPrefillPiece) {
        const uint32_t n = min(kPrefillPiece, c.n - t0), rows = rows_padded(n), split_blocks = rows_live(n) / kSplitBlockRows / kSplitGroups;
        const uint32_t up_blocks = t0 == 0 ? dens_blocks(l.h, l.d, kParts) : 0, down_blocks = t0 == 0 ? dens_blocks(l.d, l.h, kParts) : 0;
        const float* x = c.x + static_cast<size_t>(t0) * c.d;
        float* y = c.y + static_cast<size_t>(t0) * c.d;
        hipLaunchKernelGGL(prefill_prep_kernel<V>, dim3(up_blocks + down_blocks + split_blocks), dim3(kDensThreads), 0, stream, up, down,
                           up_blocks, split_blocks, 0u, x, n, rows, l.d, c.d, halves(l.x_planes), words(l.x_exp),
                           static_cast<float*>(nullptr), 0u, 1u, false);
        if (hipError_t status = hipGetLastError(); status != hipSuccess) return status;
        const PrefillPlan plan = prefill_plan(n, l.d, l.h, !kLoB);
        const bool split = plan.up.splits > 1;
        hipError_t status =
            split ? launch_chained<Epi::UpSplit, kLoB, kUpChain>(plan.up.bm, halves(l.x_planes), words(l.x_exp), up.planes, up.exps, nullptr,
                                                                 partials, nullptr, nullptr, n, l.h, l.d, plan.up.splits, l.h, stream)
                  : launch_chained<Epi::Up, kLoB, kUpChain>(plan.up.bm, halves(l.x_planes), words(l.x_exp), up.planes, up.exps, c.b_up,
                                                            nullptr, halves(l.act_planes), words(l.act_exp), n, l.h, l.d, 1, c.h, stream);
        if (status != hipSuccess) return status;
        if (split) {
            hipLaunchKernelGGL(act_planes_kernel<true>, dim3(rows_live(n) / kActRowsPerBlock, l.h / kActBlock), dim3(kThreads), 0, stream,
                               partials, plan.up.splits, c.b_up, halves(l.act_planes), reinterpret_cast<int8_t*>(w + l.act_exp), n, rows,
                               l.h, c.h);
            if (status = hipGetLastError(); status != hipSuccess) return status;
        }
        // x may be the memory of y (a call on the output of the one before): the walk reads it after y is written, so it is
        // kept where x's planes were, which nothing reads any more
        const float* kept = x;
        const uintptr_t x0 = reinterpret_cast<uintptr_t>(x), y0 = reinterpret_cast<uintptr_t>(y), size = static_cast<uintptr_t>(n) * c.d * 4;
        if (x0 < y0 + size && y0 < x0 + size) {
            float4* copy = reinterpret_cast<float4*>(w + l.x_planes);
            const uint32_t quads = static_cast<uint32_t>(size / 16);
            hipLaunchKernelGGL(copy_kernel, dim3(ceil_div(quads, kThreads)), dim3(kThreads), 0, stream, reinterpret_cast<const float4*>(x), copy, quads);
            if (status = hipGetLastError(); status != hipSuccess) return status;
            kept = reinterpret_cast<const float*>(copy);
        }
        const Walk walk{kept, c.up_off, c.up_idx, c.up_val, c.b_up, c.down_off, c.down_idx, c.down_val, c.b_down, c.d, c.h};
        const auto down_gemm = [&](auto walks, float* out) {
            return launch_chained<Epi::Down, kLoB, kPrefillDownChain, decltype(walks)::value>(
                plan.down.bm, halves(l.act_planes), words(l.act_exp), down.planes, down.exps, c.b_down, out, nullptr, nullptr, n, l.d, l.h,
                plan.down.splits, c.d, stream, walk);
        };
        if (plan.down.splits == 1) {
            status = down_gemm(std::true_type{}, y);
        } else {
            status = down_gemm(std::false_type{}, partials);
            if (status == hipSuccess)
                status = launch_reduce_splits<V>(partials, c.b_down, y, n, plan.down.splits, l.d, 0, c.d, stream, walk);
        }
        if (status != hipSuccess) return status;
    }
    return hipSuccess;
}
}  // namespace

hipError_t launch_prefill(int vt, const PrefillCall& call, hipStream_t stream) {
    return vt == kBF16 ? prefill<uint16_t>(call, stream) : prefill<float>(call, stream);
}

// Workspace of the dense sampled product (bytes, 256-aligned parts): the planes of A [rows, k_pad] and B [cols,
// k_pad] (tokens padded to a multiple of 256, split_rows' k granularity), their row binades and the GEMM's partials.
namespace {
struct GradDenseLayout {
    size_t a_planes, b_planes, a_exp, b_exp, partials, bytes;
    uint32_t k_pad, splits;
};
GradDenseLayout grad_dense_layout(uint32_t rows, uint32_t cols, uint32_t n) {
    GradDenseLayout l{};
    l.k_pad = ceil_div(n, 256) * 256;
    l.splits = dma_up_splits(rows, cols, l.k_pad);
    l.a_planes = 0;
    l.b_planes = align256(l.a_planes + dense_plane_halves(rows, l.k_pad) * 2);
    l.a_exp = align256(l.b_planes + dense_plane_halves(cols, l.k_pad) * 2);
    l.b_exp = align256(l.a_exp + static_cast<size_t>(rows) * 4);
    l.partials = align256(l.b_exp + static_cast<size_t>(cols) * 4);
    l.bytes = l.partials + static_cast<size_t>(l.splits) * rows * cols * 4;
    return l;
}
}  // namespace

size_t grad_dense_workspace_bytes(uint32_t rows, uint32_t cols, uint32_t n) {
    if (rows % kRowPad != 0 || cols % kDmaBN != 0) return 0;
    const GradDenseLayout l = grad_dense_layout(rows, cols, n);
    return l.splits == 0 ? 0 : l.bytes;
}

hipError_t launch_grad_dense(const float* row, const float* mat, const int32_t* off, const int16_t* idx, float* g, float* gb,
                             uint32_t rows, uint32_t cols, uint32_t n, uint32_t ld, void* workspace, bool narrow, hipStream_t stream) {
    const GradDenseLayout l = grad_dense_layout(rows, cols, n);
    char* w = static_cast<char*>(workspace);
    auto* a_planes = reinterpret_cast<_Float16*>(w + l.a_planes);
    auto* b_planes = reinterpret_cast<_Float16*>(w + l.b_planes);
    auto* a_exp = reinterpret_cast<int32_t*>(w + l.a_exp);
    auto* b_exp = reinterpret_cast<int32_t*>(w + l.b_exp);
    auto* partials = reinterpret_cast<float*>(w + l.partials);
    hipLaunchKernelGGL(split_pair_kernel, dim3((rows + cols) / kSplitBlockRows), dim3(kThreads), 0, stream, row, rows, a_planes, a_exp, mat, cols,
                       b_planes, b_exp, l.k_pad, ld, n);
    if (hipError_t status = hipGetLastError(); status != hipSuccess) return status;
    // narrow, in steps whose other products run on planes: row tiles of 128 where 256 leave CUs idle (an output's products and
    // their order are the same): 1024 x 4096 at 512 tokens, 128 blocks -> 256, 23.3 -> 18.3 us, a step at 50 % 275 -> 266 us; at
    // 2048 tokens 64.5 -> 50.5 us, the step 556 -> 529. Not beside the lane-per-token gathers: matrix units busy on all 256 CUs
    // take a card at its power limit to a lower clock, at which the gathers, most of such a step, take 136 us in place of 128:
    // steps at 10 % 725 -> 751 us (2048 tokens), 227 -> 231 (512), at 30 % 458 -> 483 (512); on a card below its limit 722 -> 695.
    narrow = narrow && dma_tiles(rows, cols) * l.splits <= kCus / 2;
    if (hipError_t status = narrow ? launch_chained<Epi::UpSplit, true, 0>(128, a_planes, a_exp, b_planes, b_exp, nullptr, partials, nullptr,
                                                                           nullptr, rows, cols, l.k_pad, l.splits, cols, stream)
                                   : launch_dma<Epi::UpSplit, true>(a_planes, a_exp, b_planes, b_exp, nullptr, partials, nullptr, nullptr,
                                                                    rows, cols, l.k_pad, l.splits, stream);
        status != hipSuccess)
        return status;
    hipLaunchKernelGGL(gather_dense_kernel, dim3(ceil_div(rows, kThreads / kWave)), dim3(kThreads), 0, stream, partials, l.splits, row,
                       ld, n, off, idx, g, gb, rows, cols);
    return hipGetLastError();
}

size_t train_mfma_workspace_bytes(uint32_t n, uint32_t d, uint32_t h) { return workspace_layout(n, d, h, true).bytes; }

namespace {
// x [n, d] split into planes and transposed, and the two sides densified (up_blocks, down_blocks; 0: neither).
hipError_t launch_train_prep(const DensSide& up, const DensSide& down, uint32_t up_blocks, uint32_t down_blocks, const float* x, float* x_t,
                             uint32_t n, uint32_t d, uint32_t ld, _Float16* x_planes, int32_t* x_exp, hipStream_t stream) {
    const uint32_t split_blocks = rows_live(n) / kSplitBlockRows / kSplitGroups, tiles_c = d / kTransCols;
    const uint32_t trans_blocks = ceil_div(tiles_c * ceil_div(n, kTransRows), kSplitGroups);
    hipLaunchKernelGGL(prefill_prep_kernel<float>, dim3(up_blocks + down_blocks + split_blocks + trans_blocks), dim3(kDensThreads), 0, stream, up,
                       down, up_blocks, split_blocks, trans_blocks, x, n, rows_padded(n), d, d, x_planes, x_exp, x_t, ld, tiles_c,
                       transpose_vectors(x, x_t, d, ld));
    return hipGetLastError();
}
}  // namespace

// Training forward on the planes (fp32 weights): x split into planes, the up projection as a split product (partials
// at every split count) whose epilogue (train_planes_kernel<Forward>) writes z, act (hidden-major) and the activation
// planes, then the inference down GEMM: y. x_t = x transposed for the sampled product of g_up. The workspace is laid
// out as the MFMA workspace with the training partials (train_mfma_workspace_bytes).
hipError_t launch_train_forward(const float* x, const void* up_planes, const int32_t* up_exp, const float* b_up, const void* down_planes,
                                const int32_t* down_exp, const float* b_down, void* workspace, float* x_t, float* act, float* z, float* y,
                                uint32_t n, uint32_t d, uint32_t h, uint32_t ld, hipStream_t stream, const TrainSlots* slots) {
    const Workspace w = workspace_layout(n, d, h, true);
    int32_t* words = static_cast<int32_t*>(workspace);
    char* bytes = static_cast<char*>(workspace);
    auto* x_planes = reinterpret_cast<_Float16*>(bytes + w.x_planes);
    auto* act_planes = reinterpret_cast<_Float16*>(bytes + w.act_planes);
    float* partials = reinterpret_cast<float*>(bytes + w.partials);
    // x split and transposed, and (slots) the planes densified from the values again: one launch
    const auto planes = [](const void* p) { return static_cast<_Float16*>(const_cast<void*>(p)); };
    DensSide up{}, down{};
    if (slots != nullptr) {
        up = {slots->up_off, slots->up_idx, slots->up_val, nullptr, h, h, d, kNoChains, slots_aligned(slots->up_idx, slots->up_val),
              planes(up_planes), const_cast<int32_t*>(up_exp)};
        down = {slots->down_off, slots->down_idx, slots->down_val, nullptr, d, d, h, kNoChains, slots_aligned(slots->down_idx, slots->down_val),
                planes(down_planes), const_cast<int32_t*>(down_exp)};
    }
    const uint32_t up_blocks = slots ? dens_blocks(h, d, 2) : 0, down_blocks = slots ? dens_blocks(d, h, 2) : 0;
    if (hipError_t status = launch_train_prep(up, down, up_blocks, down_blocks, x, x_t, n, d, ld, x_planes, words + w.x_binades, stream);
        status != hipSuccess)
        return status;
    const uint32_t splits = max(1u, dma_up_splits(n, h, d));
    if (hipError_t status = launch_dma<Epi::UpSplit, true>(x_planes, words + w.x_binades, static_cast<const _Float16*>(up_planes), up_exp,
                                                           nullptr, partials, nullptr, nullptr, n, h, d, splits, stream);
        status != hipSuccess)
        return status;
    hipLaunchKernelGGL(train_planes_kernel<TrainPost::Forward>, dim3(rows_live(n) / kTrainRows, h / kActBlock), dim3(kTrainThreads), 0,
                       stream, partials, splits, b_up, nullptr, z, act, act_planes, reinterpret_cast<int8_t*>(words + w.act_binades), n,
                       rows_padded(n), h, ld);
    if (hipError_t status = hipGetLastError(); status != hipSuccess) return status;
    return launch_mfma_down(kF32, down_planes, down_exp, b_down, y, workspace, n, d, h, stream);
}

// Training backward products on the planes: gy split into planes; gz = (gy W_down) * gelu'(z) as a split product over
// the planes of W_down^T [d_ff rows, d_model k] whose epilogue (train_planes_kernel<GradZ>) writes gz hidden-major and
// as planes; gx = gz W_up by the down GEMM over the planes of W_up^T [d_model rows, d_ff k], without bias.
hipError_t launch_train_backward(const float* gy, const float* z, const void* down_t_planes, const int32_t* down_t_exp,
                                 const void* up_t_planes, const int32_t* up_t_exp, void* workspace, float* gz, float* gx, uint32_t n,
                                 uint32_t d, uint32_t h, uint32_t ld, hipStream_t stream) {
    const Workspace w = workspace_layout(n, d, h, true);
    int32_t* words = static_cast<int32_t*>(workspace);
    char* bytes = static_cast<char*>(workspace);
    auto* gy_planes = reinterpret_cast<_Float16*>(bytes + w.x_planes);
    auto* gz_planes = reinterpret_cast<_Float16*>(bytes + w.act_planes);
    float* partials = reinterpret_cast<float*>(bytes + w.partials);
    hipLaunchKernelGGL(split_rows_kernel, dim3(rows_live(n) / kSplitBlockRows), dim3(kThreads), 0, stream, gy, n, rows_padded(n), d, d,
                       d, gy_planes, words + w.x_binades);
    if (hipError_t status = hipGetLastError(); status != hipSuccess) return status;
    const uint32_t splits = max(1u, dma_up_splits(n, h, d));
    if (hipError_t status = launch_dma<Epi::UpSplit, true>(gy_planes, words + w.x_binades, static_cast<const _Float16*>(down_t_planes),
                                                           down_t_exp, nullptr, partials, nullptr, nullptr, n, h, d, splits, stream);
        status != hipSuccess)
        return status;
    hipLaunchKernelGGL(train_planes_kernel<TrainPost::GradZ>, dim3(rows_live(n) / kTrainRows, h / kActBlock), dim3(kTrainThreads), 0,
                       stream, partials, splits, nullptr, z, gz, nullptr, gz_planes, reinterpret_cast<int8_t*>(words + w.act_binades), n,
                       rows_padded(n), h, ld);
    if (hipError_t status = hipGetLastError(); status != hipSuccess) return status;
    return launch_mfma_down(kF32, up_t_planes, up_t_exp, nullptr, gx, workspace, n, d, h, stream);
}

// The training backward with its planes densified per call into the workspace (train_planes_workspace_bytes): W_down^T and
// W_up^T from the transposed supports (values read by position), gy split and transposed, all in one launch, then the
// products of launch_train_backward with the same splits: the same bits.
namespace {
struct TrainPlanes {
    size_t up_planes, up_exp, down_planes, down_exp, x_exp, act_exp, x_planes, act_planes, partials, bytes;
};
TrainPlanes train_planes_layout(uint32_t n, uint32_t d, uint32_t h) {
    TrainPlanes l{};
    const size_t rows = rows_padded(n);
    size_t at = 0;
    const auto take = [&at](size_t bytes) {
        const size_t from = at;
        at = align256(at + bytes);
        return from;
    };
    l.up_planes = take(dense_plane_halves(h, d) * 2);
    l.up_exp = take(static_cast<size_t>(h) * 4);
    l.down_planes = take(dense_plane_halves(d, h) * 2);
    l.down_exp = take(static_cast<size_t>(d) * 4);
    l.x_exp = take(rows * 4);
    l.act_exp = take(rows * (h / kActBlock));
    l.x_planes = take(dense_plane_halves(rows, d) * 2);
    l.act_planes = take(dense_plane_halves(rows, h) * 2);
    l.partials = at;  // the last: no other offset depends on n's splits
    l.bytes = at + train_partial_floats(n, d, h) * 4;
    return l;
}
// Whether densifying reads a side's values by position as it goes, or from a copy gathered first: a block of each column
// chunk reads its rows' slots, twice where a wave does not hold them, and a gathered 4-byte read costs a cache line. 1024 x
// 4096: up_t at 50 % (rows of 2048 slots, 8.4 M reads) 68 us in place, 14.6 + 12 us gathered first.
bool gathers_in_place(const DensSide& side, uint32_t nnz) {
    const uint32_t reads = ceil_div(side.k, dens_chunk(2)) * (nnz / side.rows > 512 ? 2 : 1);
    return reads == 1 || static_cast<uint64_t>(reads) * nnz <= 1u << 20;
}
}  // namespace

uint64_t train_planes_workspace_bytes(uint32_t n, uint32_t d, uint32_t h) { return train_planes_layout(n, d, h).bytes; }

hipError_t launch_train_planes_backward(const TrainBackward& c, hipStream_t stream) {
    const TrainPlanes l = train_planes_layout(c.n, c.d, c.h);
    char* w = static_cast<char*>(c.workspace);
    const auto halves = [&](size_t at) { return reinterpret_cast<_Float16*>(w + at); };
    const auto words = [&](size_t at) { return reinterpret_cast<int32_t*>(w + at); };
    DensSide down_t{c.hid_off, c.hid_output, nullptr, nullptr, c.h, c.h, c.d, kNoChains, true, halves(l.up_planes), words(l.up_exp)};
    DensSide up_t{c.in_off, c.in_hidden, nullptr, nullptr, c.d, c.d, c.h, kNoChains, true, halves(l.down_planes), words(l.down_exp)};
    const auto values = [&](DensSide& side, const int32_t* pos, const float* val, float* gathered, uint32_t nnz) {
        const bool in_place = gathers_in_place(side, nnz);
        side.val = in_place ? val : gathered;
        side.pos = in_place ? pos : nullptr;
        side.vec = slots_aligned(side.idx, in_place ? static_cast<const void*>(pos) : gathered);
        return in_place ? hipSuccess : launch_gather_values(val, pos, gathered, nnz, stream);
    };
    if (hipError_t status = values(down_t, c.hid_pos, c.out_val, c.hid_val, c.nnz_down); status != hipSuccess) return status;
    if (hipError_t status = values(up_t, c.in_pos, c.up_val, c.in_val, c.nnz_up); status != hipSuccess) return status;
    if (hipError_t status = launch_train_prep(down_t, up_t, dens_blocks(c.h, c.d, 2), dens_blocks(c.d, c.h, 2), c.gy, c.gy_t, c.n, c.d, c.ld,
                                              halves(l.x_planes), words(l.x_exp), stream);
        status != hipSuccess)
        return status;
    const uint32_t rows = rows_padded(c.n);
    float* partials = reinterpret_cast<float*>(w + l.partials);
    const uint32_t splits = max(1u, dma_up_splits(c.n, c.h, c.d));
    if (hipError_t status = launch_dma<Epi::UpSplit, true>(halves(l.x_planes), words(l.x_exp), down_t.planes, down_t.exps, nullptr, partials,
                                                           nullptr, nullptr, c.n, c.h, c.d, splits, stream);
        status != hipSuccess)
        return status;
    hipLaunchKernelGGL(train_planes_kernel<TrainPost::GradZ>, dim3(rows_live(c.n) / kTrainRows, c.h / kActBlock), dim3(kTrainThreads), 0, stream,
                       partials, splits, nullptr, c.z, c.gz, nullptr, halves(l.act_planes), reinterpret_cast<int8_t*>(w + l.act_exp), c.n, rows,
                       c.h, c.ld);
    if (hipError_t status = hipGetLastError(); status != hipSuccess) return status;
    return dma_down<true>(dma_down_plan(c.n, c.d, c.h, false), halves(l.act_planes), words(l.act_exp), up_t.planes, up_t.exps, nullptr, c.gx,
                          partials, c.n, c.d, c.h, stream);
}

}  // namespace hffn
