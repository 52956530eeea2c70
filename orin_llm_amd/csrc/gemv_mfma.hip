// Matrix-vector products over quantised weight rows (Q4_K, Q5_K, Q6_K, Q8_0) on the matrix cores of gfx950
// (MI355X).
//
// The vector-ALU kernel of gemv.hip spends about three instructions per weight (byte to float,
// multiply-add, unpacking) and is bound by them at twice the time HBM needs for the bytes.  Here
// the multiply-adds run as integer matrix instructions and the vector ALU only assembles the
// weights' bytes and applies the blocks' scales:
//
//   * The activation is cut, per sub-block of the weight format (16 elements for Q6_K, 32 for
//     the others), into three signed 8-bit digits of a 24-bit integer, x = s (65536 d0 + 256 d1 + d2)
//     with s = max|x| / (2^23 - 2^16): what the reference does with one digit (quantize_q8_1_k,
//     reference: src/kernels.cu:136-157), carried to the precision of an fp32 mantissa.  Every
//     workgroup builds the digits once, in LDS (together with the RMS norm, when that is folded
//     in), with the sub-blocks' scales and sums beside them.
//   * v_mfma_i32_16x16x64_i8 then multiplies 16 weight rows by 64 elements at a time: the weights,
//     widened to bytes, are the B operand (lane (n, g) holds 16 elements of row n), and the A
//     operand's rows are (sub-block, digit) pairs, each row zero outside its own sub-block.  An
//     accumulator therefore holds, for a row of weights, the exact integer sums of four sub-blocks
//     against the three digits, already separated: lane (n, g) receives the three sums of
//     sub-block g.  They are recombined in fp32 and multiplied by the sub-block's scales:
//     d * scale * sum - dmin * min * sum(x) for Q4_K and Q5_K, d * scale * (sum - 32 sum(x)) for Q6_K,
//     d * sum for Q8_0 (reference CPU statements: src/model_cpu.cpp:70-152).
//   * Loads are made with four neighbouring lanes on 64 consecutive bytes of a row (lane = 4 * row +
//     piece: the vector cache then sees 16 runs per instruction; with the matrix instruction's own
//     lane order, lane = row + 16 * piece, it sees 64 separate 16-byte requests and the kernel runs
//     10 % slower) and moved to the matrix instruction's lanes by one lane permutation per register.
//   * The four waves of a workgroup take every fourth 256-element block of the same 16 rows and meet
//     in LDS at the end; blocks are requested one iteration ahead, across row tiles.
//   * Matrices made of whole 16-row tiles -- every matrix of a model -- take a second kernel with the same
//     arithmetic and another way to the bytes (gemv_rows_kernel, further down): rows read in lane-linear
//     runs with streaming loads and laid out for the matrix instruction through a wave's own LDS buffer,
//     which this machine's memory path serves a quarter faster.  The kernel described above remains for
//     matrices with a ragged last tile, for Q8_0 matrices that do not start on a 16-byte boundary, and for
//     rows whose digits and buffers do not fit LDS together.
#include "gemv_blocks.hpp"

// Stage marks of the kernel that reads rows in long runs: wall-clock stamps in the timeline build (waves 0-3 of a
// workgroup), nothing otherwise (fa_common.hpp).  ROWS_ITEM_STAMP marks an item's arrival in LDS and waits for the
// LDS writes first, in that build only.
#ifdef ORIN_FA_STAMPS
namespace orin_fa {
__device__ long long g_gemv_stamps[kStampWgs * 4 * kStampSlots];
}
// (its own store, all conditions in one test: wrapped around the attention kernels' macro the marks cost this kernel a
// quarter of its time)
#define ROWS_STAMP(i)                                                                                                      \
    do {                                                                                                                   \
        __builtin_amdgcn_sched_barrier(0);                                                                                 \
        const unsigned wg_ = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);                               \
        if ((threadIdx.x & 63) == 0 && threadIdx.x < 256 && wg_ < (unsigned)orin_fa::kStampWgs && (i) < orin_fa::kStampSlots) \
            orin_fa::g_gemv_stamps[(wg_ * 4 + (threadIdx.x >> 6)) * orin_fa::kStampSlots + (i)] =                          \
                (long long)__builtin_amdgcn_s_memrealtime();                                                               \
        __builtin_amdgcn_sched_barrier(0);                                                                                 \
    } while (0)
#define ROWS_ITEM_STAMP(i)                                  \
    do {                                                    \
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); \
        ROWS_STAMP(i);                                      \
    } while (0)
#else
#define ROWS_STAMP(i)
#define ROWS_ITEM_STAMP(i)
#endif

#include <stdlib.h>
#include <type_traits>

namespace orin_fa {
namespace {

// Lane i of a row of 16: lane (i + 8) % 16's value.
__device__ __forceinline__ float dpp_row_ror8(float v) {
    const int x = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(x, x, 0x128, 0xF, 0xF, false));
}

// Digits of the (optionally normalised) activation into LDS, in groups of G elements.  Thread t takes
// elements 8 t .. 8 t + 7 of every kWaves * 512.
template <int G, int kWaves>
__device__ float stage_digits(const GemvArgs& a, int first, int n_in, unsigned char* smem, float* red) {
    // Elements [first, first + n_in) of the activation.  With the RMS norm folded in (whole rows only), the
    // digits are those of x * w; the norm's scalar 1 / sqrt(mean(x^2) + eps), which needs the whole vector,
    // multiplies the finished row sums instead (returned): one pass over x.
    const int tid = threadIdx.x;
    const float* const ax = a.x + first;
    const float* const aw = a.norm_w ? a.norm_w + first : nullptr;
    float ss = 0.0f;
    XPair* pairs = reinterpret_cast<XPair*>(smem + Lds<G>::pairs_off(n_in));
    for (int e = tid * 8; e < n_in; e += kWaves * 64 * 8) {
        float x[8];
        *reinterpret_cast<float4*>(x) = *reinterpret_cast<const float4*>(ax + e);
        *reinterpret_cast<float4*>(x + 4) = *reinterpret_cast<const float4*>(ax + e + 4);
        if (aw) {
            float g[8];
            *reinterpret_cast<float4*>(g) = *reinterpret_cast<const float4*>(aw + e);
            *reinterpret_cast<float4*>(g + 4) = *reinterpret_cast<const float4*>(aw + e + 4);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                ss += x[i] * x[i];
                x[i] *= g[i];
            }
        }
        digits8<G>(x, e, n_in, smem, pairs, tid);
    }
    if (tid < 4) reinterpret_cast<unsigned*>(smem + Lds<G>::zero_off(n_in))[tid] = 0u;
    if (!aw) {
        __syncthreads();
        return 1.0f;
    }
    ss = wave_sum(ss);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
    __syncthreads();
    ss = 0.0f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) ss += red[w];
    __syncthreads(); // (red is reused for the row sums)
    return 1.0f / sqrtf(ss / (float)n_in + a.eps);
}

// T: weight type.  DUAL: two matrices (gate, up) and SiLU(gate) * up.  Grid: (workgroups, matrices); a
// workgroup walks the 16-row tiles blockIdx.x, + gridDim.x, ...
template <int T, bool DUAL, int kWaves>
__device__ __forceinline__ void gemv_mfma_body(const GemvArgs& a) {
    using F = MF<T>;
    using L = Lds<F::kGroup>;
    typedef typename F::Raw Raw;
    constexpr int M = DUAL ? 2 : 1;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    // gridDim.z workgroups share a tile's blocks (a matrix with few tiles and long rows, accumulating into y):
    // this one takes blocks [b0, b0 + nb), stages that part of the activation only, and adds its row sums to
    // y atomically.  gridDim.z = 1: the whole row, stored.
    const int nb_row = a.n_in >> 8;
    const int b0 = (int)blockIdx.z * nb_row / (int)gridDim.z, nb = ((int)blockIdx.z + 1) * nb_row / (int)gridDim.z - b0;
    const int n_in = nb << 8; // (elements this workgroup works on: LDS is laid out for them)
    float* const red = reinterpret_cast<float*>(smem + L::red_off(n_in));
    const GemvSeg seg = a.seg[blockIdx.y];
    const size_t row_bytes = a.n_seg_types ? seg.row_bytes : a.row_bytes;
    const int n_tiles = (seg.n_out + 15) >> 4;
    if ((int)blockIdx.x >= n_tiles) return; // (whole workgroup: a shorter matrix of a shared launch)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    LaneCtx c;
    c.n = lane & 15; c.g = lane >> 4; c.ln = lane >> 2; c.lg = lane & 3;
    c.src_lane4 = 4 * (4 * c.n + c.g);
    c.am = lane & 15;
    c.smem = smem;
    c.pairs = reinterpret_cast<const XPair*>(smem + L::pairs_off(n_in));
    c.n_in = n_in;
    c.zero_off = L::zero_off(n_in);
    const unsigned char* const wbase[2] = {static_cast<const unsigned char*>(seg.w),
                                           static_cast<const unsigned char*>(DUAL ? a.w_up : seg.w)};
    // (rows past the end repeat the last one; nothing is written for them.  Blocks past a row's end: the
    // last block once more, never used.)
    auto request = [&](Raw (&r)[M], int tile, int b) {
        const int row = min(tile * 16 + c.ln, seg.n_out - 1);
        b = min(b, nb - 1);
#pragma unroll
        for (int m = 0; m < M; ++m) F::load(wbase[m] + (size_t)row * row_bytes + (size_t)(b0 + b) * F::kBlockBytes, c.lg, r[m]);
    };
    Raw raw_a[M], raw_b[M];
    request(raw_a, blockIdx.x, wave);
    __builtin_amdgcn_sched_barrier(0);

    const float rinv = stage_digits<F::kGroup, kWaves>(a, b0 << 8, n_in, smem, red);

    const typename F::Addr addr = F::addr(c);
    float rowacc[M];
    auto finish = [&](const Raw (&r)[M], int b) {
#pragma unroll
        for (int m = 0; m < M; ++m) rowacc[m] += F::block(r[m], c, addr, b);
    };
    // Row tiles blockIdx.x, + gridDim.x, ...: the digits are staged once per workgroup.  The first block of
    // the next tile is requested while the last of this one is multiplied out.
    for (int tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        const int next_tile = tile + (int)gridDim.x < n_tiles ? tile + (int)gridDim.x : tile;
#pragma unroll
        for (int m = 0; m < M; ++m) rowacc[m] = 0.0f;
        // (raw_a holds block `wave` of this tile)
        for (int b = wave;; b += 2 * kWaves) {
            const bool more1 = b + kWaves < nb;
            request(raw_b, more1 ? tile : next_tile, more1 ? b + kWaves : wave);
            if (b < nb) finish(raw_a, b);
            if (!more1) { // raw_b holds the next tile's first block: hand it over
#pragma unroll
                for (int m = 0; m < M; ++m) raw_a[m] = raw_b[m];
                break;
            }
            const bool more2 = b + 2 * kWaves < nb;
            request(raw_a, more2 ? tile : next_tile, more2 ? b + 2 * kWaves : wave);
            finish(raw_b, b + kWaves);
            if (!more2) break;
        }
        // ---- the four sub-block lanes of a row, then the four waves ----
        const int row0 = tile * 16;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const float t = xor_sum(rowacc[m]);
            if (c.g == 0) red[(wave * M + m) * 16 + c.n] = t;
        }
        __syncthreads();
        if (threadIdx.x < 16 && row0 + (int)threadIdx.x < seg.n_out) {
            const int r = row0 + threadIdx.x;
            float v[M];
#pragma unroll
            for (int m = 0; m < M; ++m) {
                v[m] = 0.0f;
#pragma unroll
                for (int w = 0; w < kWaves; ++w) v[m] += red[(w * M + m) * 16 + threadIdx.x];
                v[m] *= rinv;
            }
            float y = v[0];
            if constexpr (DUAL) y = y / (1.0f + expf(-y)) * v[1]; // SiLU(gate) * up
            if (gridDim.z > 1) { // (a share of the row: y already holds what is accumulated into)
                if (seg.bias && blockIdx.z == 0) y += seg.bias[r];
                atomicAdd(seg.y + r, y);
            } else {
                if (seg.bias) y += seg.bias[r];
                if (a.accumulate) y += seg.y[r];
                seg.y[r] = y;
            }
        }
        __syncthreads(); // (the partial sums are free for the next tile)
    }
}

template <int T, bool DUAL, int kWaves>
__global__ __launch_bounds__(kWaves * 64) void gemv_mfma_kernel(const GemvArgs a) {
    gemv_mfma_body<T, DUAL, kWaves>(a);
}

// Q4_K, Q5_K and Q6_K rows read in long runs.  The kernel above fetches, per load instruction, 64 bytes of each of
// 16 rows; this machine's memory path moves that pattern at 4.6-4.7 TB/s where lane-linear runs of two whole blocks
// of a row (288 bytes) move at 5.5-5.8 TB/s, as fast as a plain streaming read (the read-only stand-ins of
// bench_aids.hip over the 66 MB of a Llama-3-8B gate/up pair, `bench.py --workload weights-read-patterns`: 14.1-14.4
// us a launch against 11.5-12.0; runs of one block 13.5, of four blocks 17.9).  Here a wave's item is CB <= 2
// consecutive blocks of each of a tile's 16 rows, of one matrix, fetched as (row, 16-byte piece) slots in row-major
// order, lane after lane, with streaming loads: every line is asked for by one instruction.  The pieces pass
// through a wave-private LDS buffer (rows padded to an odd number of pieces, so that the 16 rows a
// matrix-instruction operand is read from lie in 16 different bank groups) and come back in the matrix
// instruction's lane order: no lane permutations.  Two items per wave are on their way or in use; chunks w, w +
// kWaves, ... of a tile's blocks are wave w's, and so are those chunks' digits of the activation, which the wave
// makes for itself: no wave waits for another before the first tile's end, where the norm's sum of squares is put
// together as well.  Barriers wait for LDS only, row sums leave through stores and atomic adds without a return
// value, a tile's bias values travel with its items: nothing in the loop waits for anything but the oldest item.
// Requires whole 16-row tiles.  (Deeper request queues, three and four items a wave, were slower in both kernels,
// and so were four-block items: what bounds the kernels after the loads is the vector ALU, about 74 instructions
// per block and wave for the nibbles, the six-bit pairs and the digit sums.)
// Two matrices that become one product (gate, up) share a tile: eight rows of each.  Tiles of sixteen rows of each are
// half as many, and 896 of them on 256 CUs leave half the CUs with a fourth; 1792 are seven a CU (Llama-3-8B's pair in Q6_K
// 22.7 -> 20.9 us, Qwen2.5-1.5B's in Q4_K 7.2 -> 6.5 us).
// The matrices of a launch (q, k, v) have their own stretches of workgroups, one grid row: as grid rows, the shorter
// ones' empty workgroups were two of three (Llama-3.2-1B's q, k, v in Q8_0 5.9 -> 4.7 us).
// A launch smaller than the chip is a chain of latencies -- arguments, activation, digits, weights, products, sums, at 2 ns an
// instruction of a wave -- and this kernel's was cut where it could be: the arguments of the first requests come with the
// wave (below), the slots are stepped through without a division, the digits are made with one reciprocal and wait for the activation
// alone, and every wave has one item where the launcher can arrange it.  Per launch, before -> now: output projection of
// Qwen2.5-1.5B in Q4_K 3.9 -> 3.0 us and of Llama-3-8B 5.6 -> 4.4, q projections 4.3 -> 3.3 and 5.8 -> 4.7, down projections 5.7
// -> 4.4 and 10.8 -> 8.6 (33 MB, 3.85 TB/s), Qwen2.5-7B's down projection in Q5_K 14.5 -> 11.5 us (47 MB, 4.05 TB/s).

// What a launch's first requests need, in the kernel's leading argument words, which are in a wave's registers when it
// starts (kernel-argument preload): behind a trip to the argument block and the launch description, and with the
// divisions that the grid leaves to the kernel, the first weight request left a microsecond after the wave's start.
struct RowsHead {
    const void *w0, *w1, *w2; // the launch's matrices (two matrices that become one product: gate, up)
    const float *x, *norm_w;
    // of each matrix: tiles a workgroup takes at least | << 6 how many of its workgroups take one more | << 19 its first workgroup
    unsigned turns0, turns1, turns2;
    unsigned shape; // blocks of a row - 1 | blocks of a share of it - 1 << 7 | shares that take one more << 14 | workgroups of a share << 18
};
constexpr unsigned kMostRowsWgs = 8190, kMostRowsTurns = 62; // what these words have room for
constexpr int kMostRowsOneTurn = 16383; // (workgroups with one tile each of one matrix)
static_assert(kMaxRowShares <= 16, "share_extra: four bits of RowsHead::shape");
constexpr unsigned kNoMatrix = 8191; // as the first workgroup of a matrix that is not there
__device__ __forceinline__ int rows_seg(const RowsHead& h, int wg) {
    const unsigned first1 = h.turns1 >> 19, first2 = h.turns2 >> 19;
    return wg >= (int)first2 && first2 != kNoMatrix ? 2 : wg >= (int)first1 && first1 != kNoMatrix ? 1 : 0;
}

// What a launch says of every wave's share, so that nothing between the loads and their uses is under a condition and the
// compiler's waits are exact: the digits wait for the activation, not for the weights behind it.
//   kRowsOneItem    every wave has one item (or none): requested, digits, multiplied out, done.  The output and the q, k,
//                   v projections of most models.
//   kRowsOnePass, kRowsTwoPasses   several items, over one or two passes of digits: the first item is used as soon as it is
//                   there.  Only for launches that leave resident places empty, or whose workgroups have one tile or
//                   two: one that fills the chip with work runs longer this way (Llama-3-8B's gate/up by 1 us), its second
//                   round of requests getting in the way of the first.
//   kRowsAny        anything: the digits come behind the wave's first two items.
//   kRowsOneItemNorm  one item, with a norm, and at most one workgroup of up to four waves a CU: the norm's factor (two divisions and a
//                   root, about 60 instructions, in the wave that finishes the rows) is made behind a barrier of its own while
//                   the weights are on their way.  In the other modes it stands between the first tile's last product and its
//                   store, once a workgroup.  128 workgroups of 6 blocks in Q4_K 3.11 -> 3.04 us, in Q6_K 3.56 -> 3.44, in Q8_0 3.68 -> 3.52,
//                   256 of them 3.26 -> 3.18, 3.79 -> 3.67, 3.95 -> 3.81; but 384 3.93 -> 4.00, 4.56 -> 4.66, 4.93 -> 5.09, and with eight
//                   waves 224 workgroups 4.2 -> 4.35: there the vector ALU has other waves' work to do meanwhile.
enum : int { kRowsAny = 0, kRowsOnePass = 1, kRowsTwoPasses = 2, kRowsOneItem = 3, kRowsOneItemNorm = 4 };

template <int T, bool DUAL, int kWaves, int CB, int kMode>
__device__ __forceinline__ void gemv_rows_body(const RowsHead h, const GemvArgs& a) {
    using F = MF<T>;
    using L = Lds<F::kGroup>;
    using G = RowsGeom<T, CB>;
    constexpr int P = G::P, R = G::R, NL = G::NL;
    constexpr int kTileOut = DUAL ? 8 : 16; // outputs of a tile: two matrices give eight rows each to its sixteen
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    ROWS_STAMP(0);
    const void* w_mine = h.w0;
    unsigned turns = h.turns0;
    unsigned next = h.turns1;
    const int seg = DUAL ? 0 : rows_seg(h, (int)blockIdx.x);
    if (seg == 1) w_mine = h.w1, turns = h.turns1, next = h.turns2;
    if (seg == 2) w_mine = h.w2, turns = h.turns2, next = ~0u;
    const int seg_wg = (int)blockIdx.x - (int)(turns >> 19), grid_x = (int)min(next >> 19, h.shape >> 18) - (int)(turns >> 19); // among the matrix's workgroups
    // (what a mode says of the launch is a constant here: the way to the first request is scalar instructions, 2 ns each.  Of eight waves
    // only for Q6_K in runs, 14 blocks a row, 224 tiles 5.13 -> 4.88 us; Q4_K was slower for it, 4.2 -> 4.4.)
    constexpr bool kOneItem = kMode == kRowsOneItem || kMode == kRowsOneItemNorm, kWholeRows = DUAL || kMode == kRowsOneItemNorm;
    constexpr bool kAhead = kOneItem && kWaves < 8, kStraight = kOneItem && (kWaves < 8 || F::kRun);
    const int nb_row = (int)(h.shape & 0x7fu) + 1, share_blocks = kWholeRows ? nb_row : (int)((h.shape >> 7) & 0x7fu) + 1;
    const int share_extra = kWholeRows ? 0 : (int)((h.shape >> 14) & 15u), share = kWholeRows ? 0 : (int)blockIdx.z;
    const int n_mine = kStraight ? 1 : (int)(turns & 63u) + (seg_wg < (int)((turns >> 6) & 0x1fffu) ? 1 : 0); // tiles of this workgroup, one at least
    const int b0 = share * share_blocks + min(share, share_extra) * G::kUnit;
    const int nb = share_blocks + (share < share_extra ? G::kUnit : 0);
    const int n_in = nb << 8;
    const unsigned row_bytes = (unsigned)nb_row * F::kBlockBytes;
    float* const red = reinterpret_cast<float*>(smem + L::red_off(n_in));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); // (scalar: what follows from it stays in scalar registers)
    unsigned char* const transit = smem + L::red_off(n_in) + kRowsRedBytes + wave * G::kWaveBytes;
    const int n_chunks = (int)((unsigned)(nb + CB - 1) / CB);
    const int my_chunks = kStraight ? (wave < n_chunks ? 1 : 0) : (int)((unsigned)(n_chunks + kWaves - 1 - wave) / kWaves);
    const int total = n_mine * my_chunks;
    const bool has_norm = kMode == kRowsOneItemNorm || h.norm_w != nullptr;
    float* const wave_ss = red + 2 * kMaxWaves * 2 * 16;
    if (kMode != kRowsAny && total == 0) { // (fewer chunks than waves: this wave only leaves its zeros and keeps the barriers' count)
        if (lane == 0) wave_ss[wave] = 0.0f;
        if (kMode == kRowsOneItemNorm) lds_barrier();
        for (int t = 0; t < n_mine; ++t) {
            if (lane < 16) red[(t & 1) * (kMaxWaves * 2 * 16) + wave * 16 + lane] = 0.0f;
            lds_barrier();
        }
        return;
    }

    // ---- requests ----
    // slot 64 i + lane of an item: (row, piece), row-major
    unsigned goff[NL];
    int loff[NL];
    auto slots = [&] {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const unsigned s = 64u * i + (unsigned)lane, row = s / G::kRowPieces;
            const unsigned r = DUAL ? row & 7u : row; // (of its matrix)
            // (slots past the sixteenth row: cut to the item's last piece by the request -- or some row's first of two matrices --
            // and to the buffer's spare piece here)
            if constexpr (F::kRun) {
                const unsigned piece = s - __umul24(row, G::kRowPieces);
                goff[i] = __umul24(r, row_bytes) + (piece + 1 == (unsigned)G::kRowPieces ? (unsigned)F::kLastPiece : 16u * piece);
            } else if constexpr (F::kBlockBytes == 16 * P) {
                if constexpr (DUAL) goff[i] = __umul24(r, row_bytes) + 16u * (s - __umul24(row, G::kRowPieces));
                else goff[i] = __umul24(row, row_bytes - 16u * G::kRowPieces) + 16u * s;
            } else {
                const unsigned piece = s - __umul24(row, G::kRowPieces), k = piece >= (unsigned)P ? piece - P : piece;
                goff[i] = __umul24(r, row_bytes) + (piece >= (unsigned)P ? F::kBlockBytes : 0u) + (unsigned)F::piece_off((int)k);
            }
            const unsigned l = 16u * (R == G::kRowPieces ? s : s + row);
            loff[i] = (int)(64 * i + 63 >= 16 * G::kRowPieces ? min(l, 16u * R * 16u) : l);
        }
    };
    const unsigned char *const w_first = static_cast<const unsigned char*>(w_mine), *const w_second = static_cast<const unsigned char*>(h.w1);
    int rq_tile = seg_wg, rq_c = wave;
    size_t rq_off = (size_t)((unsigned)seg_wg * (unsigned)kTileOut) * row_bytes + (size_t)((unsigned)(b0 + wave * CB) * (unsigned)F::kBlockBytes);
    const size_t next_tile = (size_t)((unsigned)grid_x * (unsigned)kTileOut) * row_bytes - (size_t)((unsigned)(my_chunks * (kWaves * CB)) * (unsigned)F::kBlockBytes);
    constexpr int kRing = kOneItem ? 1 : 2; // items on their way or in use
    u32x4 buf[kRing][NL];
    float bias_v[kRing];
    auto request = [&](u32x4 (&r)[NL], bool real = true) {
        // pieces past the chunk's end in rows above the last are the row's next blocks or the next row's first (fetched,
        // never used); in the last row they are cut to the last piece
        unsigned limit = (kTileOut - 1u) * row_bytes;
        if constexpr (F::kRun) limit += (unsigned)F::kLastPiece;
        else limit += (unsigned)((min(CB, nb - rq_c * CB) - 1) * F::kBlockBytes + F::piece_off(P - 1));
        if (!real) limit = 0; // (one address for all: the same count of loads on every path)
        const unsigned char *const first = w_first + rq_off, *const second = w_second + rq_off;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            // slots 8 * kRowPieces ... are the second matrix's: one instruction at most has both
            constexpr int kFirst = DUAL ? 8 * G::kRowPieces : 64 * NL;
            const unsigned char* const base = 64 * i + 63 < kFirst ? first : 64 * i >= kFirst ? second : 64 * i + lane < kFirst ? first : second;
            // whole runs, read once: streaming loads
            const unsigned char* const p = base + min(goff[i], limit);
            if constexpr (F::kAlign == 16) r[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
            else if constexpr (F::kAlign == 4) r[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_a4*>(p));
            else r[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_a2*>(p));
        }
    };
    auto advance = [&] { // to the next item
        rq_c += kWaves;
        rq_off += kWaves * CB * F::kBlockBytes;
        if (rq_c >= n_chunks) {
            rq_c = wave;
            rq_tile += grid_x;
            rq_off += next_tile;
        }
    };
    // ---- the activation's digits: every wave makes those of its own chunks (it multiplies no others), so
    // nothing waits for another wave before the first tile's end; the norm's sum of squares is put together
    // there.  A pass is 512 elements: a chunk of two blocks, or two chunks of one.  The first passes' loads go
    // out ahead of the weight requests (loads return in order). ----
    const float* const ax = h.x + (b0 << 8);
    const float* const aw = has_norm ? h.norm_w + (b0 << 8) : ax; // (always a load)
    XPair* const pairs = reinterpret_cast<XPair*>(smem + L::pairs_off(n_in));
    const int n_passes = CB == 2 ? my_chunks : (int)((unsigned)(my_chunks + 1) / 2u);
    const int pass_lane = CB == 2 ? lane * 8 : (lane >> 5) * (kWaves * 256) + (lane & 31) * 8;
    auto elem = [&](int ps) { return (CB == 2 ? (wave + ps * kWaves) * 512 : (wave + 2 * ps * kWaves) * 256) + pass_lane; };
    auto fetch = [&](const float* p, int e, float (&v)[8]) {
        const float4* const q = reinterpret_cast<const float4*>(reinterpret_cast<const char*>(p) + (unsigned)e * 4u); // (scalar base, 32-bit offset)
        *reinterpret_cast<float4*>(v) = q[0];
        *reinterpret_cast<float4*>(v + 4) = q[1];
    };
    float ss = 0.0f;
    auto digits = [&](float (&x)[8], const float (&g)[8], int e) {
        if (has_norm) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                ss += x[i] * x[i];
                x[i] *= g[i];
            }
        }
        digits8<F::kGroup>(x, e, n_in, smem, pairs, lane);
    };
    // The wave's first kPre passes are fetched ahead of the weight requests: fetched behind them a chunk's few floats
    // wait for two items of weights, and the wave's first item for all its digits (the stage marks below, read in the
    // timeline build: first digits 1.4 us after the requests, the second chunk's 2.1 us later, the first item 0.5 us after
    // that).
    constexpr int kPre = kWaves == 8 ? 2 : 4; // (eight-wave workgroups: fewer chunks a wave, and registers for four waves a SIMD)
    float xs[kPre][8], gs[kPre][8]; // (read under the conditions they are loaded under)
    // (what follows the requests: the other arguments, in one batch, and what a lane needs to know of itself)
    float* seg_y;
    const float* seg_bias;
    float norm_eps;
    bool adds;
    LaneCtx c;
    typename F::Addr addr;
    auto request_bias = [&](float& bias, int tile) {
        if constexpr (!DUAL) bias = *(seg_bias ? seg_bias + tile * 16 + c.n : h.x); // (always a load: the same count on every path)
    };
    auto behind_requests = [&] {
        __builtin_amdgcn_sched_barrier(0);
        ROWS_STAMP(1);
        seg_y = a.seg[seg].y;
        seg_bias = a.seg[seg].bias;
        norm_eps = a.eps;
        adds = a.accumulate || share_blocks != nb_row;
        asm volatile("" ::"s"(seg_y), "s"(seg_bias), "s"(norm_eps), "s"(a.accumulate));
        c.n = lane & 15; c.g = lane >> 4; c.ln = 0; c.lg = 0; c.src_lane4 = 0;
        c.am = lane & 15;
        c.smem = smem;
        c.pairs = pairs;
        c.n_in = n_in;
        c.zero_off = L::zero_off(n_in);
        addr = F::addr(c);
        // (the first items' bias values: the first tile's, except where every item is a tile's last)
        request_bias(bias_v[0], seg_wg);
        if constexpr (kRing == 2) request_bias(bias_v[1], my_chunks == 1 && n_mine > 1 ? seg_wg + grid_x : seg_wg);
        if (lane < 4) reinterpret_cast<unsigned*>(smem + L::zero_off(n_in))[lane] = 0u; // (every wave writes the same zeros)
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (kMode != kRowsAny) {
        constexpr int kPasses = kMode == kRowsTwoPasses ? 2 : 1;
#pragma unroll
        for (int i = 0; i < kPasses; ++i) {
            const int e = min(elem(i), n_in - 8);
            fetch(ax, e, xs[i]);
            fetch(aw, e, gs[i]);
        }
        __builtin_amdgcn_sched_barrier(0);
        slots();
        request(buf[0]);
        if constexpr (kRing == 2) {
            if (total > 1) advance();
            request(buf[1], total > 1);
            advance();
        }
        behind_requests();
#pragma unroll
        for (int i = 0; i < kPasses; ++i) {
            const int e = elem(i);
            if (e < n_in) digits(xs[i], gs[i], e);
        }
    } else {
#pragma unroll
        for (int i = 0; i < kPre; ++i)
            if (i < n_passes) {
                const int e = min(elem(i), n_in - 8);
                fetch(ax, e, xs[i]);
                fetch(aw, e, gs[i]);
            }
        __builtin_amdgcn_sched_barrier(0);
        slots();
        if (total > 0) {
            request(buf[0]);
            advance();
        }
        if (total > 1) {
            request(buf[1]);
            advance();
        }
        behind_requests();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // (both items, see above)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kPre; ++i)
            if (i < n_passes) {
                const int e = elem(i);
                if (e < n_in) digits(xs[i], gs[i], e);
            }
        for (int ps = kPre; ps < n_passes; ++ps) { // (rows longer still: these loads queue behind the weights)
            const int e = elem(ps);
            if (e < n_in) {
                float x[8], g[8];
                fetch(ax, e, x);
                fetch(aw, e, g);
                digits(x, g, e);
            }
        }
    }
    float rinv = 0.0f;
    auto norm_factor = [&] {
        float ss = 0.0f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) ss += wave_ss[w];
        rinv = 1.0f / sqrtf(ss / (float)n_in + norm_eps);
    };
    if (has_norm) {
        ss = wave_sum(ss);
        if (lane == 0) wave_ss[wave] = ss;
        if constexpr (kMode == kRowsOneItemNorm) {
            lds_barrier();
            if (wave == 0) norm_factor();
        }
    }
    ROWS_STAMP(2);
    [[maybe_unused]] int n_consumed = 0;
    int set = 0;
    auto tile_end = [&](int tile, float rowacc, float bias) {
        float* const mine = red + set * (kMaxWaves * 2 * 16);
        set ^= 1;
        const float t = xor_sum(rowacc);
        if (c.g == 0) mine[wave * 16 + c.n] = t;
        lds_barrier();
        if (threadIdx.x < 16) {
            float y = 0.0f;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) y += mine[w * 16 + threadIdx.x];
            if (has_norm) { // (every wave has left its sum of squares before its first barrier here)
                if (kMode != kRowsOneItemNorm && tile == seg_wg) norm_factor();
                y *= rinv;
            }
            if constexpr (DUAL) { // SiLU(gate) * up: rows 0-7 and 8-15
                const float up = dpp_row_ror8(y);
                y = y / (1.0f + expf(-y)) * up;
            } else if (seg_bias && share == 0) {
                y += bias;
            }
            const int r = tile * kTileOut + (int)threadIdx.x;
            if (!DUAL || threadIdx.x < 8) {
                if (adds) atomicAdd(seg_y + r, y); // (one writer a row and share: with one share the sum is the plain one)
                else seg_y[r] = y;
            }
        }
        ROWS_STAMP(13);
    };
    if (kMode == kRowsAny && total == 0) { // (here and not ahead of the requests: the loads' order and waits as they are cost 4 % less)
        for (int t = 0; t < n_mine; ++t) tile_end(seg_wg + t * grid_x, 0.0f, 0.0f);
        return;
    }
    int cs_tile = seg_wg, cs_c = wave;
    float rowacc = 0.0f;
    auto consume = [&](const u32x4 (&r)[NL], float bias) {
        auto words = [&](auto jc) {
            constexpr int j = decltype(jc)::value;
            if constexpr (F::kRun) return F::template run_words<j>(transit + c.n * R * 16, c);
            else return F::words(transit + (c.n * R + j * P) * 16, c);
        };
        auto park = [&] {
#pragma unroll
            for (int i = 0; i < NL; ++i) *reinterpret_cast<u32x4*>(transit + loff[i]) = r[i];
            ROWS_ITEM_STAMP(3 + n_consumed);
            ++n_consumed;
        };
        const int cb = min(CB, nb - cs_c * CB);
        float v;
        // (unrolled over CB with a test per block, not a loop over cb: every LDS offset is a constant of its instruction)
        if constexpr (kAhead) {
            // What the products take from the activation is fetched while the weights are on their way, and all of an item's
            // weights are asked of LDS at once: one trip to LDS between their arrival and the products, not one for every
            // few operands.  Per launch, before -> now: Qwen2.5-1.5B's q, k, v (v in Q6_K) 3.62 -> 3.50 us, gate/up in Q4_K 5.95 -> 5.87,
            // in Q6_K 7.16 -> 7.04, in Q8_0 8.75 -> 7.97, down projection 5.20 -> 5.10, output 2.73 -> 2.70; Llama-3.2-1B's q, k, v 4.03 -> 3.90,
            // output 2.86 -> 2.78.  (Not with eight waves, whose fetches keep LDS busy for longer than the weights are away: Q4_K,
            // 14 blocks, 32 tiles 3.72 -> 3.87, 224 tiles 4.2 -> 4.27.)
            typename F::Digits x[CB][2];
#pragma unroll
            for (int j = 0; j < CB; ++j)
#pragma unroll
                for (int h = 0; h < 2; ++h) x[j][h] = F::digits(c, addr, cs_c * CB + j, h);
            __builtin_amdgcn_sched_barrier(0);
            park();
            const typename F::Words w0 = words(IntC<0>{}), w1 = words(IntC<CB - 1>{});
            __builtin_amdgcn_sched_barrier(0);
            v = F::product(w0, [&](int h) { return x[0][h]; }, c);
            if constexpr (CB == 2) {
                const float second = F::product(w1, [&](int h) { return x[1][h]; }, c);
                v += F::kRun || cb == 2 ? second : 0.0f;
            }
        } else {
            park();
            auto block = [&](auto jc) {
                constexpr int j = decltype(jc)::value;
                const auto of_half = [&](int h) { return F::digits(c, addr, cs_c * CB + j, h); };
                if constexpr (F::kRun) return F::product(F::template run_words<j>(transit + c.n * R * 16, c), of_half, c);
                else return F::from_lds(transit + (c.n * R + j * P) * 16, of_half, c);
            };
            v = block(IntC<0>{});
            static_assert(CB <= 2, "blocks of an item");
            if constexpr (CB == 2)
                if (F::kRun || cb == 2) v += block(IntC<1>{});
        }
        rowacc += v;
        cs_c += kWaves;
        if (kStraight || cs_c >= n_chunks) {
            tile_end(cs_tile, rowacc, bias);
            cs_c = wave;
            cs_tile += grid_x;
            rowacc = 0.0f;
        }
    };
    auto request_next = [&](int j) {
        request_bias(bias_v[j], rq_tile);
        request(buf[j]);
        advance();
    };
    if constexpr (kRing == 1) {
        consume(buf[0], bias_v[0]);
    } else {
        // Steady state: every item consumed is followed by the request kRing items on, which exists: no branch around
        // a load, so the compiler's wait counts are exact.
        int k = 0;
        for (; k + 2 * kRing <= total; k += kRing) {
#pragma unroll
            for (int j = 0; j < kRing; ++j) {
                consume(buf[j], bias_v[j]);
                request_next(j);
            }
        }
        // the last two or three items (or the only one)
        if (k < total) consume(buf[0], bias_v[0]);
        if (k + 2 < total) request_next(0);
        if (k + 1 < total) consume(buf[1], bias_v[1]);
        if (k + 2 < total) consume(buf[0], bias_v[0]);
    }
    ROWS_STAMP(14);
}

#define ROWS_HEAD_ARGS const void *w0, const void *w1, const void *w2, const float *x, const float *norm_w, unsigned turns0, unsigned turns1, unsigned turns2, unsigned shape
template <int T, bool DUAL, int kWaves, int CB, int kMode>
__global__ __launch_bounds__(kWaves * 64) void gemv_rows_kernel(ROWS_HEAD_ARGS, const GemvArgs a) {
    gemv_rows_body<T, DUAL, kWaves, CB, kMode>(RowsHead{w0, w1, w2, x, norm_w, turns0, turns1, turns2, shape}, a);
}

// Matrices of different block types in one launch (the q, k, v projections of a file that keeps attn_v in
// Q6_K): a workgroup belongs to one matrix and runs that matrix's code.
template <int kWaves>
__global__ __launch_bounds__(kWaves * 64) void gemv_mfma_mixed_kernel(const GemvArgs a) {
    switch (a.seg[blockIdx.y].type) {
    case kQ4_K: gemv_mfma_body<kQ4_K, false, kWaves>(a); break;
    case kQ5_K: gemv_mfma_body<kQ5_K, false, kWaves>(a); break;
    case kQ6_K: gemv_mfma_body<kQ6_K, false, kWaves>(a); break;
    default: gemv_mfma_body<kQ8_0, false, kWaves>(a); break;
    }
}

// The same for the kernel that reads rows in long runs (no Q8_0 there: a file of that format has no other beside it).
// (nothing is cut into shares here: RowsHead::shape's bits for those carry the types, two bits each)
constexpr unsigned rows_type_code(int type) { return type == kQ4_K ? 0u : type == kQ5_K ? 1u : type == kQ6_K ? 2u : 3u; }
template <int kWaves, int CB, int kMode>
__global__ __launch_bounds__(kWaves * 64) void gemv_rows_mixed_kernel(ROWS_HEAD_ARGS, const GemvArgs a) {
    const RowsHead h{w0, w1, w2, x, norm_w, turns0, turns1, turns2, (shape & ~0x3ff80u) | (shape & 0x7fu) << 7};
    switch ((shape >> (7 + 2 * rows_seg(h, (int)blockIdx.x))) & 3u) {
    case rows_type_code(kQ4_K): gemv_rows_body<kQ4_K, false, kWaves, CB, kMode>(h, a); break;
    case rows_type_code(kQ5_K): gemv_rows_body<kQ5_K, false, kWaves, CB, kMode>(h, a); break;
    case rows_type_code(kQ6_K): gemv_rows_body<kQ6_K, false, kWaves, CB, kMode>(h, a); break;
    default:
        if constexpr (CB == 2) gemv_rows_body<kQ6_KRun, false, kWaves, CB, kMode>(h, a);
        break;
    }
}

// The leading arguments of a launch of `wgs` workgroups for every share of a row (as many as the matrices have tiles, or
// fewer, which then divide over the matrices as the tiles do), and whether they hold it.  A row is cut into shares of whole units.
bool rows_head(const GemvArgs& a, int wgs, int shares, int unit, RowsHead& h) {
    const int nb = a.n_in / 256, units = nb / unit;
    if (shares > units) return false;
    const void* w[3] = {};
    unsigned tiles[3] = {}, turns[3] = {kNoMatrix << 19, kNoMatrix << 19, kNoMatrix << 19}, total = 0, first = 0;
    for (int i = 0; i < a.n_seg; ++i) total += tiles[i] = (unsigned)a.seg[i].n_out / (a.w_up ? 8 : 16);
    for (int i = 0; i < a.n_seg; ++i) {
        const unsigned rest = (unsigned)wgs - first, more = (unsigned)(a.n_seg - 1 - i); // (one for every matrix behind this one)
        const unsigned mine = i + 1 == a.n_seg ? min(rest, tiles[i]) : min(rest - more, max(1u, (unsigned)((size_t)tiles[i] * (unsigned)wgs / total)));
        if (mine < 1 || tiles[i] / mine > kMostRowsTurns) return false;
        w[i] = a.seg[i].w;
        turns[i] = tiles[i] / mine | tiles[i] % mine << 6 | first << 19;
        first += mine;
    }
    h = RowsHead{w[0], a.w_up ? a.w_up : w[1], w[2], a.x, a.norm_w, turns[0], turns[1], turns[2],
                 (unsigned)(nb - 1) | (unsigned)(units / shares * unit - 1) << 7 | (unsigned)(units % shares) << 14 | first << 18};
    return (first <= kMostRowsWgs || (a.n_seg == 1 && first == tiles[0] && first <= (unsigned)kMostRowsOneTurn)) && shares <= kMaxRowShares && nb <= 128;
}
#define ROWS_HEAD_OF(h) (h).w0, (h).w1, (h).w2, (h).x, (h).norm_w, (h).turns0, (h).turns1, (h).turns2, (h).shape

constexpr size_t kMfmaLdsMax = 96u * 1024u;

template <int T>
size_t lds_bytes(int n_in) { return Lds<MF<T>::kGroup>::bytes(n_in); }

// The long-run kernel where it applies: whole 16-row tiles, LDS within the limit, and of Q8_0 only matrices that start on
// a 16-byte boundary.
bool rows_enabled() {
    static const bool on = getenv("ORIN_GEMV_NO_ROWS") == nullptr;
    return on;
}
// Its workgroups per CU: three (staging is each wave's own business there, so a workgroup more costs little and
// hides more of the others' waits) or two (rows_two_a_cu()); ORIN_GEMV_MFMA_WGS_PER_CU overrides as for the other kernel.
int rows_wgs_per_cu(int given, int usual) {
    static const bool env = getenv("ORIN_GEMV_MFMA_WGS_PER_CU") != nullptr;
    return env ? given : usual;
}

// Tiles of a launch's matrices: 16 rows, or 8 of each of two.
int rows_tiles(const GemvArgs& a) {
    int n = 0;
    for (int i = 0; i < a.n_seg; ++i) n += a.seg[i].n_out / (a.w_up ? 8 : 16);
    return n;
}

int g_rows_resident = 768; // workgroups of four waves the chip holds at once (three a CU; set by the launcher)

bool rows_norm_first(const GemvArgs& a, int wgs) { return a.norm_w && wgs * 3 <= g_rows_resident; } // (kRowsOneItemNorm)

template <int T, bool DUAL, int kWaves, int CB>
bool launch_rows_as(const GemvArgs& a, int wgs, int shares, hipStream_t stream) {
    constexpr int kUnit = RowsGeom<T, CB>::kUnit;
    const int n_in_wg = (a.n_in / 256 / kUnit + shares - 1) / shares * kUnit * 256;
    const size_t lds = RowsGeom<T, CB>::lds_bytes(n_in_wg, kWaves);
    if (lds > kMfmaLdsMax) return false;
    RowsHead h;
    if (!rows_head(a, wgs, shares, kUnit, h)) return false;
    const dim3 grid(h.shape >> 18, 1, shares);
    const int per_wave = ((n_in_wg / 256 + CB - 1) / CB + kWaves - 1) / kWaves, passes = CB == 2 ? per_wave : (per_wave + 1) / 2; // of a tile, at most
    auto go = [&](auto mode) {
        hipLaunchKernelGGL((gemv_rows_kernel<T, DUAL, kWaves, CB, decltype(mode)::value>), grid, dim3(kWaves * 64), lds, stream, ROWS_HEAD_OF(h), a);
    };
    if (per_wave == 1 && wgs == rows_tiles(a)) {
        if constexpr (kWaves == 4) {
            if (rows_norm_first(a, wgs)) {
                go(std::integral_constant<int, kRowsOneItemNorm>());
                return true;
            }
        }
        go(std::integral_constant<int, kRowsOneItem>());
        return true;
    }
    // (two matrices' tiles are half as large: up to three tiles for two workgroups)
    // Workgroups of eight waves (q, k, v of Llama-3-8B in Q8_0 9.6 -> 8.9 us): up to half the waves that are resident.
    const bool few = DUAL ? wgs * 3 >= rows_tiles(a) * 2 : wgs * shares <= g_rows_resident * (kWaves == 4 ? 3 : 2) / 4;
    if (few && passes <= 2) {
        if (passes == 1) go(std::integral_constant<int, kRowsOnePass>());
        else go(std::integral_constant<int, kRowsTwoPasses>());
        return true;
    }
    go(std::integral_constant<int, kRowsAny>());
    return true;
}

// Q8_0's 34-byte blocks: 256 elements are seventeen whole 16-byte pieces where the matrix starts on one, and the loads are
// then aligned and the runs go through LDS as they are (MF<kQ8_0>::from_lds).  Llama-3.2-1B's shapes, per launch with 64
// bytes of each of 16 rows per instruction -> in long runs: gate/up 13.7 -> 9.8 us (35.7 MB, 3.65 TB/s), down 8.6 -> 6.8,
// q, k, v 8.4 -> 6.5, output projection 6.5 -> 4.5, logits 63.4 -> 45.8 us (279 MB, 6.1 TB/s).
bool rows_base_ok(int type, const void* w) { return type != kQ8_0 || (reinterpret_cast<uintptr_t>(w) & 15u) == 0; }

// Q6_K in runs of two blocks (kQ6_KRun): rows of an even number of blocks, at least two a share, in matrices that start on a word.
bool rows_run_base_ok(const void* w) { return (reinterpret_cast<uintptr_t>(w) & 3u) == 0; }
bool rows_runs_ok(const GemvArgs& a, int shares) {
    const int nb = a.n_in / 256;
    bool ok = nb % 2 == 0 && nb / 2 >= shares && (!a.w_up || rows_run_base_ok(a.w_up));
    for (int i = 0; i < a.n_seg; ++i) ok = ok && rows_run_base_ok(a.seg[i].w);
    return ok;
}

// Workgroups of as many waves as a row has items of two blocks, two or three, where every workgroup has one tile: 0 for the four
// (or eight) waves of the other launches.  Four waves take a row of 4 blocks a block at a time, in runs half as long (and in
// Q6_K from any 2-byte boundary), and of a row of 5 or 6 blocks leave the fourth wave its place and nothing to do: with many
// workgroups a CU longer runs and more tiles in flight win, with few a wave's shorter chain does.  Four waves -> two or three,
// us a launch, 1024 elements a row: 151936 rows in Q6_K 30.9 -> 26.0, in Q4_K 21.7 -> 19.6, in Q5_K 24.3 -> 23.3, in Q8_0 31.0 ->
// 29.3; 16384 rows (four workgroups a CU) 5.9 -> 5.5, 5.0 -> 4.5, 5.25 -> 5.0, 6.1 -> 6.1; 12288 rows 4.9 -> 4.9, 4.3 -> 4.25, 4.4 ->
// 4.7, 5.1 -> 5.2.  1536 elements a row: 151936 rows in Q6_K 38.6 -> 36.6, in Q5_K 32.9 -> 31.6, in Q8_0 47.2 -> 42.3, in Q4_K 27.0
// -> 27.1 (not taken); 16384 rows 6.95 -> 6.93, 6.1 -> 6.3, 8.1 -> 7.8; two matrices of 8960 rows 8.1 -> 7.6, 6.7 -> 6.8, 9.05 ->
// 8.9.  In Q8_0, whose items of one block these would otherwise be, three waves are at least as fast at every size (64 tiles
// of two matrices 3.9 -> 3.7).
template <int T>
int rows_small_waves(const GemvArgs& a, int wgs, int shares, int nb) {
    const int tiles = rows_tiles(a), cus = g_rows_resident / 3;
    if (shares != 1 || wgs != tiles || nb < 4 || nb > 6 || (T == kQ6_K && !rows_runs_ok(a, 1))) return 0;
    if (nb == 4) return tiles >= 4 * cus ? 2 : 0;
    if (T == kQ8_0) return 3;
    return T != kQ4_K && tiles >= (T == kQ6_K && a.w_up ? 4 : 6) * cus ? 3 : 0;
}

template <int T, bool DUAL, int kWaves>
bool launch_rows_one_item(const GemvArgs& a, int wgs, hipStream_t stream) {
    const size_t lds = RowsGeom<T, 2>::lds_bytes(a.n_in, kWaves);
    RowsHead h;
    if (lds > 64u * 1024u || !rows_head(a, wgs, 1, RowsGeom<T, 2>::kUnit, h)) return false;
    auto go = [&](auto mode) {
        hipLaunchKernelGGL((gemv_rows_kernel<T, DUAL, kWaves, 2, decltype(mode)::value>), dim3(h.shape >> 18), dim3(kWaves * 64), lds, stream, ROWS_HEAD_OF(h), a);
    };
    if constexpr (T == kQ8_0 && kWaves == 3) { // (the others here are launches of several workgroups a CU)
        if (rows_norm_first(a, wgs)) {
            go(std::integral_constant<int, kRowsOneItemNorm>());
            return true;
        }
    }
    go(std::integral_constant<int, kRowsOneItem>());
    return true;
}

template <int T>
bool launch_rows(const GemvArgs& a, int wgs, int shares, bool wide, int nb_wg, hipStream_t stream) {
    if (!rows_enabled()) return false;
    for (int i = 0; i < a.n_seg; ++i)
        if (a.seg[i].n_out % 16 != 0 || !rows_base_ok(T, a.seg[i].w)) return false;
    if (a.w_up && !rows_base_ok(T, a.w_up)) return false;
    if (const int waves = wide ? 0 : rows_small_waves<T>(a, wgs, shares, nb_wg)) {
        constexpr int R = T == kQ6_K ? (int)kQ6_KRun : T;
        if (waves == 2 ? (a.w_up ? launch_rows_one_item<R, true, 2>(a, wgs, stream) : launch_rows_one_item<R, false, 2>(a, wgs, stream))
                       : (a.w_up ? launch_rows_one_item<R, true, 3>(a, wgs, stream) : launch_rows_one_item<R, false, 3>(a, wgs, stream))) return true;
    }
    // Q8_0: 272 bytes are a long run already, so two blocks only where they make one item of a wave's share, and with eight waves,
    // whose buffers then leave room for one workgroup a CU, only up to a workgroup a CU (two blocks against one: 4096 x 4096 5.7 and
    // 6.05 us, 4096 x 1024 4.7 and 5.2; 4096 x 6144, 384 workgroups, 9.3 and 8.4).
    if constexpr (T == kQ8_0) {
        if (wide) return nb_wg <= 16 && wgs <= g_rows_resident / 3 ? launch_rows_as<T, false, 8, 2>(a, wgs, shares, stream) : launch_rows_as<T, false, 8, 1>(a, wgs, shares, stream);
        if (!a.w_up && nb_wg > 4 && nb_wg <= 8 && wgs == rows_tiles(a)) return launch_rows_as<T, false, 4, 2>(a, wgs, shares, stream);
        // One matrix in many turns: two-block items, where a run of one block begins and ends inside a line that the next wave's fetches again
        // (logits of Llama-3-8B 92.7 -> 87.8 us, 6.4 TB/s, of Qwen2.5-7B 99.6 -> 93.2).  With fewer turns the longer last item costs more (even
        // at five, 4 % slower at four, 7 at three, 28 at one and a third), and so does a wave without an item (8 blocks a row: 47.5 -> 52.4).
        // From 19 blocks on two workgroups fit a CU instead of three, and it is faster still (152064 rows, one block -> two: of 20 blocks
        // 141 -> 133, 32 214 -> 197, 72 484 -> 445); up to where the buffers and the digits fit LDS, where one-block items take over (80
        // blocks 517 us; the kernel that does not read in runs 731).  18 blocks, nine items for four waves, lose where some workgroups
        // have a turn more than others and there are few turns (of 768 workgroups, 8 1/2 turns 87.4 -> 96.7 us, 10 1/2 108 -> 116, 12 1/2
        // 129 -> 133; but 10 whole ones 103 -> 97, 14 1/2 150 -> 142, 21 208 -> 198); 17 blocks, whose ninth item is half as long, do not.
        const int turns = rows_tiles(a) / wgs;
        const bool uneven = nb_wg == 18 && turns < 13 && rows_tiles(a) % wgs != 0;
        if (!a.w_up && nb_wg >= 14 && turns >= 8 && !uneven && RowsGeom<T, 2>::lds_bytes(nb_wg * 256, 4) <= kMfmaLdsMax)
            return launch_rows_as<T, false, 4, 2>(a, wgs, shares, stream);
        return a.w_up ? launch_rows_as<T, true, 4, 1>(a, wgs, shares, stream) : launch_rows_as<T, false, 4, 1>(a, wgs, shares, stream);
    }
    else { // (the other branch returned)
    // runs of 288 (352) bytes read within a few percent of longer ones, and the wave's last item, which nothing
    // overlaps, is half as long as with four blocks
    const int cb = min(kRowsMaxCb, (nb_wg + 3) / 4);
    if constexpr (T == kQ6_K) {
        if (rows_runs_ok(a, shares) && (wide || cb == 2))
            return wide ? launch_rows_as<kQ6_KRun, false, 8, 2>(a, wgs, shares, stream)
                        : a.w_up ? launch_rows_as<kQ6_KRun, true, 4, 2>(a, wgs, shares, stream) : launch_rows_as<kQ6_KRun, false, 4, 2>(a, wgs, shares, stream);
    }
    if (wide) return launch_rows_as<T, false, 8, 2>(a, wgs, shares, stream); // (sixteen blocks at least; never two matrices)
    if (a.w_up) {
        return cb == 1 ? launch_rows_as<T, true, 4, 1>(a, wgs, shares, stream) : launch_rows_as<T, true, 4, 2>(a, wgs, shares, stream);
    }
    return cb == 1 ? launch_rows_as<T, false, 4, 1>(a, wgs, shares, stream) : launch_rows_as<T, false, 4, 2>(a, wgs, shares, stream);
    }
}

// Two workgroups a CU instead of three for one matrix or pair that takes the chip several turns: each makes the digits of the whole row for
// itself and fetches activation and norm weights, and the weights of two, two items a wave, are enough on their way.  Where a row's items come out
// even among the four waves, or, of one matrix and of Q6_K, one short of it; with fewer the waves that have none leave too
// little under way (1536 tiles of 9 to 12 blocks +2 to +4 %, 2048 +10 %; 18 and 20 blocks 0 to +6 %).  Q8_0, whose items are one block: pairs from
// 12 blocks on (8 to 10: -2 to +5 %; one matrix: its items are chosen by turns, as measured with three).  us a launch, three -> two:
//   two matrices of 14336 rows (7 tiles a CU)   of 16 blocks: Q4_K 14.67 -> 13.50, Q5_K 17.41 -> 15.96, Q6_K 20.24 -> 18.42, Q8_0 25.4 -> 23.9
//     of 24: 20.2 -> 19.45, 23.8 -> 22.8, 28.3 -> 26.8, 36.8 -> 35.8; of 32: 25.4 -> 24.1, 30.0 -> 28.9, 40.6 -> 34.2, 47.1 -> 45.5
//   of 18944 rows (9 1/4)   of 14 blocks: Q6_K 23.3 -> 22.9, Q8_0 30.2 -> 29.7 (Q4_K 16.4 -> 17.1, Q5_K 19.6 -> 20.5: not taken)
//   one matrix of 152064 rows   of 14 blocks: 51.1 -> 49.5, 62.1 -> 60.9, 74.6 -> 73.6; of 16: 55.0 -> 53.8, 66.5 -> 65.8, 81.3 -> 80.3
// Tiles a CU, rounded up, at which three are the faster: four where a pair's rows have 16 blocks or fewer (800 tiles of 16 blocks in Q4_K by three
// 9.1, by two 9.5; one matrix of them 9.2, 8.6); and, in Q4_K and Q5_K, six where they have 21 to 24 (1300 tiles of 24: 16.2, 16.9; 1552 to 1744,
// seven a CU, 1 to 7 % faster by two; of Q6_K only pairs of 22 and 24), eight where they have more than 16 or are a pair's (2000 tiles: pairs of
// 16 blocks 14.7, 15.3, one of 22 20.1, 20.5; 2064 to 2256 3 to 6 % faster by two), ten likewise up to 24.  Of 2055 launches, 784 to 8000 tiles of 12
// to 32 blocks, two were over 1.2 % slower at 127, up to 6 %; of 420 that the lines leave to three, each timed both ways in turn, three are over
// 1.2 % faster at 153, up to 5 %, and slower at 23, up to 2, most of those since taken by two.
// (Not where two would take more turns than rows_head() has room for: the launch would leave this kernel.)
template <int T>
bool rows_two_a_cu(const GemvArgs& a, int tiles, int cu_count) {
    const int nb = a.n_in / 256, last = (nb + 1) / 2 % 4, per_cu = (tiles + cu_count - 1) / cu_count;
    if (a.n_seg != 1 || tiles <= 3 * cu_count || nb > 32 || tiles / (2 * cu_count) > (int)kMostRowsTurns) return false;
    if (T == kQ8_0) return a.w_up && nb >= 12 && (nb != 16 || per_cu > 4);
    if (a.w_up && nb <= 16 && per_cu <= 4) return false;
    if (per_cu == 6 && nb > 16 && nb <= 24 && (T != kQ6_K || (a.w_up && nb % 2 == 0))) return false;
    if (T != kQ6_K && (a.w_up || nb > 16) && (per_cu == 8 || (per_cu == 10 && nb <= 24))) return false;
    return nb >= 14 && (last == 0 || (last == 3 && (!a.w_up || T == kQ6_K)));
}

template <int T>
hipError_t launch(const GemvArgs& a, int cu_count, hipStream_t stream) {
    int max_out = 0;
    for (int i = 0; i < a.n_seg; ++i) max_out = max(max_out, a.seg[i].n_out);
    const int cap = a.mfma_wgs_per_cu > 0 ? cu_count * a.mfma_wgs_per_cu : (max_out + 15) / 16;
    const dim3 grid(min((max_out + 15) / 16, cap), a.n_seg);
    dim3 g3 = grid;
    // A matrix with too few tiles to fill the chip whose rows are long, accumulating into y without a norm (output
    // and down projections): 2 or 4 workgroups share a tile's blocks, each staging its own part of the activation.
    const int nb_row = a.n_in / 256;
    int ks = 1;
    if (a.accumulate && !a.w_up && !a.norm_w && (int)(grid.x * grid.y) <= cu_count) ks = nb_row >= 32 ? 4 : nb_row >= 12 ? 2 : 1;
    if (a.k_split_override > 0) ks = a.accumulate && !a.w_up && !a.norm_w ? min(a.k_split_override, nb_row) : 1;
    g3.z = ks;
    // Eight waves a workgroup where a row has the blocks to share out and a workgroup has one tile only (a
    // second tile would have amortised the staging instead).
    const bool wide = ks == 1 && nb_row >= 16 && !a.w_up && (int)grid.x == (max_out + 15) / 16;
    {
        g_rows_resident = cu_count * 3;
        const int tiles = rows_tiles(a);
        const int per_cu = rows_wgs_per_cu(a.mfma_wgs_per_cu, rows_two_a_cu<T>(a, tiles, cu_count) ? 2 : 3);
        // One item a wave where a row is short enough: as many workgroups as there are tiles, for the chip to hand out, and
        // no second turn.  Of two matrices up to 8 blocks (Qwen2.5-1.5B's gate/up in Q4_K 6.5 -> 6.1 us; 16 blocks in workgroups
        // of eight waves: Llama-3-8B's 15.0 -> 17.4), in Q8_0 up to 6 (rows_small_waves(); 8 blocks: Llama-3.2-1B's 9.9 -> 10.2 us); of one
        // matrix up to 6, which would leave a fourth of the waves of long-lived workgroups without a chunk
        // (Qwen2.5-1.5B's logits in Q6_K 38.4 -> 35.7 us; 8 blocks: Llama-3.2-1B's in Q5_K 32.6 -> 34.4).
        const bool one_item = nb_row <= (!a.w_up || T == kQ8_0 ? 6 : 8) && tiles <= kMostRowsOneTurn;
        const int wgs = one_item || per_cu <= 0 ? tiles : min(tiles, cu_count * per_cu);
        // Shares of a row of a matrix that is accumulated into: up to 8 blocks, so that every wave has one item.  Digits
        // are each share's own, so more shares make no more of them, and the chip evens out what workgroups of two long
        // shares a CU did not (Qwen2.5-7B's down projection in Q5_K 13.9 -> 11.5 us, Llama-3-8B's in Q4_K 10.0 -> 8.6).  Smaller
        // ones where that still leaves CUs empty (output projection of Qwen2.5-1.5B: 3.15 -> 3.0 us).
        int ks_r = ks;
        if (a.k_split_override <= 0) {
            ks_r = 1;
            if (a.accumulate && !a.w_up && !a.norm_w && tiles <= cu_count) {
                ks_r = min((nb_row + 7) / 8, kMaxRowShares);
                while (tiles * ks_r * 2 <= cu_count && ks_r * 2 <= kMaxRowShares && nb_row >= ks_r * 4) ks_r *= 2;
            }
        }
        // Eight waves from 9 blocks a row on, which gives a wave one item up to 16 (Qwen2.5-7B's q, k, v in Q5_K and Q6_K 8.4 ->
        // 6.4 us); of Q8_0, up to 15 blocks only where there are three workgroups on two CUs at most: 288 of them 6.85 -> 6.36
        // us with 9 blocks, 8.25 -> 7.46 with 12, 8.26 -> 8.06 with 14, 384 of them 7.0 -> 6.65, 8.5 -> 7.8, 9.04 -> 9.0; with 448
        // 7.2 -> 7.1, 9.45 -> 9.1, but 9.6 -> 9.8.
        const bool wide_r = ks_r == 1 && nb_row > (T == kQ8_0 && 2 * tiles > 3 * cu_count ? 15 : 8) && !a.w_up && wgs == tiles;
        if (launch_rows<T>(a, wgs, ks_r, wide_r, (nb_row + ks_r - 1) / ks_r, stream)) return hipGetLastError();
    }
    const size_t lds = lds_bytes<T>((nb_row + ks - 1) / ks * 256);
    if (a.w_up) {
        if (wide) hipLaunchKernelGGL((gemv_mfma_kernel<T, true, 8>), g3, dim3(512), lds, stream, a);
        else hipLaunchKernelGGL((gemv_mfma_kernel<T, true, 4>), g3, dim3(256), lds, stream, a);
    } else {
        if (wide) hipLaunchKernelGGL((gemv_mfma_kernel<T, false, 8>), g3, dim3(512), lds, stream, a);
        else hipLaunchKernelGGL((gemv_mfma_kernel<T, false, 4>), g3, dim3(256), lds, stream, a);
    }
    return hipGetLastError();
}

template <int T, bool DUAL>
hipError_t allow() {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemv_mfma_kernel<T, DUAL, 4>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMfmaLdsMax);
    if (e != hipSuccess) return e;
    return hipFuncSetAttribute(reinterpret_cast<const void*>(&gemv_mfma_kernel<T, DUAL, 8>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMfmaLdsMax);
}

hipError_t allow_lds(const void* kernel) { return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMfmaLdsMax); }

template <int T, bool DUAL, int kWaves, int CB>
hipError_t allow_rows() {
    hipError_t e;
    if ((e = allow_lds(reinterpret_cast<const void*>(&gemv_rows_kernel<T, DUAL, kWaves, CB, kRowsOnePass>))) != hipSuccess) return e;
    if ((e = allow_lds(reinterpret_cast<const void*>(&gemv_rows_kernel<T, DUAL, kWaves, CB, kRowsTwoPasses>))) != hipSuccess) return e;
    if ((e = allow_lds(reinterpret_cast<const void*>(&gemv_rows_kernel<T, DUAL, kWaves, CB, kRowsOneItem>))) != hipSuccess) return e;
    if constexpr (kWaves == 4)
        if ((e = allow_lds(reinterpret_cast<const void*>(&gemv_rows_kernel<T, DUAL, kWaves, CB, kRowsOneItemNorm>))) != hipSuccess) return e;
    return allow_lds(reinterpret_cast<const void*>(&gemv_rows_kernel<T, DUAL, kWaves, CB, kRowsAny>));
}

template <int kWaves, int CB>
hipError_t allow_mixed() {
    hipError_t e = allow_lds(reinterpret_cast<const void*>(&gemv_rows_mixed_kernel<kWaves, CB, kRowsOneItem>));
    if constexpr (kWaves == 4)
        if (e == hipSuccess) e = allow_lds(reinterpret_cast<const void*>(&gemv_rows_mixed_kernel<kWaves, CB, kRowsOneItemNorm>));
    return e != hipSuccess ? e : allow_lds(reinterpret_cast<const void*>(&gemv_rows_mixed_kernel<kWaves, CB, kRowsAny>));
}

hipError_t allow_rows_runs() {
    hipError_t e;
    if ((e = allow_rows<kQ6_KRun, false, 8, 2>()) != hipSuccess) return e;
    if ((e = allow_rows<kQ6_KRun, false, 4, 2>()) != hipSuccess) return e;
    return allow_rows<kQ6_KRun, true, 4, 2>();
}

template <int T>
hipError_t allow_rows_all() {
    hipError_t e;
    if ((e = allow_rows<T, false, 8, 2>()) != hipSuccess) return e;
    if ((e = allow_rows<T, false, 4, 1>()) != hipSuccess) return e;
    if ((e = allow_rows<T, false, 4, 2>()) != hipSuccess) return e;
    if ((e = allow_rows<T, true, 4, 1>()) != hipSuccess) return e;
    return allow_rows<T, true, 4, 2>();
}

} // namespace

// Every matrix of a block type (Q4_K, Q5_K, Q6_K, Q8_0), each its own type (GemvSeg::type, row_bytes filled in by the caller).
hipError_t gemv_mfma_mixed_launch(GemvArgs a, int cu_count, hipStream_t stream) {
    drop_stale_error();
    int max_out = 0;
    for (int i = 0; i < a.n_seg; ++i) max_out = max(max_out, a.seg[i].n_out);
    const int cap = a.mfma_wgs_per_cu > 0 ? cu_count * a.mfma_wgs_per_cu : (max_out + 15) / 16;
    const dim3 grid(min((max_out + 15) / 16, cap), a.n_seg);
    a.n_seg_types = 1;
    bool rows = rows_enabled();
    for (int i = 0; i < a.n_seg; ++i) rows = rows && a.seg[i].n_out % 16 == 0 && a.seg[i].type != kQ8_0;
    if (rows) {
        const int per_cu = rows_wgs_per_cu(a.mfma_wgs_per_cu, 3), nb = a.n_in / 256;
        const int tiles = rows_tiles(a);
        const int wgs = per_cu > 0 ? min(tiles, cu_count * per_cu) : tiles;
        const bool wide_r = nb > 8 && wgs == tiles; // (as in launch() above)
        RowsHead h;
        if (rows_head(a, wgs, 1, 1, h)) {
            h.shape &= ~0x3ff80u;
            const bool two = wide_r || nb > 4; // blocks an item
            for (int i = 0; i < a.n_seg; ++i) {
                const bool runs = a.seg[i].type == kQ6_K && two && nb % 2 == 0 && rows_run_base_ok(a.seg[i].w);
                h.shape |= rows_type_code(runs ? kQ6_KRun : a.seg[i].type) << (7 + 2 * i);
            }
            auto go = [&](auto waves, auto blocks) {
                constexpr int W = decltype(waves)::value, CB = decltype(blocks)::value;
                // (the largest of the types' layouts: Q6_K's digits in groups of 16, Q5_K's 11 pieces a block are within Q6_K's 14)
                const size_t lds = RowsGeom<kQ6_K, CB>::lds_bytes(a.n_in, W);
                if (lds > kMfmaLdsMax) return false;
                const dim3 gr(h.shape >> 18), block(W * 64);
                if constexpr (W == 4) {
                    if (nb <= W * CB && wgs == tiles && rows_norm_first(a, wgs)) {
                        hipLaunchKernelGGL((gemv_rows_mixed_kernel<W, CB, kRowsOneItemNorm>), gr, block, lds, stream, ROWS_HEAD_OF(h), a);
                        return true;
                    }
                }
                if (nb <= W * CB && wgs == tiles) hipLaunchKernelGGL((gemv_rows_mixed_kernel<W, CB, kRowsOneItem>), gr, block, lds, stream, ROWS_HEAD_OF(h), a);
                else hipLaunchKernelGGL((gemv_rows_mixed_kernel<W, CB, kRowsAny>), gr, block, lds, stream, ROWS_HEAD_OF(h), a);
                return true;
            };
            using One = std::integral_constant<int, 1>;
            using Two = std::integral_constant<int, 2>;
            const bool done = wide_r ? go(std::integral_constant<int, 8>(), Two())
                                     : (!two ? go(std::integral_constant<int, 4>(), One()) : go(std::integral_constant<int, 4>(), Two()));
            if (done) return hipGetLastError();
        }
    }
    const size_t lds = max(lds_bytes<kQ4_K>(a.n_in), lds_bytes<kQ6_K>(a.n_in));
    const bool wide = a.n_in / 256 >= 16 && (int)grid.x == (max_out + 15) / 16; // (as in launch() above)
    if (wide) hipLaunchKernelGGL((gemv_mfma_mixed_kernel<8>), grid, dim3(512), lds, stream, a);
    else hipLaunchKernelGGL((gemv_mfma_mixed_kernel<4>), grid, dim3(256), lds, stream, a);
    return hipGetLastError();
}

bool gemv_mfma_ok(int type, const GemvArgs& a) {
    if (a.n_in % 256 != 0) return false;
    if (type == kQ4_K || type == kQ5_K || type == kQ8_0) return lds_bytes<kQ4_K>(a.n_in) <= kMfmaLdsMax;
    if (type == kQ6_K) return lds_bytes<kQ6_K>(a.n_in) <= kMfmaLdsMax;
    return false;
}

hipError_t gemv_mfma_launch(int type, const GemvArgs& a, int cu_count, hipStream_t stream) {
    drop_stale_error();
    switch (type) {
    case kQ4_K: return launch<kQ4_K>(a, cu_count, stream);
    case kQ5_K: return launch<kQ5_K>(a, cu_count, stream);
    case kQ6_K: return launch<kQ6_K>(a, cu_count, stream);
    case kQ8_0: return launch<kQ8_0>(a, cu_count, stream);
    default: return hipErrorInvalidValue;
    }
}

// More than 64 KB of LDS per workgroup (rows longer than about 16k elements) needs to be allowed once.
hipError_t gemv_mfma_allow_lds() {
    hipError_t e;
    if ((e = allow<kQ4_K, false>()) != hipSuccess) return e;
    if ((e = allow<kQ4_K, true>()) != hipSuccess) return e;
    if ((e = allow<kQ6_K, false>()) != hipSuccess) return e;
    if ((e = allow<kQ6_K, true>()) != hipSuccess) return e;
    if ((e = allow<kQ5_K, false>()) != hipSuccess) return e;
    if ((e = allow<kQ5_K, true>()) != hipSuccess) return e;
    if ((e = allow<kQ8_0, false>()) != hipSuccess) return e;
    if ((e = allow<kQ8_0, true>()) != hipSuccess) return e;
    if ((e = allow_rows_all<kQ4_K>()) != hipSuccess) return e;
    if ((e = allow_rows_all<kQ5_K>()) != hipSuccess) return e;
    if ((e = allow_rows_all<kQ6_K>()) != hipSuccess) return e;
    if ((e = allow_rows_runs()) != hipSuccess) return e;
    if ((e = allow_rows<kQ8_0, false, 8, 1>()) != hipSuccess) return e;
    if ((e = allow_rows<kQ8_0, false, 8, 2>()) != hipSuccess) return e;
    if ((e = allow_rows<kQ8_0, false, 4, 2>()) != hipSuccess) return e;
    if ((e = allow_rows<kQ8_0, false, 4, 1>()) != hipSuccess) return e;
    if ((e = allow_rows<kQ8_0, true, 4, 1>()) != hipSuccess) return e;
    if ((e = allow_mixed<8, 2>()) != hipSuccess) return e;
    if ((e = allow_mixed<4, 1>()) != hipSuccess) return e;
    if ((e = allow_mixed<4, 2>()) != hipSuccess) return e;
    if ((e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemv_mfma_mixed_kernel<8>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMfmaLdsMax)) != hipSuccess) return e;
    return hipFuncSetAttribute(reinterpret_cast<const void*>(&gemv_mfma_mixed_kernel<4>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMfmaLdsMax);
}

hipError_t gemv_stamps(long long* host, size_t n) {
#ifdef ORIN_FA_STAMPS
    if (n > (size_t)kStampWgs * 4 * kStampSlots) return hipErrorInvalidValue;
    hipError_t e = hipMemcpyFromSymbol(host, HIP_SYMBOL(g_gemv_stamps), n * sizeof(long long)); // (synchronises with the device)
    void* dev = nullptr;
    if (e == hipSuccess) e = hipGetSymbolAddress(&dev, HIP_SYMBOL(g_gemv_stamps));
    if (e == hipSuccess) e = hipMemset(dev, 0, sizeof(g_gemv_stamps)); // the next launch starts from an empty table
    return e;
#else
    (void)host; (void)n;
    return hipErrorNotSupported;
#endif
}

} // namespace orin_fa
