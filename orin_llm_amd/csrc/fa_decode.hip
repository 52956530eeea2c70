// Single-token GQA attention over the fp16 KV cache for gfx950 (MI355X): a split-KV kernel
// spread over every CU plus a log-sum-exp combine kernel.
//
// Replaces the reference's flash_attention_decode_mma_k and its launcher (reference:
// src/kernels.cu:1105-1345, 1983-2000), which runs one block per KV head.
//
//   * The visible cache rows [0, *d_pos] of one KV head are cut into 32-row tiles.  Workgroup
//     (KV head, split s) is 8 wave64s; wave w takes tile s*8 + w and then every
//     (8 * n_splits)-th tile after it (runs shorter than 8 at a short position in a long cache,
//     see the kernel), so at 32k context each wave streams one or two tiles and
//     every byte of K and V is fetched exactly once, by 128-bit loads with the non-temporal hint.
//   * K rows go straight from memory into MFMA A-operand order (lane (col, grp) takes row col,
//     bytes (kk*4 + grp)*16): the score product needs no LDS round trip.  V rows are loaded
//     coalesced, parked in the wave's LDS slice and read back transposed (ds_read_b64_tr_b16).
//   * All query heads of the KV head's group (up to 16 per workgroup) are the 16 columns of
//     S^T = K Q^T and O^T = V^T P on v_mfma_f32_16x16x32_f16, so the group shares one pass
//     over K and V.  The matrix pipe is idle most of the time here, so Q and P are carried as
//     fp16 hi + lo pairs and the result is accurate to fp32 rounding.
//   * The position is read on the device; the launch shape depends only on by-value arguments,
//     so the launch can be captured in a graph and replayed after the position changes.  The
//     position and the query heads are requested together, first thing; a split that the
//     position leaves without a tile exits without having touched the cache (at a short
//     position in a long cache that is nearly all of them), and so does a wave without one, on its
//     way to the merge.  Tiles are fetched whole: rows at
//     or past the position are masked (K) or zeroed on their way into LDS (V).
//   * Partials (reference maximum, row sum, O) of the 8 waves are merged through LDS and
//     written per split; the combine kernel merges the splits that were active.
#include "fa_common.hpp"

#include <string.h>

#include <type_traits>

// Stage marks: wall-clock stamps in the timeline build, nothing otherwise (fa_common.hpp).
#ifdef ORIN_FA_STAMPS
namespace orin_fa {
__device__ long long g_decode_stamps[kStampWgs * kDecodeWaves * kStampSlots];
}
#define FA_STAMP(i) ORIN_FA_STAMP_STORE(orin_fa::g_decode_stamps, orin_fa::kDecodeWaves, i)
#else
#define FA_STAMP(i)
#endif

// Cut-off builds (-DORIN_FA_DECODE_PROBE=flags, liborin_fa_probe_<flags>.so; measurement aids whose RESULTS ARE
// WRONG by design): the split kernel with parts taken out, so that bench.py's cut-off workload can say
// what each part costs.  1: no combine launch.  2: the kernel leaves once its first tile has arrived
// (no products, no merge, no partial).  4: the position is n_ctx - 1, not read from memory.
// 8: no query loads.  16: K fetched whole lines at a time like V (its contents then in the wrong
// lanes).  0 in the library proper, where none of this exists.
#ifndef ORIN_FA_DECODE_PROBE
#define ORIN_FA_DECODE_PROBE 0
#endif

namespace orin_fa {
namespace {
constexpr int kProbe = ORIN_FA_DECODE_PROBE;
constexpr bool kProbeNoCombine = (kProbe & 1) != 0, kProbeCutOff = (kProbe & 2) != 0, kProbeConstPos = (kProbe & 4) != 0,
               kProbeNoQuery = (kProbe & 8) != 0, kProbeKWholeLines = (kProbe & 16) != 0;

template <int D>
struct DGeom {
    static constexpr int kSteps = D / 32;                      // MFMA k-steps over head_dim
    static constexpr int kDBlk = D / 16;                       // 16-wide output blocks over head_dim
    static constexpr int kRowBV = D * 2 + 32;                  // bytes per V row in LDS (32 B pad spreads the transposing reads)
    static constexpr int kChunksPerRow = D / 8;                // 16-byte chunks per KV row
    static constexpr int kLoads = kTile * kChunksPerRow / 64;  // 16-byte V loads per lane per tile
    static constexpr int kTileBV = kTile * kRowBV;             // one V tile in LDS
    static constexpr int kOStride = D + 4;                     // floats per column in the merge buffer
    static constexpr int kMergeB = 16 * kOStride * 4;
    static constexpr int kWaveB = (kTileBV > kMergeB) ? kTileBV : kMergeB;
    static constexpr int kMlOff = kDecodeWaves * kWaveB;       // (m, l) per wave per column follow the wave slices
    // The group's query heads: two planes of operands, the fp16 values and what rounding to them left off, [16][kQPlaneB / 16]; or
    // (angles that come late) fp32 [16][kQStride].  Padded so that the operand reads of 16 heads miss each other's banks.
    static constexpr int kQOff = kMlOff + kDecodeWaves * 16 * 2 * 4;
    static constexpr int kQRowB = D * 2 + 16, kQPlaneB = 16 * kQRowB;
    static constexpr int kQStride = D + 4;
    static constexpr int kLdsB = kQOff + 2 * kQPlaneB;
    static_assert(2 * kQPlaneB >= 16 * kQStride * 4, "either form");
};

// 16 bytes a lane through a descriptor (base, byte count): zeros, and no access, at kNowhere.
constexpr int kNowhere = 0x7ffffff8;
__device__ __forceinline__ f4 load16(const float* base, unsigned bytes, int off) {
    return __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(make_rsrc(base, bytes), off, 0, 0));
}
// What a launch does besides attending (see the kernel).
enum : int { kPlain = 0, kStore = 1, kRotate = 2, kRotateNeox = 3, kRotateLate = 4 };

// kStore: the current token's K and V rows arrive as fp32 beside the cache (FaArgs::k_new, v_new).  The workgroup whose tiles
// include row *d_pos takes that row from them -- rounded to fp16 exactly as the store kernel rounds -- instead of from the
// cache, and writes it to the cache on the way: the store kernel's launch is saved and the result is the same bit for bit.
// kRotate, kRotateNeox (rotate + store): q and k_new arrive before the rotary embedding, and the workgroups rotate them (the
// inputs stay as they are) by the caller's table of angles: "normal" pairs are neighbours, "neox" pairs half a head
// apart.  Same arithmetic as the rotary kernel, so again bit for bit what the separate launches give, two launches
// in the place of seven.  A rotation that does not span the whole head, or has no table, is kRotateLate's: every
// wave keeps a table in LDS (a power, a sine and a cosine a pair, which must not sit ahead of the tile requests) and rotates the whole
// query behind the workgroup's meeting, and the new row is made ready by the wave whose last tile holds it.
//
// A launch is a chain -- position and query, tile, products, merge -- in which a wave issues an instruction every 2 ns, so what
// can be done once is done once, and off the way from a tile's arrival to the result:
//   * each wave makes operands of the piece of the query it has fetched (rotates it, splits it into the two fp16 parts) ahead of
//     the tile requests, and the pieces meet in LDS as operands.  (Every wave used to convert, and for "neox" rotate, the whole query.)
//   * the new row is made ready by a wave without a tile, while the owner's tile travels, or ahead of the meeting where all have one.  (The
//     owner used to, which took longer than its tile: products 1.1 us after its requests instead of 0.6.)
//   * a run of one tile (a position short of a tile a split) goes from registers to the result, without the merge through LDS; a
//     wave's first tile rescales nothing; rows past the position are voided in the last tile only; and the tile with another behind it is code
//     of its own, so that every wait is for what is used next.
// Rotate + store + attend, us a launch pair, caches emptied between replays, before -> now: Qwen2.5-1.5B at 200 of 4096 7.6 -> 6.5, at 4095 7.9 ->
// 7.0, at 32767 of 32768 11.7 -> 11.2; Llama-3-8B at 1000 of 8192 7.75 -> 6.8, at 8191 11.5 -> 11.1; Qwen2.5-7B at 16001 of 32768 12.3 ->
// 11.2; Llama-3.2-1B at 1777 of 8192 7.1 -> 6.6.  Plain decode 6.2 -> 6.05, 6.75 -> 6.6, the same within 2 % at 32767, 6.7 -> 6.5, 11.3 -> 11.25, 11.25 ->
// 11.15, 6.3 -> 6.2.  Without a table (every layer with rows of its own) 6.9 -> 6.5, 7.6 -> 7.3, 11.5 -> 11.35; "normal" pairs 7.55 -> 6.8,
// 11.75 -> 11.3; 12.0 -> 11.75; 6.7 -> 6.25.
template <int D, int MODE>
__global__ __launch_bounds__(kDecodeWaves * 64) void fa_decode_split_kernel(
    // What the first loads need comes first, as scalars: the leading kernel arguments are handed
    // to a wave in registers when it starts (kernel-argument preload), so the position and the
    // query can be requested at once instead of behind a trip to memory for their addresses.
    // (no __restrict__ on these: loads the compiler knows to be invariant are free to sink past
    // the statements below that hold them in place)
    // Plain decode needs nothing but these 14 words: no trip to the launch's argument block at
    // all, which is slower than the trip for the position (the caches hold that).  So: the grid
    // is (KV head, head group, split) and says what n_kv and n_hgroups would; n_splits, r and the sign that goes into Q share
    // a word (splits_r = n_splits | negative scale << 15 | r << 16); scale_heads = |scale| log2(e) as its bits | n_head << 32, or,
    // with a table of angles, the table's address (those two then come from the argument block, being needed last); dst is where
    // this kernel writes: the partial outputs (followed by the (m, l) pairs) when there are splits, else `out` itself.
    const int* d_pos, const float* q, const uint16_t* kc, const uint16_t* vc,
    const int n_ctx, const unsigned splits_r, const uint64_t scale_heads, float* dst,
    const FaArgs a) { // (a: what the store and rotate variants need besides)
    using G = DGeom<D>;
    constexpr int kWaves = kDecodeWaves;
    constexpr int kThreads = kWaves * 64;
    constexpr bool STORE = MODE != kPlain, TABLE = MODE == kRotate || MODE == kRotateNeox, NEOX = MODE == kRotateNeox, LATE = MODE == kRotateLate;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    FA_STAMP(0);

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15; // MFMA column (query head of the group) / row (KV row or head_dim index) of the lane
    const int grp = lane >> 4; // lane-group: 8-wide k slice of an operand, 4-row slice of an accumulator

    const int n_splits = splits_r & 0x7fffu, r = splits_r >> 16;
    const float qsign = (splits_r & 0x8000u) != 0 ? -1.0f : 1.0f;
    // Workgroup -> (KV head, head group, split); the KV head varies fastest in dispatch order.
    const int kvh = blockIdx.x, hg = blockIdx.y, id = blockIdx.z;

    unsigned char* const vs = smem + wave * G::kWaveB;

    const uint16_t *const k_head = kc + (size_t)kvh * n_ctx * D, *const v_head = vc + (size_t)kvh * n_ctx * D;
    const int k_lane = col * D * 2 + grp * 16, v_lane = lane * 16; // where a lane's first pieces lie in a tile

    u32x4 kreg[2 * G::kSteps], vreg[G::kLoads];
    auto fetch_k = [&](int tile) {
        const __amdgpu_buffer_rsrc_t krs = make_rsrc(k_head, (unsigned)n_ctx * D * 2);
        const int at = tile * kTile * D * 2 + (kProbeKWholeLines ? lane * 16 : k_lane);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int kk = 0; kk < G::kSteps; ++kk)
                kreg[t * G::kSteps + kk] = buf_load16<true>(krs, at + (kProbeKWholeLines ? (t * G::kSteps + kk) * 1024 : t * 16 * D * 2 + kk * 64));
    };
    auto fetch_v = [&](int tile) {
        const __amdgpu_buffer_rsrc_t vrs = make_rsrc(v_head, (unsigned)n_ctx * D * 2);
        const int at = tile * kTile * D * 2 + v_lane;
#pragma unroll
        for (int i = 0; i < G::kLoads; ++i) vreg[i] = buf_load16<true>(vrs, at + i * 1024);
    };
    // ---- query heads: requested before the first tile, so that they arrive before it (a wave's
    // loads complete in order) and the score product can start while V is still on its way ----
    const int pos = kProbeConstPos ? n_ctx - 1 - (d_pos == nullptr) : *d_pos; // (read here, ahead of the statement below that may write memory: a scalar load)
    // Columns past the group's heads are padding: their loads carry an offset past the descriptor's
    // end, which the hardware answers with zeros without going to memory.
    // The workgroup fetches its group's heads once, a piece of four elements per lane, neighbouring lanes on one head; the pieces
    // meet in LDS further down.  (Every wave fetching all of them itself was seven more load instructions a wave whose lanes each count
    // as a look-up of their own in the vector cache, a quarter again of the kernel's look-ups, all
    // of them in the queue ahead of the tile requests: 0.4 us per launch.)
    constexpr int kHeadLanes = D / 4;
    const int my_head = wave * (64 / kHeadLanes) + lane / kHeadLanes, e0 = (lane % kHeadLanes) * 4; // (head_dim 64: the first four waves have all sixteen)
    [[maybe_unused]] f4 q_share, cs[2];
    if constexpr (!LATE) {
        const bool valid = my_head < 16 && hg * 16 + my_head < r;
        q_share = kProbeNoQuery ? f4{1.0f, 2.0f, (float)lane, 3.0f} : load16(q, 0x7ffffff0u, valid ? ((kvh * r + hg * 16 + my_head) * D + e0) * 4 : kNowhere);
    }
    // (table of angles) The piece's (cos, sin): two pairs, or four, of which it holds one half; the new K row's pieces have the same.
    const float* const angles = ptr_arg<const float>(TABLE ? scale_heads : 0);
    if constexpr (TABLE) {
        const int at = (NEOX ? e0 & (D / 2 - 1) : e0 / 2) * 8;
        cs[0] = load16(angles, D * 4, at);
        if constexpr (NEOX) cs[1] = load16(angles, D * 4, at + 16);
    }
    // (kRotateLate) The same by pieces of operands: wave w asks for piece (w & 1) of k-step (w >> 1) of every head.
    const int hl = hg * 16 + col;
    const bool valid = hl < r;
    const int q_off = valid ? ((kvh * r + hl) * D + grp * 8) * 4 : kNowhere;
    static_assert(kWaves % (2 * G::kSteps) == 0, "a piece per wave (the same piece twice at head_dim 64)");
    const int q_piece = __builtin_amdgcn_readfirstlane(wave) & (2 * G::kSteps - 1);
    const int q_e0 = (q_piece >> 1) * 32 + grp * 8 + (q_piece & 1) * 4; // the piece's first element of its head
    float4 q_late = float4{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (LATE)
        q_late = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(make_rsrc(q, 0x7ffffff0u), q_off, (q_piece >> 1) * 128 + (q_piece & 1) * 16, 0));
    // (kRotateLate) lane i < n_rot/2 of every wave fetches what pair i's angle needs: its
    // cosine and sine when the caller supplies them, else its frequency factor if there is one.
    // Both loads are made by every lane, from an address that can be read either way (the query,
    // when the array is absent): a load under a branch makes the compiler wait for every load
    // issued so far where the branch ends.
    float2 cs_given = float2{1.0f, 0.0f};
    float ff_given = 1.0f;
    if constexpr (LATE) {
        const int pi = min(lane, a.n_rot / 2 - 1);
        const float* anp = a.rope_angles ? a.rope_angles + 2 * pi : q;
        const float* ffp = a.freq_factors ? a.freq_factors + pi : q;
        cs_given = *reinterpret_cast<const float2*>(anp);
        ff_given = *ffp;
    }
    // (store, rotate + store) The new row, in as few loads as will do: which workgroup owns it depends on the position, which
    // is still on its way, and a load issued later, while the CU's tiles stream in, holds its wave up for a few
    // hundred cycles each.  For the last wave, which makes the row ready (kRotateLate: for every wave); the others' loads go nowhere (under
    // a branch, the last wave would wait for the row where it waits for its share of the query).  K: the lane's piece, as of
    // the query; V: piece lane % (D/8), eight elements.
    constexpr int kRowWave = kWaves - 1;
    [[maybe_unused]] f4 k_raw, v_raw[2];
    if constexpr (STORE) {
        const float *const kp = a.k_new + (size_t)kvh * D, *const vp = a.v_new + (size_t)kvh * D;
        const int v_e0 = (lane % G::kChunksPerRow) * 8;
        const bool mine = LATE || wave == kRowWave;
        k_raw = load16(kp, D * 4, mine ? e0 * 4 : kNowhere);
        v_raw[0] = load16(vp, D * 4, mine ? v_e0 * 4 : kNowhere);
        v_raw[1] = load16(vp, D * 4, mine ? v_e0 * 4 + 16 : kNowhere);
    }
    __builtin_amdgcn_sched_barrier(0); // the small loads first: they return first, and nothing that needs them waits for a tile

    // The query loads above are used only behind the early return below, and left alone the
    // compiler moves them there, behind the wait for the position.  A statement that may write
    // memory keeps them on this side of the branch, where they overlap the load of the position.
    // The first tile is NOT requested here: a workgroup that turns out to be inactive would pull
    // 128 KB of cache rows for nothing -- at a short position in a long cache, all of them but a
    // few, tens of megabytes per launch that the active ones then queue behind.
    asm volatile("" ::: "memory");
    // (store and rotate variants) The arguments that did not arrive in registers are fetched
    // here, in the trip to memory that brings the position: left alone, the compiler fetches
    // each where it is first used, behind the first tile's arrival.  (Fetched behind the tile
    // requests instead, they queue behind the chip's 33 MB of tile traffic: 0.5 us per layer.)
    const float c2 = TABLE ? a.c : __uint_as_float((unsigned)scale_heads);
    const int n_head = TABLE ? a.n_head : (int)(scale_heads >> 32);
    if constexpr (MODE != kPlain) {
        const void *p0 = a.k_new, *p1 = a.v_new;
        asm volatile("" ::"s"(p0), "s"(p1), "s"(a.n_rot), "s"(a.neox), "s"(c2), "s"(n_head), "s"(pos));
    }
    __builtin_amdgcn_sched_barrier(0);
    float* const part_o = dst;
    float* const part_ml = dst + (size_t)n_splits * n_head * D; // [n_head][split][2]

    int p = pos < 0 ? 0 : pos;
    const int npos = (p > n_ctx - 1 ? n_ctx - 1 : p) + 1; // rows [0, npos) are visible
    const bool store = STORE && pos >= 0 && pos < n_ctx;   // (a position outside the cache stores nothing, as the store kernel)
    const int n_tiles = (npos + kTile - 1) / kTile;
    // Tiles go to the splits in runs of `wu` consecutive tiles, one per wave: eight when there are
    // enough tiles to keep every wave of every split busy (runs of 128 KB of K and of V), fewer
    // at a short position in a long cache, whose few tiles then spread over as many workgroups
    // (CUs, each with its own 64 B/clk into the vector cache) as there are instead of filling a
    // few workgroups' eight waves.  (Interleaving single tiles among the splits at every length
    // cost 8 % at full length on Qwen2.5-7B: neighbouring 8 KB pieces then alternate between XCDs.)
    int wu = 0; // = min(ceil(n_tiles / n_splits), 8), by halves: a division is three times as long, and the tile requests wait for it
    static_assert(kWaves == 8, "three halves");
#pragma unroll
    for (int h = 4; h > 0; h >>= 1) wu += n_tiles > (wu + h) * n_splits ? h : 0;
    ++wu;
    const int tile_first = wave < wu ? id * wu + wave : n_tiles; // (n_tiles: none)
    const int tile_step = wu * n_splits;
    int tile = tile_first;
    const int own_tile = n_tiles - 1; // the new row's
    if (id * wu >= n_tiles) {
        // Inactive split: it leaves "no row seen" for its heads, so that the combine kernel can tell
        // without reading the position itself (one more trip to memory on its short critical path);
        // the partial outputs are left as they are and get weight zero.
        if (threadIdx.x < 16 && hg * 16 + (int)threadIdx.x < r) {
            const size_t mi = (size_t)(kvh * r + hg * 16 + threadIdx.x) * n_splits + id; // [head][split]
            part_ml[mi * 2 + 0] = -INFINITY;
            part_ml[mi * 2 + 1] = 0.0f;
        }
        return;
    }
    float* const qs = reinterpret_cast<float*>(smem + G::kQOff);
    __shared__ __attribute__((aligned(16))) float sh_cs_all[LATE ? kWaves : 1][D / 2][2];
    __shared__ __attribute__((aligned(16))) _Float16 sh_krow_all[LATE ? kWaves : 1][D];
    __shared__ __attribute__((aligned(16))) _Float16 sh_vrow[STORE && !LATE ? D : 8];
    __shared__ int sh_row_there;
    // (said to be LDS: a generic pointer's accesses count as memory's too, and every wait behind one is for everything)
    [[maybe_unused]] auto* const row_there = (__attribute__((address_space(3))) volatile int*)&sh_row_there;
    float (*const sh_cs)[2] = sh_cs_all[LATE ? wave : 0];
    const bool rot_early = LATE && !a.neox && a.rope_angles != nullptr; // (the query is rotated piece by piece before it is parked)
    // A piece of the query or of the new K row, rotated.
    [[maybe_unused]] auto rotate4 = [&](f4 x) {
        if constexpr (NEOX) { // element e goes with e + D/2: the lane's piece is the first or the second of the pair, the other one 16 (8) lanes away
            const bool second = e0 >= D / 2;
            f4 y;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float lo, hi;
                if constexpr (D == 128) { // both halves of the pair land in both lanes
                    const u32x2 s = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[e]), __float_as_uint(x[e]), false, false);
                    lo = __uint_as_float(s.x);
                    hi = __uint_as_float(s.y);
                } else {
                    const int b = __float_as_int(x[e]);
                    const float other = __int_as_float(__builtin_amdgcn_update_dpp(b, b, 0x128, 0xF, 0xF, false)); // row_ror:8
                    lo = second ? other : x[e];
                    hi = second ? x[e] : other;
                }
                rope_rotate(lo, hi, cs[e / 2][e % 2 * 2], cs[e / 2][e % 2 * 2 + 1]);
                y[e] = second ? hi : lo;
            }
            return y;
        } else if constexpr (TABLE) {
            float x0 = x[0], x1 = x[1], x2 = x[2], x3 = x[3];
            rope_rotate(x0, x1, cs[0][0], cs[0][1]);
            rope_rotate(x2, x3, cs[0][2], cs[0][3]);
            return f4{x0, x1, x2, x3};
        } else {
            return x;
        }
    };
    // The query pieces meet in LDS: each wave parks the piece it fetched, then a barrier that
    // waits for LDS only.  Ahead of the tile requests, where the eight waves are still in
    // step (the position and the pieces arrive together); behind them the waves are microseconds
    // apart -- the load unit takes a CU's 128 KB of requests as fast as memory answers them --
    // and a barrier there holds every wave's products until the last has all its requests out.
    if constexpr (LATE) {
        float4 q_park = q_late;
        // "Normal" pairs are neighbours, so the piece a wave fetched holds two whole pairs: with the caller's
        // table of angles at hand the wave rotates just those before it parks the piece.  (Without a table the angles are a power,
        // a sine and a cosine away.)
        if (rot_early) {
            if (lane < a.n_rot / 2) {
                sh_cs[lane][0] = cs_given.x;
                sh_cs[lane][1] = cs_given.y;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const int e0 = q_e0, last = max(a.n_rot / 2 - 1, 0);
            const float2 c0 = *reinterpret_cast<const float2*>(sh_cs[min(e0 / 2, last)]);
            const float2 c1 = *reinterpret_cast<const float2*>(sh_cs[min(e0 / 2 + 1, last)]);
            float x0 = q_park.x, x1 = q_park.y, y0 = q_park.z, y1 = q_park.w;
            rope_rotate(x0, x1, c0.x, c0.y);
            rope_rotate(y0, y1, c1.x, c1.y);
            q_park.x = e0 < a.n_rot ? x0 : q_park.x;
            q_park.y = e0 < a.n_rot ? x1 : q_park.y;
            q_park.z = e0 + 2 < a.n_rot ? y0 : q_park.z;
            q_park.w = e0 + 2 < a.n_rot ? y1 : q_park.w;
        }
        *reinterpret_cast<float4*>(qs + col * G::kQStride + q_e0) = q_park;
    } else {
        // The piece as operands: rotated, then its fp16 value and what that leaves off.
        const f4 x = rotate4(q_share);
        h4 hi, lo;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float xe = x[e] * qsign;
            hi[e] = (_Float16)xe;
            lo[e] = (_Float16)(xe - (float)hi[e]);
        }
        if (my_head < 16) {
            unsigned char* const park = smem + G::kQOff + my_head * G::kQRowB + e0 * 2;
            *reinterpret_cast<h4*>(park) = hi;
            *reinterpret_cast<h4*>(park + G::kQPlaneB) = lo;
        }
    }
    [[maybe_unused]] int own_wave = -1; // the wave of this workgroup whose tiles include the new row's, if any (not kRotateLate)
    [[maybe_unused]] auto make_row = [&] {
        // The new row: rotated and converted as the rotary kernel and the store kernel would, into LDS for the wave that
        // owns it, which takes it instead of what its tile brings back, and into the cache (no other wave reads that row, so
        // the order of this write and that read does not matter; one head group's workgroup writes it).
        const f4 k = rotate4(k_raw);
        h4 kh;
#pragma unroll
        for (int e = 0; e < 4; ++e) kh[e] = (_Float16)k[e];
        h8 vh;
#pragma unroll
        for (int e = 0; e < 8; ++e) vh[e] = (_Float16)v_raw[e / 4][e % 4];
        if (lane < kHeadLanes) *reinterpret_cast<h4*>(sh_krow_all[0] + e0) = kh;
        if (lane < G::kChunksPerRow) *reinterpret_cast<h8*>(sh_vrow + lane * 8) = vh;
        // (a wave's LDS writes are made in order: who sees the flag sees the row)
        asm volatile("" ::: "memory");
        *row_there = 1;
        if (hg == 0) {
            const size_t row_off = ((size_t)kvh * n_ctx + pos) * D;
            if (lane < kHeadLanes) *reinterpret_cast<h4*>(const_cast<uint16_t*>(kc) + row_off + e0) = kh;
            if (lane < G::kChunksPerRow) *reinterpret_cast<h8*>(const_cast<uint16_t*>(vc) + row_off + lane * 8) = vh;
        }
    };
    if constexpr (STORE && !LATE) {
        int last = own_tile; // where the last visible tile lies in a turn of all splits (a few turns at most)
        while (last >= tile_step) last -= tile_step;
        own_wave = store && last - id * wu < wu ? last - id * wu : -1; // (negative: another split's)
        // By the last wave: behind the meeting where it has no tile of its own, while the owner's tile is on its way (the owner waits for the
        // flag), and ahead of it where it has.
        if (wave == kRowWave) {
            if (own_wave >= 0 && wu == kWaves) make_row();
            else *row_there = 0;
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if constexpr (STORE && !LATE)
        if (wave == kRowWave && own_wave >= 0 && wu < kWaves) make_row();

    // m_ref: reference maximum of the raw scores (before the scale); l_run: this lane's share of
    // the row sum; o: O^T accumulators, lane (col, grp) holds head_dim rows db*16 + grp*4 + i.
    float m_ref = -INFINITY, l_run = 0.0f;
    f4 o[G::kDBlk];
#pragma unroll
    for (int db = 0; db < G::kDBlk; ++db) o[db] = f4{0.f, 0.f, 0.f, 0.f};
    // A wave without a tile (most, at a short position) goes straight to the merge.  (Asking for some tile all the same, so as
    // to keep loads out of branches, seven such waves kept their CU's load unit busy for 1.2 us ahead of the eighth's
    // values: Qwen2.5-1.5B at position 200 of 4096 6.7 -> 5.9 us a launch pair, Qwen2.5-7B at 2000 of 32768 8.0 -> 6.7.)
    if (tile < n_tiles) {
        fetch_k(tile);
        fetch_v(tile);
        asm volatile("" ::: "memory"); // (as above: ahead of the conversions that follow, not behind them)
        __builtin_amdgcn_sched_barrier(0);
        FA_STAMP(1);
        if constexpr (kProbeCutOff) { // (cut-off build: wait for the tile, keep every load alive, leave)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            unsigned acc = LATE ? __float_as_uint(q_late.x) ^ __float_as_uint(q_late.w) : __float_as_uint(q_share[0]) ^ __float_as_uint(q_share[3]);
#pragma unroll
            for (int i = 0; i < 2 * G::kSteps; ++i) acc ^= kreg[i].x ^ kreg[i].y ^ kreg[i].z ^ kreg[i].w;
#pragma unroll
            for (int i = 0; i < G::kLoads; ++i) acc ^= vreg[i].x ^ vreg[i].y ^ vreg[i].z ^ vreg[i].w;
            if (acc == 0x9E3779B9u) part_ml[0] = 1.0f;
            if (acc != 0x9E3779BAu) return;
        }
        // (the query pieces met ahead of the tile requests; the operands are picked up while the first tile is on its way)
        h8 qhi[G::kSteps], qlo[G::kSteps];
        [[maybe_unused]] u32x4 k_new16[G::kSteps], v_new16 = u32x4{0u, 0u, 0u, 0u};
        [[maybe_unused]] bool owner = wave == own_wave; // (kRotateLate: further down)
        if constexpr (!LATE) {
            const unsigned char* const op = smem + G::kQOff + col * G::kQRowB + grp * 16;
#pragma unroll
            for (int kk = 0; kk < G::kSteps; ++kk) {
                qhi[kk] = *reinterpret_cast<const h8*>(op + kk * 64);
                qlo[kk] = *reinterpret_cast<const h8*>(op + kk * 64 + G::kQPlaneB);
            }
            if constexpr (STORE) {
                if (wave == own_wave) {
                    while (*row_there == 0) {} // (the last wave sets it, whatever the others do)
                    asm volatile("" ::: "memory");
#pragma unroll
                    for (int kk = 0; kk < G::kSteps; ++kk) k_new16[kk] = *reinterpret_cast<const u32x4*>(sh_krow_all[0] + (kk * 4 + grp) * 8);
                    v_new16 = *reinterpret_cast<const u32x4*>(sh_vrow + (lane % G::kChunksPerRow) * 8);
                }
            }
        } else {
            const float qmul = valid ? qsign : 0.0f;
            float qf[G::kSteps][8]; // this lane's 8 elements of every k-step: head_dim indices kk*32 + grp*8 + 0..7
#pragma unroll
            for (int kk = 0; kk < G::kSteps; ++kk) {
                const float4 x0 = *reinterpret_cast<const float4*>(qs + col * G::kQStride + kk * 32 + grp * 8);
                const float4 x1 = *reinterpret_cast<const float4*>(qs + col * G::kQStride + kk * 32 + grp * 8 + 4);
                qf[kk][0] = x0.x; qf[kk][1] = x0.y; qf[kk][2] = x0.z; qf[kk][3] = x0.w;
                qf[kk][4] = x1.x; qf[kk][5] = x1.y; qf[kk][6] = x1.z; qf[kk][7] = x1.w;
            }
            // (rotate + store) the rotation of this lane's 8 elements of every k-step, by the wave's table
            // x0, x1: this lane's elements of k-steps kk and kk + kSteps/2 (head_dim indices kk*32 + grp*8 + e
            // and the same + head_dim/2)
            auto rotate2 = [&](float (&x0)[8], float (&x1)[8], int kk) {
                if (a.neox) { // n_rot == D (checked by the host): element e pairs with e + D/2
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const int i = kk * 32 + grp * 8 + e;
                        rope_rotate(x0[e], x1[e], sh_cs[i][0], sh_cs[i][1]);
                    }
                } else {      // elements 2i and 2i + 1, below n_rot
                    // No branch per pair: el0 differs from lane to lane, and a branch around each pair's table
                    // read makes the wave wait out sixteen LDS round trips one after the other (1.7 us of a
                    // Llama-3-8B launch).  Every lane reads an entry (its own, or the table's last), all reads
                    // go out together, and a pair past n_rot keeps its values by a select.
                    const int last = max(a.n_rot / 2 - 1, 0); // (n_rot = 0: nothing is rotated, entry 0 is read and not used)
                    float2 cs0[4], cs1[4];
#pragma unroll
                    for (int e = 0; e < 8; e += 2) {
                        const int el0 = kk * 32 + grp * 8 + e, el1 = el0 + D / 2;
                        cs0[e / 2] = *reinterpret_cast<const float2*>(sh_cs[min(el0 / 2, last)]);
                        cs1[e / 2] = *reinterpret_cast<const float2*>(sh_cs[min(el1 / 2, last)]);
                    }
#pragma unroll
                    for (int e = 0; e < 8; e += 2) {
                        const int el0 = kk * 32 + grp * 8 + e, el1 = el0 + D / 2;
                        float a0 = x0[e], a1 = x0[e + 1], b0 = x1[e], b1 = x1[e + 1];
                        rope_rotate(a0, a1, cs0[e / 2].x, cs0[e / 2].y);
                        rope_rotate(b0, b1, cs1[e / 2].x, cs1[e / 2].y);
                        x0[e] = el0 < a.n_rot ? a0 : x0[e];
                        x0[e + 1] = el0 < a.n_rot ? a1 : x0[e + 1];
                        x1[e] = el1 < a.n_rot ? b0 : x1[e];
                        x1[e + 1] = el1 < a.n_rot ? b1 : x1[e + 1];
                    }
                }
            };
            // (cos, sin) of pair i at the raw position, as the rotary kernel forms them
            // A table per wave (head_dim <= 128: a wave's 64 lanes cover the pairs), so that no wave
            // waits here for the others: the waves of a workgroup get their loads out at very
            // different times when the whole chip is requesting its first tiles.  Write and reads
            // are the same wave's, and a wave's LDS operations complete in order.
            static_assert(D / 2 <= 64, "one lane per pair");
            const int half = a.n_rot / 2;
            if (!rot_early && lane < half) {
                if (!a.rope_angles) {
                    float freq = rope_freq_of(a.freq, lane);
                    if (a.freq_factors) freq /= ff_given;
                    const float ang = (float)pos * freq;
                    sincosf(ang, &cs_given.y, &cs_given.x);
                }
                sh_cs[lane][0] = cs_given.x;
                sh_cs[lane][1] = cs_given.y;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (!rot_early) {
#pragma unroll
                for (int kk = 0; kk < G::kSteps / 2; ++kk) rotate2(qf[kk], qf[kk + G::kSteps / 2], kk);
            }
            // ---- query heads -> B operands, fp16 hi + lo ----
#pragma unroll
            for (int kk = 0; kk < G::kSteps; ++kk) {
                const float* x = qf[kk];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float xe = x[e] * qmul;
                    qhi[kk][e] = (_Float16)xe;
                    qlo[kk][e] = (_Float16)(xe - (float)qhi[kk][e]);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        FA_STAMP(2);
        const int v_rd = (grp * 4 + (col >> 2)) * G::kRowBV + (col & 3) * 8; // + h*16 rows, + db*32 bytes

        // (kRotateLate) The new row is made ready here, while the tiles travel, by the one wave whose tiles
        // include the row's (the last visible tile: the wave's own last): converted -- and the K row rotated -- as the
        // store kernel and the rotary kernel would, the pieces this lane is to substitute and to write kept in
        // registers.  At that tile only the substitution and the two cache writes are left.  (Made ready at the tile
        // itself, as it used to be, the LDS round trips and the rotation sat between the arrival of the launch's last
        // tile and its products: 0.7 us of a Qwen2.5-1.5B launch pair at 32k.)  The row's loads went out ahead of the
        // tile requests, so waiting for them waits for no tile.
        if constexpr (LATE) {
#pragma unroll
            for (int kk = 0; kk < G::kSteps; ++kk) k_new16[kk] = u32x4{0u, 0u, 0u, 0u};
            int last = tile_first; // this wave's last tile (a few steps at most)
            while (last + tile_step <= own_tile) last += tile_step;
            owner = store && last == own_tile;
            if (owner) {
                // (Nothing below may be started ahead of this branch: the compiler would otherwise
                // convert the new row in every wave.)
                auto here = [](float x) { // a copy the compiler cannot make anywhere else
                    float y;
                    asm volatile("v_mov_b32 %0, %1" : "=v"(y) : "v"(x));
                    return y;
                };
                const float4 v_own[2] = {float4{here(v_raw[0].x), here(v_raw[0].y), here(v_raw[0].z), here(v_raw[0].w)},
                                         float4{here(v_raw[1].x), here(v_raw[1].y), here(v_raw[1].z), here(v_raw[1].w)}};
                {
                    // K: lane i (of D/4) holds elements 4 i ..: it rotates those -- a "neox" pair's other half is the lane's
                    // D/8 away -- and converts them, and the lanes pick the pieces they hold of a K row out of LDS.  (Every lane
                    // rotating the 32 elements it will hold was 250 instructions, 0.6 us of the launch whose last tile is
                    // this wave's.)
                    float x[4] = {here(k_raw.x), here(k_raw.y), here(k_raw.z), here(k_raw.w)};
                    {
                        const int e0 = (lane % (D / 4)) * 4;
                        if (a.neox) {
                            const bool second = e0 >= D / 2;
                            const int i0 = second ? e0 - D / 2 : e0;
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const float other = __shfl_xor(x[e], D / 8);
                                float lo = second ? other : x[e], hi = second ? x[e] : other;
                                rope_rotate(lo, hi, sh_cs[i0 + e][0], sh_cs[i0 + e][1]);
                                x[e] = second ? hi : lo;
                            }
                        } else {
                            const int last_pair = max(a.n_rot / 2 - 1, 0);
#pragma unroll
                            for (int e = 0; e < 4; e += 2) {
                                float lo = x[e], hi = x[e + 1];
                                const int i = min((e0 + e) / 2, last_pair);
                                rope_rotate(lo, hi, sh_cs[i][0], sh_cs[i][1]);
                                x[e] = e0 + e < a.n_rot ? lo : x[e];
                                x[e + 1] = e0 + e < a.n_rot ? hi : x[e + 1];
                            }
                        }
                    }
                    _Float16* const krow = sh_krow_all[wave];
                    h4 h;
#pragma unroll
                    for (int e = 0; e < 4; ++e) h[e] = (_Float16)x[e];
                    if (lane < D / 4) *reinterpret_cast<h4*>(krow + lane * 4) = h;
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
                    for (int kk = 0; kk < G::kSteps; ++kk) k_new16[kk] = *reinterpret_cast<const u32x4*>(krow + (kk * 4 + grp) * 8);
                }
                h8 vh;
                vh[0] = (_Float16)v_own[0].x; vh[1] = (_Float16)v_own[0].y; vh[2] = (_Float16)v_own[0].z; vh[3] = (_Float16)v_own[0].w;
                vh[4] = (_Float16)v_own[1].x; vh[5] = (_Float16)v_own[1].y; vh[6] = (_Float16)v_own[1].z; vh[7] = (_Float16)v_own[1].w;
                v_new16 = __builtin_bit_cast(u32x4, vh);
                // The cache gets the row now (one head group's wave writes it): whatever the tile request that is under
                // way brings back for this row is replaced from the registers above, and no other wave reads it, so the
                // order of the two does not matter, and stores issued here are long done when the kernel ends.
                if (hg == 0) {
                    const int row = pos % kTile;
                    const size_t row_off = ((size_t)kvh * n_ctx + pos) * D;
                    if (col == row % 16) {
#pragma unroll
                        for (int kk = 0; kk < G::kSteps; ++kk)
                            *reinterpret_cast<u32x4*>(const_cast<uint16_t*>(kc) + row_off + (kk * 4 + grp) * 8) = k_new16[kk];
                    }
                    if (lane < G::kChunksPerRow) *reinterpret_cast<u32x4*>(const_cast<uint16_t*>(vc) + row_off + lane * 8) = v_new16;
                }
            }
        }
        // One tile; `more`: another follows, which is asked for as its registers become free.  (Two copies, with and without: under a
        // condition in one, the compiler's waits at the loop's top are for K and V both, and the products start with V's arrival.)
        auto attend = [&](auto morec) {
            constexpr bool more = decltype(morec)::value;
            if constexpr (STORE) {
                if (owner && tile == own_tile) { // the tile of the new row: into the operand registers
                    const int row = pos % kTile;
                    if (col == row % 16) {
#pragma unroll
                        for (int kk = 0; kk < G::kSteps; ++kk)
#pragma unroll
                            for (int t = 0; t < 2; ++t) // (constant register indices: a computed one sends the array to scratch memory)
                                if (row / 16 == t) kreg[t * G::kSteps + kk] = k_new16[kk];
                    }
                }
            }
            // ---- S^T = K Q^T : rows = KV row (sub-tile t, row col), columns = query head ----
            f4 s[2], s2[2]; // the Q-lo product runs as its own accumulation chain
#pragma unroll
            for (int t = 0; t < 2; ++t) s[t] = s2[t] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < G::kSteps; ++kk)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const h8 ka = __builtin_bit_cast(h8, kreg[t * G::kSteps + kk]);
                    s[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka, qhi[kk], s[t], 0, 0, 0);
                    s2[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka, qlo[kk], s2[t], 0, 0, 0);
                }
            s[0] += s2[0];
            s[1] += s2[1];
            if constexpr (more) fetch_k(tile + tile_step); // the operand registers are free again
            FA_STAMP(3);

            // ---- softmax weights; lane (col, grp) holds rows t*16 + grp*4 + i of its column ----
            float v[8];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[t * 4 + i] = s[t][i];
            const int rows_left = npos - tile * kTile; // rows of this tile below the position (>= 32: all)
            if (rows_left < kTile) { // the last tile: rows past the position do not exist
                const int lim = rows_left - grp * 4;
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[t * 4 + i] = t * 16 + i < lim ? v[t * 4 + i] : -INFINITY;
            }
            float mx = fmaxf(fmaxf(v[0], v[1]), v[2]);
            mx = fmaxf(fmaxf(mx, v[3]), v[4]);
            mx = fmaxf(fmaxf(mx, v[5]), v[6]);
            mx = xor_max(fmaxf(mx, v[7]));
            // move the reference only when this tile's maximum is far above it (or it is unset)
            const bool move = (mx - m_ref) * c2 > kLazy || (m_ref == -INFINITY && mx > -INFINITY);
            if (tile == tile_first) { // (nothing summed up yet)
                m_ref = mx > -INFINITY ? mx : m_ref;
            } else if (__builtin_amdgcn_ballot_w64(move) != 0) {
                const float alpha = move ? fast_exp2((m_ref - mx) * c2) : 1.0f; // unset reference -> 0
                if (move) m_ref = mx;
                l_run *= alpha;
#pragma unroll
                for (int db = 0; db < G::kDBlk; ++db) o[db] *= alpha;
            }
            // exponent = s*c2 - m_ref*c2 + shift; a column that has seen no visible row keeps weight 0
            const float nb = (m_ref == -INFINITY) ? kPShift : kPShift - m_ref * c2;
            h8 ph, pl;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float pe = fast_exp2(__builtin_fmaf(v[e], c2, nb));
                l_run += pe;
                ph[e] = (_Float16)pe;
                pl[e] = (_Float16)(pe - (float)ph[e]);
            }

            __builtin_amdgcn_sched_barrier(0); // (the weights are made while V is still on its way)
            // head_dim 64 and kRotateLate: the next tile's K is waited for here, ahead of the request for its V.  Without the wait a wave has both on
            // their way nearly all the time, and in caches of a power of two of rows many KV heads at the same row, walked together, fall
            // on the same memory channels.  us a launch pair, rotate + store + attend, with table, without -> with the wait: 32 KV heads of 64, 8192 rows 20.2 ->
            // 18.6 (8232 rows: 15.2 both), 16 of them 12.75 -> 12.0; without a table, head_dim 128, 28 / 4 heads at 32000 of 32768 16.1 -> 15.2,
            // 32 / 32 at 4000 of 4096 16.1 -> 15.3.  With a table, head_dim 128 is the faster without: 28 / 4 heads 15.2, 15.4.
            if constexpr (more && (D == 64 || LATE)) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            // ---- V: registers -> this wave's LDS slice (K was needed first and arrives first) ----
            auto park_v = [&](auto whole) {
#pragma unroll
                for (int i = 0; i < G::kLoads; ++i) {
                    const int c = i * 64 + lane;
                    // rows at or past the position may hold anything; their weights are zero, and 0 * NaN is not
                    const u32x4 x = decltype(whole)::value || (c / G::kChunksPerRow) < rows_left ? vreg[i] : u32x4{0u, 0u, 0u, 0u};
                    *reinterpret_cast<u32x4*>(vs + (c / G::kChunksPerRow) * G::kRowBV + (c % G::kChunksPerRow) * 16) = x;
                }
            };
            if (rows_left < kTile) park_v(std::false_type());
            else park_v(std::true_type());
            if constexpr (STORE) // the new row, over what its tile brought back
                if (owner && tile == own_tile && lane < G::kChunksPerRow)
                    *reinterpret_cast<u32x4*>(vs + (pos % kTile) * G::kRowBV + lane * 16) = v_new16;
            if constexpr (more) fetch_v(tile + tile_step);
            wave_lds_sync();

            // ---- O^T += V^T P : rows = head_dim index, columns = query head, k = the tile's 32 KV rows
            //      in the order (grp, t, i) that matches the layout P already has ----
#pragma unroll
            for (int db = 0; db < G::kDBlk; ++db) {
                const h4 v0 = lds_read_tr(vs + v_rd + db * 32);
                const h4 v1 = lds_read_tr(vs + v_rd + 16 * G::kRowBV + db * 32);
                const h8 va = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
                o[db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, ph, o[db], 0, 0, 0);
                o[db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pl, o[db], 0, 0, 0);
            }
            if constexpr (more) wave_lds_sync(); // the slice is overwritten by the next tile
        };
        for (; tile + tile_step < n_tiles; tile += tile_step) attend(std::true_type());
        attend(std::false_type());
    } else { // (marks for the timeline build)
        FA_STAMP(1);
        FA_STAMP(2);
    }

    FA_STAMP(4);
    if (wu == 1) { // one wave has had a tile: nothing to merge
        if (wave != 0) return;
        FA_STAMP(5); // (nothing to hand over, nobody to wait for)
        FA_STAMP(6);
        const float l_tot = xor_sum(l_run);
        const int head = kvh * r + hl;
        if (!valid) return;
        const float inv = n_splits > 1 ? 1.0f : l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
        float* const po = n_splits > 1 ? part_o + ((size_t)id * n_head + head) * D : dst + (size_t)head * D; // (no splits: dst is the output)
#pragma unroll
        for (int db = 0; db < G::kDBlk; ++db) *reinterpret_cast<f4*>(po + db * 16 + grp * 4) = o[db] * inv;
        if (n_splits > 1 && grp == 0) {
            const size_t mi = (size_t)head * n_splits + id;
            part_ml[mi * 2 + 0] = (m_ref == -INFINITY) ? -INFINITY : m_ref * c2;
            part_ml[mi * 2 + 1] = l_tot;
        }
        FA_STAMP(7);
        return;
    }
    // ---- merge the waves through LDS ----
    float* const ml = reinterpret_cast<float*>(smem + G::kMlOff);
    float* const obuf = reinterpret_cast<float*>(smem + wave * G::kWaveB);
    const float l_tot = xor_sum(l_run);
    if (grp == 0) {
        ml[(wave * 16 + col) * 2 + 0] = (m_ref == -INFINITY) ? -INFINITY : m_ref * c2; // log2 units
        ml[(wave * 16 + col) * 2 + 1] = l_tot;
    }
#pragma unroll
    for (int db = 0; db < G::kDBlk; ++db)
        *reinterpret_cast<f4*>(obuf + col * G::kOStride + db * 16 + grp * 4) = o[db];
    FA_STAMP(5);
    __syncthreads();
    FA_STAMP(6);

    // (waves from the wu-th on have had no tile: two cases, so that the sums of a full run are not read under conditions)
    auto merge = [&](auto waves) {
        constexpr int W = decltype(waves)::value;
        for (int idx = threadIdx.x; idx < 16 * (D / 4); idx += kThreads) {
            const int c = idx / (D / 4);
            const int d4 = (idx % (D / 4)) * 4;
            const int h_local = hg * 16 + c;
            if (h_local >= r) continue;
            float mw[W], lw[W];
            float m_all = -INFINITY;
#pragma unroll
            for (int w = 0; w < W; ++w) {
                mw[w] = ml[(w * 16 + c) * 2 + 0];
                lw[w] = ml[(w * 16 + c) * 2 + 1];
                m_all = fmaxf(m_all, mw[w]);
            }
            float l_all = 0.0f;
            f4 acc = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < W; ++w) {
                const float wgt = fast_exp2(mw[w] - m_all); // a wave that had no tile has m = -inf -> weight 0
                l_all += lw[w] * wgt;
                acc += *reinterpret_cast<const f4*>(smem + w * G::kWaveB + ((size_t)c * G::kOStride + d4) * 4) * wgt;
            }
            const int head = kvh * r + h_local;
            if (n_splits > 1) {
                const size_t pi = (size_t)id * n_head + head;
                *reinterpret_cast<f4*>(part_o + pi * D + d4) = acc;
                if (d4 == 0) {
                    const size_t mi = (size_t)head * n_splits + id; // [head][split]: a head's pairs are one run of memory for the combine kernel
                    part_ml[mi * 2 + 0] = m_all;
                    part_ml[mi * 2 + 1] = l_all;
                }
            } else {
                const float inv = l_all > 0.0f ? 1.0f / l_all : 0.0f;
                *reinterpret_cast<f4*>(dst + (size_t)head * D + d4) = acc * inv; // (no splits: dst is the output)
            }
        }
    };
    if (wu <= 2) merge(std::integral_constant<int, 2>());
    else merge(std::integral_constant<int, kWaves>());
    FA_STAMP(7);
}

// Log-sum-exp merge of the decode splits.  One workgroup of 8 waves per (query head, 64-wide
// slice of head_dim); wave w takes the partial outputs of splits w, w + 8, ...; lane = element
// of the slice.  The kernel is little more than a trip to memory, so everything is shaped to
// make that one trip and little else:
//   * a head's (m, l) pairs are one run of memory ([head][split]): every wave fetches all of them
//     with one coalesced load per 64 splits (lane = split) and finds the overall maximum and the
//     overall row sum itself, with lane-swap reductions, while its partial outputs are still on
//     their way -- so no wave waits for another's statistics, and the weights of a wave's own
//     splits are lane reads;
//   * a wave's split indices are uniform, so the address arithmetic of the partial outputs
//     stays in the scalar unit and every load is one coalesced 256 bytes (per-thread 64-bit
//     address arithmetic for every load cost more than the trip);
//   * every load is issued before anything is waited on, and nothing else is read (not even the
//     position: splits that were inactive for it have said so in their (m, l)).
// The 8 waves' weighted sums meet in LDS behind the kernel's only barrier.  Partial outputs of
// inactive splits hold stale data and are never multiplied.
//   * the grid is (KV head, slice, head of its group): workgroups go to the eight XCDs in turn, so a KV head's partial results are merged
//     where they were written (8 KV heads), or where a half of them was (4), and the trip ends in that XCD's L2 instead of behind
//     it.  Rotate + store + attend, us a pair: Llama-3-8B at 1000 of 8192 6.55 -> 6.30, at 8191 10.86 -> 10.66,
//     Llama-3.2-1B at 1777 6.17 -> 5.99, Qwen2.5-7B at 16001 11.24 -> 11.01; two KV heads, four XCDs each, as before.
// PER: splits per wave (n_splits <= 8 * PER; the launcher picks the smallest that fits).
template <int D, int PER>
__global__ __launch_bounds__(512) void fa_decode_combine_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                                 float* __restrict__ out, const int n_splits, const int n_head, const int r) {
    constexpr int kGroups = 8;
    constexpr int kRounds = (kGroups * PER + 63) / 64; // (m, l) pairs per lane
    static_assert(kGroups * PER <= kMaxSplits, "more slots than splits can be");
    __shared__ float sh_acc[kGroups][64];
    const int head = (int)blockIdx.x * r + (int)blockIdx.z;
    const int lane = threadIdx.x & 63;
    const int d = (int)blockIdx.y * 64 + lane;
    const int sg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // (slots past n_splits read split 0 again and are voided below: a load under a branch
    // would make the compiler wait for the loads before it where the branch ends)
    float2 ml[kRounds];
    const float* const pm = part_ml + (size_t)head * n_splits * 2;
#pragma unroll
    for (int rd = 0; rd < kRounds; ++rd) {
        const int s = lane + 64 * rd;
        ml[rd] = *reinterpret_cast<const float2*>(pm + (s < n_splits ? s : 0) * 2);
    }
    float x[PER];
    const int stride = n_head * D; // (a split's partial outputs; the whole array is below 2^31 bytes)
    const float* const po = part_o + head * D + d;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int s = sg + j * kGroups;
        x[j] = po[(s < n_splits ? s : 0) * stride];
    }
    // ---- the head's statistics, in every wave, while the partial outputs travel ----
    float m_all = -INFINITY;
#pragma unroll
    for (int rd = 0; rd < kRounds; ++rd) {
        if (lane + 64 * rd >= n_splits) ml[rd] = float2{-INFINITY, 0.0f};
        m_all = fmaxf(m_all, ml[rd].x);
    }
    m_all = wave_max(m_all);
    float w[kRounds], l_all = 0.0f;
#pragma unroll
    for (int rd = 0; rd < kRounds; ++rd) {
        w[rd] = ml[rd].x > -INFINITY ? fast_exp2(ml[rd].x - m_all) : 0.0f; // (no split active at all: every weight 0)
        l_all = __builtin_fmaf(ml[rd].y, w[rd], l_all);
    }
    l_all = wave_sum(l_all);
    // ---- this wave's splits: split sg + 8j sits in lane (8j mod 64) + sg of round 8j / 64 ----
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const float wj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w[(j * kGroups) / 64]), ((j * kGroups) % 64) + sg));
        if (wj > 0.0f) acc = __builtin_fmaf(x[j], wj, acc); // (what a weightless split left behind may be anything)
    }
    sh_acc[sg][lane] = acc;
    __syncthreads();
    if (sg == 0) {
        float tot = 0.0f;
#pragma unroll
        for (int g = 0; g < kGroups; ++g) tot += sh_acc[g][lane];
        out[head * D + d] = l_all > 0.0f ? tot / l_all : 0.0f;
    }
}

template <int D>
hipError_t launch(const FaArgs& a, hipStream_t stream) {
    if (a.n_splits > 0x7fff || a.r > 0xffff || a.n_hgroups > 0xffff) return hipErrorInvalidValue;
    constexpr int lds = DGeom<D>::kLdsB;
    const dim3 g(a.n_kv, a.n_hgroups, a.n_splits), b(kDecodeWaves * 64);
    const unsigned splits_r = (unsigned)a.n_splits | (a.qsign < 0.0f ? 0x8000u : 0u) | (unsigned)a.r << 16;
    unsigned scale;
    memcpy(&scale, &a.c, sizeof(scale));
    const bool rotate = a.k_new && a.n_rot > 0, table = rotate && a.rope_angles && a.n_rot == D;
    const uint64_t scale_heads = table ? arg_ptr(a.rope_angles) : arg_pair(scale, (unsigned)a.n_head);
    float* const dst = a.n_splits > 1 ? a.part_o : a.out;
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, g, b, lds, stream, a.d_pos, a.q, a.kc, a.vc, a.n_ctx, splits_r, scale_heads, dst, a); };
    if (table && a.neox) go(fa_decode_split_kernel<D, kRotateNeox>);
    else if (table) go(fa_decode_split_kernel<D, kRotate>);
    else if (rotate) go(fa_decode_split_kernel<D, kRotateLate>);
    else if (a.k_new) go(fa_decode_split_kernel<D, kStore>);
    else go(fa_decode_split_kernel<D, kPlain>);

    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || a.n_splits == 1 || kProbeNoCombine) return e;
    const dim3 cgrid(a.n_kv, D / 64, a.r);
#define ORIN_FA_COMBINE_ARGS a.part_o, a.part_ml, a.out, a.n_splits, a.n_head, a.r
    if (a.n_splits <= 32) hipLaunchKernelGGL((fa_decode_combine_kernel<D, 4>), cgrid, dim3(512), 0, stream, ORIN_FA_COMBINE_ARGS);
    else if (a.n_splits <= 64) hipLaunchKernelGGL((fa_decode_combine_kernel<D, 8>), cgrid, dim3(512), 0, stream, ORIN_FA_COMBINE_ARGS);
    else if (a.n_splits <= 128) hipLaunchKernelGGL((fa_decode_combine_kernel<D, 16>), cgrid, dim3(512), 0, stream, ORIN_FA_COMBINE_ARGS);
    else hipLaunchKernelGGL((fa_decode_combine_kernel<D, 32>), cgrid, dim3(512), 0, stream, ORIN_FA_COMBINE_ARGS);
#undef ORIN_FA_COMBINE_ARGS
    return hipGetLastError();
}

} // namespace

hipError_t decode_launch(const FaArgs& a, int head_dim, hipStream_t stream) {
    drop_stale_error();
    return head_dim == 128 ? launch<128>(a, stream) : launch<64>(a, stream);
}

// The split kernel uses more than 64 KB of dynamic LDS; the opt-in is set once at init so
// that no launch path touches function attributes (decode runs under stream capture).
namespace {
template <int D, int MODE>
hipError_t allow_lds() {
    const auto kernel = fa_decode_split_kernel<D, MODE>;
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                               DGeom<D>::kLdsB);
}
} // namespace

hipError_t decode_allow_lds() {
    hipError_t e;
    auto all = [&](auto dc) {
        constexpr int D = decltype(dc)::value;
        if ((e = allow_lds<D, kPlain>()) != hipSuccess) return e;
        if ((e = allow_lds<D, kStore>()) != hipSuccess) return e;
        if ((e = allow_lds<D, kRotate>()) != hipSuccess) return e;
        if ((e = allow_lds<D, kRotateNeox>()) != hipSuccess) return e;
        return allow_lds<D, kRotateLate>();
    };
    return all(IntC<128>{}) != hipSuccess ? e : all(IntC<64>{});
}

hipError_t decode_stamps(long long* host, size_t n) {
#ifdef ORIN_FA_STAMPS
    if (n > (size_t)kStampWgs * kDecodeWaves * kStampSlots) return hipErrorInvalidValue;
    hipError_t e = hipMemcpyFromSymbol(host, HIP_SYMBOL(g_decode_stamps), n * sizeof(long long)); // (synchronises with the device)
    void* dev = nullptr;
    if (e == hipSuccess) e = hipGetSymbolAddress(&dev, HIP_SYMBOL(g_decode_stamps));
    if (e == hipSuccess) e = hipMemset(dev, 0, sizeof(g_decode_stamps)); // the next launch starts from an empty table
    return e;
#else
    (void)host; (void)n;
    return hipErrorNotSupported;
#endif
}

} // namespace orin_fa
