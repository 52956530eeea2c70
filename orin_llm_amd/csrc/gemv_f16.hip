// Matrix-vector products over F16 weight rows for gfx950 (MI355X): y = W x for one token, bound by the rows' bytes alone
// (two bytes a weight and one v_fma_mix_f32; the activation stays fp32, as in the reference's CPU backend,
// src/model_cpu.cpp:153-167, and its gemv_plain_k, src/kernels.cu:430-470).
//
//   * A row is read as runs of 1 KB: a load instruction of a wave is 512 consecutive elements, and the workgroup's waves
//     take neighbouring runs.  (The kernel of gemv.hip gives a lane 32 consecutive elements, four loads 64 bytes apart,
//     and leaves putting the lines together to the vector cache.)
//   * A wave keeps its runs for every row, so its share of the activation -- 8 floats a lane and run -- sits in
//     registers, and a workgroup fetches the activation once.
//   * Rows go in batches, the next batch requested before the last is multiplied out; the waves' sums meet in LDS behind one
//     barrier a batch that waits for LDS only.
//   * The matrices of a launch (q, k, v) are one sequence of batches, so that workgroups get equal shares of all of them.
//     (As rows of the grid, two of three 1024-row matrices kept 512 workgroups each busy for two rows.)
//   * The RMS norm is folded in as in gemv_mfma.hip: products of x w, the norm's scalar applied to the finished sums.
// What a workgroup needs ahead of its first request is in registers when it starts, rows are addressed by descriptors in scalar registers, so
// that nothing waits for a load but its use, and a launch of one matrix asks nothing of which one (kMulti).
// Llama-3-8B's shapes, per launch, with gemv.hip's kernel -> now: q, k, v 34.1 -> 10.65 us (50 MB), output projection 11.9 -> 7.65 (34 MB),
// gate/up 47.7 -> 37.0 (235 MB, 6.35 TB/s: what the fastest plain read of that size reaches), down 25.0 -> 20.5 us (117 MB, 5.7).
#include "layer_common.hpp"

#include <type_traits>

namespace orin_fa {
namespace {

constexpr int kRun = 512;      // elements of a row that a wave's load instruction covers
constexpr int kMostRuns = 8;   // of a row, per wave

__device__ __forceinline__ void lds_meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// RUNS: runs of a row per wave.  RB: rows of a matrix in a batch.
// What the first requests need comes in the leading arguments, in registers when a wave starts: the matrices (w1: of two that become
// one product the second), the batches that end with the first matrix, with the second and with the last, and
//   shape   n_in, 16 bits | rows of each matrix's last batch - 1, 4 bits each
template <int RUNS, int RB, bool DUAL, int kWaves, bool kMulti>
__global__ __launch_bounds__(kWaves * 64) void gemv_f16_kernel(const uint64_t w0, const uint64_t w1, const uint64_t w2, const float* x_in, const float* norm_w,
                                                              const unsigned b01, const unsigned b012, const unsigned total, const unsigned shape, const GemvArgs a) {
    constexpr int M = DUAL ? 2 : 1, R = M * RB;
    __shared__ float sh_part[2][kWaves][R];
    __shared__ float sh_ss[kWaves];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n_in = (int)(shape & 0xffffu);
    const unsigned row_bytes = (unsigned)n_in * 2u;

    unsigned off[RUNS]; // of this lane's 16 bytes of each run; past the row's end: its last 16 bytes, whose products are discarded
#pragma unroll
    for (int j = 0; j < RUNS; ++j) off[j] = min((unsigned)((j * kWaves + wave) * kRun + lane * 8) * 2u, row_bytes - 16u);

    // (the launcher's RUNS is the smallest that covers the row: only a wave's last run can reach past its end)
    const bool last_live = ((RUNS - 1) * kWaves + wave) * kRun + lane * 8 < n_in;

    struct Batch {
        int seg, row, rows;      // matrix, first row, rows of it
        unsigned second, third;  // all ones where it is of the second matrix or behind it, of the third
    };
    auto past = [](unsigned b, unsigned limit) { return 0u - ((unsigned)(limit - b) >> 31); }; // all ones where b > limit (both below 2^31)
    // (Captured by value: by reference the choices become loads from the stack.  And as masks of words: a comparison's outcome becomes a
    // number by way of a vector register, and what follows from it then stays in those.)
    auto batch_of = [b01, b012, total, shape, past](unsigned b) {
        if constexpr (!kMulti) {
            const unsigned last = past(b, total - 2u);
            return Batch{0, (int)b * RB, RB == 1 ? 1 : (int)((shape >> 16 & 15u & last) | ((RB - 1u) & ~last)) + 1, 0u, 0u};
        }
        const unsigned second = past(b, b01 - 1u), third = past(b, b012 - 1u); // all ones or zero
        const unsigned first = (b01 & second & ~third) | (b012 & third), end = (b01 & ~second) | (b012 & second & ~third) | (total & third);
        const unsigned last = past(b, end - 2u), seg = (second & 1u) + (third & 1u);
        return Batch{(int)seg, (int)(b - first) * RB, (int)((shape >> (16u + 4u * seg) & 15u & last) | ((RB - 1u) & ~last)) + 1, second, third};
    };
    h8 w[2][M][RB][RUNS];
    auto request = [w0, w1, w2, total, row_bytes, &off, batch_of, past](h8 (&r)[M][RB][RUNS], unsigned b) {
        // Past the end: the last batch's rows, of no bytes, and never used.  (Read once more, they were as many bytes again in a launch of one
        // turn: 128 rows of 14336 elements 5.05 -> 4.2 us, 768 of 8192 5.0 -> 4.55, q, k, v of 128, 32, 32 rows of 2048 3.45 -> 3.15.)
        const unsigned bytes = row_bytes & past(total, b);
        const Batch t = batch_of(min(b, total - 1));
        const uint64_t second = (uint64_t)(int64_t)(int)t.second, third = (uint64_t)(int64_t)(int)t.third;
        const uint64_t mine = !kMulti ? w0 : (w0 & ~second) | (w1 & second & ~third) | (w2 & third);
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int i = 0; i < RB; ++i) {
                // (The row's address as a descriptor's base, in scalar registers: an address in vector registers takes some that loads
                // under way return to, and the wait for them puts an end to two batches on their way.  A row that is not there is one of
                // no bytes.)
                const auto rsrc = make_rsrc(ptr_arg<const unsigned char>(m ? w1 : mine) + (size_t)(unsigned)(t.row + i) * row_bytes, i == 0 ? bytes : bytes & past((unsigned)t.rows, (unsigned)i));
#pragma unroll
                for (int j = 0; j < RUNS; ++j) r[m][i][j] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off[j], 0, 2)); // (streaming)
            }
    };
    // the activation's loads first (loads return in order), then the first batch
    float x[RUNS][8], ss = 0.0f;
    {
        float g[RUNS][8];
#pragma unroll
        for (int j = 0; j < RUNS; ++j) {
            const int e = (int)(off[j] >> 1);
            *reinterpret_cast<float4*>(x[j]) = *reinterpret_cast<const float4*>(x_in + e);
            *reinterpret_cast<float4*>(x[j] + 4) = *reinterpret_cast<const float4*>(x_in + e + 4);
            const float* const nw = norm_w ? norm_w + e : x_in + e; // (always a load)
            *reinterpret_cast<float4*>(g[j]) = *reinterpret_cast<const float4*>(nw);
            *reinterpret_cast<float4*>(g[j] + 4) = *reinterpret_cast<const float4*>(nw + 4);
        }
        __builtin_amdgcn_sched_barrier(0);
        request(w[0], blockIdx.x);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < RUNS; ++j) {
            const bool live = j < RUNS - 1 || last_live;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float v = live ? x[j][i] : 0.0f;
                ss += v * v;
                x[j][i] = norm_w ? v * g[j][i] : v;
            }
        }
    }
    const bool has_norm = norm_w != nullptr;
    if (has_norm) {
        ss = wave_sum(ss);
        if (lane == 0) sh_ss[wave] = ss; // (read behind the first batch's barrier)
    }
    int set = 0;
    auto finish = [&](const h8 (&r)[M][RB][RUNS], unsigned b) {
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int i = 0; i < RB; ++i) {
                float acc = 0.0f, whole = 0.0f;
#pragma unroll
                for (int j = 0; j < RUNS; ++j) {
                    whole = acc;
#pragma unroll
                    for (int k = 0; k < 8; ++k) acc = __builtin_fmaf((float)r[m][i][j][k], x[j][k], acc);
                }
                acc = wave_sum(last_live ? acc : whole); // (a select, not a factor of zero: the row's last weights may be infinite)
                if (lane == 0) sh_part[set][wave][m * RB + i] = acc;
            }
        lds_meet();
        const Batch t = batch_of(b);
        if ((int)threadIdx.x < t.rows) {
            const GemvSeg& seg = a.seg[t.seg];
            const int row = t.row + (int)threadIdx.x;
            float v[M];
#pragma unroll
            for (int m = 0; m < M; ++m) {
                v[m] = 0.0f;
#pragma unroll
                for (int u = 0; u < kWaves; ++u) v[m] += sh_part[set][u][m * RB + (int)threadIdx.x];
            }
            if (has_norm) {
                float s2 = 0.0f;
#pragma unroll
                for (int u = 0; u < kWaves; ++u) s2 += sh_ss[u];
                const float rinv = 1.0f / sqrtf(s2 / (float)n_in + a.eps);
#pragma unroll
                for (int m = 0; m < M; ++m) v[m] *= rinv;
            }
            float y = v[0];
            if constexpr (DUAL) y = y / (1.0f + expf(-y)) * v[1]; // SiLU(gate) * up
            if (seg.bias) y += seg.bias[row];
            if (a.accumulate) atomicAdd(seg.y + row, y); // (one writer a row: a plain sum, without waiting for y)
            else seg.y[row] = y;
        }
        set ^= 1; // (two sets: one barrier a batch)
    };
    for (unsigned b = blockIdx.x; b < total; b += 2 * gridDim.x) {
        request(w[1], b + gridDim.x);
        finish(w[0], b);
        if (b + gridDim.x >= total) break;
        request(w[0], b + 2 * gridDim.x);
        finish(w[1], b + gridDim.x);
    }
}

template <int RUNS, bool DUAL, int kWaves, int RB>
hipError_t launch_batches(const GemvArgs& g, int cu_count, hipStream_t stream) {
    static_assert(RB <= 16, "rows of a batch: four bits of `shape`");
    constexpr int R = (DUAL ? 2 : 1) * RB;
    const unsigned cus = (unsigned)cu_count, row_bytes = (unsigned)g.n_in * 2u;
    unsigned ends[3] = {}, total = 0, shape = (unsigned)g.n_in;
    for (int i = 0; i < 3; ++i) {
        if (i < g.n_seg) {
            total += (unsigned)(g.seg[i].n_out + RB - 1) / RB;
            shape |= (unsigned)((g.seg[i].n_out - 1) % RB) << (16 + 4 * i);
        }
        ends[i] = total;
    }
    // Workgroups a CU (four waves): one, or two where the two batches of one are short of 64 KB, its waves' last runs being partly idle, and
    // two turns of the chip do not take all batches; of several matrices up to 64 KB; and with rows of up to 2048 elements, eight rows a
    // batch, where one more batch a CU is a long turn: of several matrices, and of pairs up to four turns.  us a launch, one -> two: of
    // 5120 elements 5120 rows 11.6 -> 10.25, q, k, v of 5120, 1280 and 1280 17.8 -> 14.75, pairs of 4096 17.3 -> 16.0, but 768 rows alone
    // 3.75 -> 4.1; of 3072 elements q, k, v of 4096, 1024 and 1024 9.25 -> 8.6, but 2048 rows alone 4.3 -> 4.55; of 4096 elements 4096
    // rows 7.35 -> 7.55; of 2048 elements q, k, v of 2048, 512 and 512 5.2 -> 4.95, pairs of 1536 5.15 -> 4.9, but of 6144 10.65 -> 11.0.
    const unsigned under_way = 2u * R * row_bytes;
    const bool multi = g.n_seg > 1;
    bool two = false;
    if constexpr (kWaves == 4)
        two = RUNS == 1 ? multi || (DUAL && total < 4 * cus) : total > 2 * cus && under_way <= (multi ? 64u : 48u) * 1024u;
    const unsigned wgs = min(total, cus * (kWaves == 1 ? 4u : kWaves < 4 || two ? 2u : 1u));
    auto go = [&](auto multic) {
        constexpr bool kMulti = !DUAL && decltype(multic)::value;
        hipLaunchKernelGGL((gemv_f16_kernel<RUNS, RB, DUAL, kWaves, kMulti>), dim3(wgs), dim3(kWaves * 64), 0, stream, arg_ptr(g.seg[0].w),
                           arg_ptr(g.w_up ? g.w_up : g.seg[1].w), arg_ptr(g.seg[2].w), g.x, g.norm_w, ends[0], ends[1], ends[2], shape, g);
    };
    if (multi) go(std::true_type());
    else go(std::false_type());
    return hipGetLastError();
}

template <int RUNS, bool DUAL, int kWaves>
hipError_t launch_as(const GemvArgs& g, int cu_count, hipStream_t stream) {
    // Rows in a batch: some 64 KB a CU on their way, in few workgroups -- each fetches the activation and the norm's weights
    // for itself, 4 waves of 5 KB to 16 KB in each of two batches.  us a launch, three workgroups a CU with half the rows a batch
    // (two, of long rows, with one) -> this: Llama-3-8B's q, k, v 11.5 -> 10.65, output 8.25 -> 7.65, gate/up 41.0 -> 37.0 (6.35 TB/s),
    // down 21.8 -> 20.5, logits 158.5 -> 155.2 (6.8 TB/s); two workgroups a CU with these batches 11.35, 8.35, 37.6, 21.6, 160.5.
    // Eight waves, whose rows are over 45 KB: one (two: 28672 elements, 4096 rows 35.4 -> 36.5 us, q, k, v of 4096, 1024 and 1024 51.65 ->
    // 53.5, 640 rows 8.65 -> 10.3).  11 to 15: two, but up to three rows a CU one, which is less for the busiest CU (18944 elements, 640 rows
    // by two 7.95, by one 7.05 us, 128 rows 5.3 and 4.4, 1024 rows 8.9 both; q, k, v of 4096, 1024 and 1024 35.25 and 39.5).
    constexpr int M = DUAL ? 2 : 1;
    if constexpr (kWaves > 8 && !DUAL) {
        long long rows = 0;
        for (int i = 0; i < g.n_seg; ++i) rows += g.seg[i].n_out;
        return rows <= 3 * cu_count ? launch_batches<RUNS, DUAL, kWaves, 1>(g, cu_count, stream) : launch_batches<RUNS, DUAL, kWaves, 2>(g, cu_count, stream);
    } else {
        constexpr int RB = kWaves > 4 ? 1 : RUNS * M <= 8 && RUNS <= 4 ? 8 / (RUNS * M) : DUAL ? 1 : 2;
        return launch_batches<RUNS, DUAL, kWaves, RB>(g, cu_count, stream);
    }
}

template <int RUNS, int kWaves>
hipError_t launch_runs(const GemvArgs& g, int cu_count, hipStream_t stream) {
    return g.w_up ? launch_as<RUNS, true, kWaves>(g, cu_count, stream) : launch_as<RUNS, false, kWaves>(g, cu_count, stream);
}

} // namespace

// As many waves a workgroup as a row has runs, four from there on up to rows of 16384 elements, 11 to 15 with three runs each up to 23040, eight
// beyond (at most 32768).  (Rows of two and three runs by four waves, the others idle, and by two and three, two workgroups a CU: 151936 rows of
// 1024 45.4 -> 41.0 us, 4096 rows 4.84 -> 4.31; 151936 rows of 1536 62.6 -> 60.1, two matrices of 8960 11.54 -> 11.32.  3584 rows by eight waves and
// by 11 to 15: of 16896 20.7 -> 19.7, of 22016 27.7 -> 26.6; from 24576 on eight are as fast or faster, 29.3 and 29.6.)
hipError_t gemv_f16_launch(const GemvArgs& g, int cu_count, hipStream_t stream) {
    const int runs = (g.n_in + kRun - 1) / kRun;
    if (runs > 45) {
        switch ((runs + 7) / 8) {
        case 6: return launch_runs<6, 8>(g, cu_count, stream);
        case 7: return launch_runs<7, 8>(g, cu_count, stream);
        case 8: return launch_runs<8, 8>(g, cu_count, stream);
        default: return hipErrorInvalidValue;
        }
    }
    if (runs > 4 * kMostRuns) {
        switch ((runs + 2) / 3) {
        case 11: return launch_runs<3, 11>(g, cu_count, stream);
        case 12: return launch_runs<3, 12>(g, cu_count, stream);
        case 13: return launch_runs<3, 13>(g, cu_count, stream);
        case 14: return launch_runs<3, 14>(g, cu_count, stream);
        default: return launch_runs<3, 15>(g, cu_count, stream);
        }
    }
    switch (runs) {
    case 1: return launch_runs<1, 1>(g, cu_count, stream);
    case 2: return launch_runs<1, 2>(g, cu_count, stream);
    case 3: return launch_runs<1, 3>(g, cu_count, stream);
    case 4: return launch_runs<1, 4>(g, cu_count, stream);
    }
    switch ((runs + 3) / 4) {
    case 2: return launch_runs<2, 4>(g, cu_count, stream);
    case 3: return launch_runs<3, 4>(g, cu_count, stream);
    case 4: return launch_runs<4, 4>(g, cu_count, stream);
    case 5: return launch_runs<5, 4>(g, cu_count, stream);
    case 6: return launch_runs<6, 4>(g, cu_count, stream);
    case 7: return launch_runs<7, 4>(g, cu_count, stream);
    default: return launch_runs<8, 4>(g, cu_count, stream);
    }
}

} // namespace orin_fa
