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
// Llama-3-8B's shapes, per launch, before -> now: q, k, v 34.1 -> 11.2 us (50 MB), output projection 11.9 -> 8.0 (34 MB), gate/up
// 47.7 -> 40.8 (235 MB, 5.75 TB/s: what a plain read reaches), down 25.0 -> 21.7 us (117 MB).
#include "layer_common.hpp"

namespace orin_fa {
namespace {

constexpr int kRun = 512;      // elements of a row that a wave's load instruction covers
constexpr int kMostRuns = 8;   // of a row, per wave

struct F16Args {
    GemvArgs g;
    int batches[3]; // of each matrix
};

__device__ __forceinline__ void lds_meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// RUNS: runs of a row per wave.  RB: rows of a matrix in a batch.
template <int RUNS, int RB, bool DUAL, int kWaves>
__global__ __launch_bounds__(kWaves * 64) void gemv_f16_kernel(const F16Args a) {
    constexpr int M = DUAL ? 2 : 1, R = M * RB;
    __shared__ float sh_part[2][kWaves][R];
    __shared__ float sh_ss[kWaves];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n_in = a.g.n_in;
    const unsigned row_bytes = (unsigned)n_in * 2u;

    unsigned off[RUNS]; // of this lane's 16 bytes of each run; past the row's end: its last 16 bytes, whose products are discarded
#pragma unroll
    for (int j = 0; j < RUNS; ++j) off[j] = min((unsigned)((j * kWaves + wave) * kRun + lane * 8) * 2u, row_bytes - 16u);

    // (the launcher's RUNS is the smallest that covers the row: only a wave's last run can reach past its end)
    const bool last_live = ((RUNS - 1) * kWaves + wave) * kRun + lane * 8 < n_in;

    const int b01 = a.batches[0], b012 = b01 + a.batches[1], total = b012 + a.batches[2];
    auto seg_of = [&](int b, int& row) {
        const int s = b < b01 ? 0 : b < b012 ? 1 : 2;
        row = (b - (s == 0 ? 0 : s == 1 ? b01 : b012)) * RB;
        return s;
    };
    h8 w[2][M][RB][RUNS];
    auto request = [&](h8 (&r)[M][RB][RUNS], int b) {
        int row;
        const int s = seg_of(min(b, total - 1), row); // (past the end: the last batch once more; never used)
        const GemvSeg& seg = a.g.seg[s];
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int i = 0; i < RB; ++i) {
                const unsigned char* const p = static_cast<const unsigned char*>(m ? a.g.w_up : seg.w) + (size_t)min(row + i, seg.n_out - 1) * row_bytes;
#pragma unroll
                for (int j = 0; j < RUNS; ++j) r[m][i][j] = __builtin_nontemporal_load(reinterpret_cast<const h8*>(p + off[j]));
            }
    };
    // the activation's loads first (loads return in order), then the first batch
    float x[RUNS][8], ss = 0.0f;
    {
        float g[RUNS][8];
#pragma unroll
        for (int j = 0; j < RUNS; ++j) {
            const int e = (int)(off[j] >> 1);
            *reinterpret_cast<float4*>(x[j]) = *reinterpret_cast<const float4*>(a.g.x + e);
            *reinterpret_cast<float4*>(x[j] + 4) = *reinterpret_cast<const float4*>(a.g.x + e + 4);
            const float* const nw = a.g.norm_w ? a.g.norm_w + e : a.g.x + e; // (always a load)
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
                x[j][i] = a.g.norm_w ? v * g[j][i] : v;
            }
        }
    }
    const bool has_norm = a.g.norm_w != nullptr;
    if (has_norm) {
        ss = wave_sum(ss);
        if (lane == 0) sh_ss[wave] = ss; // (read behind the first batch's barrier)
    }
    int set = 0;
    auto finish = [&](const h8 (&r)[M][RB][RUNS], int b) {
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
        int row0;
        const GemvSeg& seg = a.g.seg[seg_of(b, row0)];
        const int row = row0 + (int)threadIdx.x;
        if ((int)threadIdx.x < RB && row < seg.n_out) {
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
                const float rinv = 1.0f / sqrtf(s2 / (float)n_in + a.g.eps);
#pragma unroll
                for (int m = 0; m < M; ++m) v[m] *= rinv;
            }
            float y = v[0];
            if constexpr (DUAL) y = y / (1.0f + expf(-y)) * v[1]; // SiLU(gate) * up
            if (seg.bias) y += seg.bias[row];
            if (a.g.accumulate) atomicAdd(seg.y + row, y); // (one writer a row: a plain sum, without waiting for y)
            else seg.y[row] = y;
        }
        set ^= 1; // (two sets: one barrier a batch)
    };
    for (int b = blockIdx.x; b < total; b += 2 * (int)gridDim.x) {
        request(w[1], b + (int)gridDim.x);
        finish(w[0], b);
        if (b + (int)gridDim.x >= total) break;
        request(w[0], b + 2 * (int)gridDim.x);
        finish(w[1], b + (int)gridDim.x);
    }
}

template <int RUNS, bool DUAL, int kWaves>
hipError_t launch_as(const GemvArgs& g, int cu_count, hipStream_t stream) {
    // rows in a batch: about 4 KB a wave on their way beside what is being multiplied out
    constexpr int RB = RUNS * (DUAL ? 2 : 1) <= 2 ? 4 / (RUNS * (DUAL ? 2 : 1)) : 1;
    // workgroups that are resident at once: longer shares of a row take more registers
    constexpr int kPerCu = kWaves == 8 ? 1 : RUNS >= 5 ? 2 : 3;
    F16Args a{};
    a.g = g;
    int total = 0;
    for (int i = 0; i < g.n_seg; ++i) total += a.batches[i] = (g.seg[i].n_out + RB - 1) / RB;
    const int wgs = min(total, cu_count * kPerCu);
    hipLaunchKernelGGL((gemv_f16_kernel<RUNS, RB, DUAL, kWaves>), dim3(wgs), dim3(kWaves * 64), 0, stream, a);
    return hipGetLastError();
}

template <int RUNS, int kWaves>
hipError_t launch_runs(const GemvArgs& g, int cu_count, hipStream_t stream) {
    return g.w_up ? launch_as<RUNS, true, kWaves>(g, cu_count, stream) : launch_as<RUNS, false, kWaves>(g, cu_count, stream);
}

} // namespace

// Four waves a workgroup up to rows of 16384 elements, eight beyond (at most 32768).
hipError_t gemv_f16_launch(const GemvArgs& g, int cu_count, hipStream_t stream) {
    const int runs = (g.n_in + kRun - 1) / kRun;
    if (runs > 4 * kMostRuns) {
        switch ((runs + 7) / 8) {
        case 5: return launch_runs<5, 8>(g, cu_count, stream);
        case 6: return launch_runs<6, 8>(g, cu_count, stream);
        case 7: return launch_runs<7, 8>(g, cu_count, stream);
        case 8: return launch_runs<8, 8>(g, cu_count, stream);
        default: return hipErrorInvalidValue;
        }
    }
    switch ((runs + 3) / 4) {
    case 1: return launch_runs<1, 4>(g, cu_count, stream);
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
