// Rotary position embedding for gfx950 (MI355X), in place on fp32 rows [rows][head_dim].
//
// Replaces the reference's rope_neox_k / rope_normal_k and their four wrappers (reference:
// src/kernels.cu:1619-1657, 2059-2075; CPU statement src/model_cpu.cpp:179-203; call sites
// src/model_gpu.cu:277-279, 379-381).  Pair i of a row is rotated by the angle pos * freq_i,
// freq_i = theta^(-2i/n_rot) (divided by freq_factors[i] when given); "neox" pairs element i
// with i + n_rot/2, "normal" pairs 2i with 2i + 1; elements at or past n_rot are left alone.
// pos = n_past + row / heads (batch form) or *d_pos (single-token form, read on the device).
//
// Two kernels: rope_pieces_kernel for the shapes models have (n_rot a multiple of 8, 16-byte aligned
// rows), all 128-bit accesses, and rope_kernel for any even n_rot.  In rope_kernel,
// every head of a token shares the token's angles, so one thread owns (token, pair, group of up
// to 8 heads): the block's first threads compute the frequency of each pair once into LDS, each
// thread forms its angle and one sine/cosine, then rotates its heads; all loads are issued
// before any of that arithmetic -- where the reference spends a power, a sine and a cosine per
// element pair of every head.
// Arithmetic (rope_freq, rope_rotate in fa_common.hpp) follows the CPU statement operation by
// operation in fp32.  Sine and cosine are the accurate library versions (full range
// reduction), not the fast hardware approximations the reference's GPU path uses.  They are taken
// together: one range reduction (100 instructions where the angle is large) instead of two, the same
// bits as sinf and cosf give (all 2^32 floats compared once, with the compiler that check_toolchain() in
// build.py asks for).  Back to back in a graph, rotary and
// cache rows of 512 tokens, apart -> together: 12 + 2 heads of 128 2.87 -> 2.82 us, 32 + 8 heads
// 4.75 -> 4.59, 28 + 4 heads 4.04 -> 3.94; 301 tokens of 32 + 8 heads of 64 3.12 -> 3.07.
#include "fa_common.hpp"

namespace orin_fa {
namespace {

constexpr int kHeadsPerThread = 8;
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));

// The rotated rows and the cache rows are read next by another kernel, on other compute units:
// streaming stores send them on instead of leaving them dirty in this die's cache until the
// kernel ends.
__device__ __forceinline__ void store_stream(float* p, const float4& v) {
    __builtin_nontemporal_store(f4{v.x, v.y, v.z, v.w}, reinterpret_cast<f4*>(p));
}

template <bool NEOX, bool IND>
__global__ __launch_bounds__(256) void rope_kernel(float* x, int tokens, int heads, int head_dim, const RopeFreq f, int n_past,
                                                   const int* d_pos, const float* freq_factors) {
#pragma clang fp contract(off)
    __shared__ float sh_freq[128];
    const int half = f.n_rot / 2;
    const int n_hgroups = (heads + kHeadsPerThread - 1) / kHeadsPerThread;
    // pair index fastest, then head group, then token; a block covers whole runs of pairs when
    // half divides 256, otherwise every thread computes its own frequency
    const bool shared_freq = half <= 128 && (256 % half) == 0;
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    const bool active = t < (long long)tokens * n_hgroups * half;
    const int i = (int)(t % half);
    const long long th = t / half;
    const int hgroup = (int)(th % n_hgroups), token = (int)(th / n_hgroups);
    const int h0 = hgroup * kHeadsPerThread;
    float* row = x + ((size_t)token * heads + h0) * head_dim;
    const int i0 = NEOX ? i : 2 * i, i1 = NEOX ? i + half : 2 * i + 1;
    // The loads go out first: nothing they need depends on the angle, and the power, sine and
    // cosine below then run while the rows are on their way.
    float x0[kHeadsPerThread], x1[kHeadsPerThread];
#pragma unroll
    for (int u = 0; u < kHeadsPerThread; ++u)
        if (active && h0 + u < heads) {
            x0[u] = row[(size_t)u * head_dim + i0];
            x1[u] = row[(size_t)u * head_dim + i1];
        }
    const int pos = IND ? *d_pos : n_past + token;
    if (shared_freq && (int)threadIdx.x < half) {
        sh_freq[threadIdx.x] = rope_freq(threadIdx.x, f, freq_factors);
    }
    if (shared_freq) __syncthreads();
    if (!active) return;
    float freq;
    if (shared_freq) {
        freq = sh_freq[i];
    } else {
        freq = rope_freq(i, f, freq_factors);
    }
    const float ang = (float)pos * freq;
    float s, c;
    sincosf(ang, &s, &c);
#pragma unroll
    for (int u = 0; u < kHeadsPerThread; ++u)
        if (h0 + u < heads) {
            rope_rotate(x0[u], x1[u], c, s);
            row[(size_t)u * head_dim + i0] = x0[u];
            row[(size_t)u * head_dim + i1] = x1[u];
        }
}

// The same rotation for the shapes models have (n_rot a multiple of 8, rows 16-byte aligned), and with it, in one launch,
// the whole of what a prefill layer does ahead of its attention (reference call sites: src/model_gpu.cu:378-382): K rows
// are also stored to the cache as fp16 (rounded from the rotated fp32 value, as the store kernel rounds what the rotary
// kernel wrote), V rows are stored.
//
// A piece is four adjacent pairs of one head -- "neox": elements 4j..4j+3 and the four n_rot/2 further on; "normal":
// elements 8j..8j+7 -- so every load and store is a full 128-bit access that a wave makes on whole cache lines.  A block
// takes a few tokens (as many as it has threads for their angles) and a few heads, of Q, K and V in that order: its
// threads ask for their pieces, form one (cos, sin) each for the block's table in LDS, and rotate.  These launches are
// short chains, not bandwidth: a wave issues an instruction every 2 ns, so what counts is how many stand between a
// thread's start and its stores.  Per thread that is one sine and cosine (four, when a thread formed the angles of its own
// pieces), no power (a product of doubles the host prepares; 300 instructions) and 32-bit index arithmetic by
// multiplication (64-bit divisions: 500).  Measured, per launch: 45 tokens
// of Qwen2.5-1.5B (Q, K and V rows) 4.3 -> 3.0 us, a single token's Q rows 4.0 -> 2.9 us, 301 tokens of Llama-3.2-1B's Q rows
// 4.1 -> 3.9; 512 tokens of Llama-3-8B (25 MB) stay at the memory's 7.7 us.  Two or four pieces per thread, which form an
// angle once for more heads, were no faster at any size (512 tokens of Qwen2.5-7B 4.5 with one, 4.9 with two; 4096 tokens
// 31.2, 31.9, 32.6 with one, two, four).
//
// The cache rows go out as ordinary stores, Q and K as streaming ones: the attention of the same chunk reads the new rows
// once per query tile and head group, and finds them in the last-level cache where a streaming store had sent them past it.
// This launch and the attention behind it, 512 tokens at the start of a sequence, streaming -> ordinary: Qwen2.5-1.5B 11.6
// -> 10.5 us, Qwen3-0.6B 13.1 -> 12.0, Llama-3-8B 17.7 -> 17.2; 512 tokens at 4096, where they are an eighth of the rows
// read, 27.0 -> 26.7, 31.5 -> 31.2, 46.4 -> 46.5.
constexpr int kRopeThreads = 256;
constexpr int kRopePieceHeads = 65535 * (kRopeThreads / 64); // heads of a token a grid can hold: a block takes four or more

// What the first loads need comes first, as scalars that are in a wave's registers when it starts (kernel-argument preload); the
// rest in as few bytes as will do (launch_lean()).
//   counts   tokens | heads of Q, K and V together << 32
//   heads    heads of Q << 0 | of K << 32
//   shape    pairs of a head, 10 bits | pieces of a head, 7 | tokens of a block, 10 | log2 of its heads, 5 | head_dim << 32
//   magic    x / pieces = x * magic >> 16, x < 256 | the same for pairs, x < 256, << 32
struct RopeRest {
    uint16_t *kc, *vc;
    const int* d_pos;
    const float* freq_factors;
    double step; // theta^(-2 / n_rot), 0: no power of two (RopeFreq)
    float theta;
    int n_past, n_ctx;
};

// rope_freq() of the plan whose first double is `step`: the same squares, taken here.
__device__ __forceinline__ float rope_freq_of_step(int i, int n_rot, const RopeRest& a) {
    RopeFreq f;
    f.theta = a.theta;
    f.n_rot = n_rot;
    f.by_steps = a.step != 0.0;
    double s = a.step;
#pragma unroll
    for (int k = 0; k < 8; ++k, s *= s) f.step[k] = s;
    return rope_freq(i, f, a.freq_factors);
}

template <bool NEOX>
__global__ __launch_bounds__(kRopeThreads) void rope_pieces_kernel(const uint64_t q_bits, const uint64_t k_bits, const uint64_t v_bits, const uint64_t counts,
                                                                   const uint64_t heads, const uint64_t shape, const uint64_t magic, const RopeRest a) {
#pragma clang fp contract(off)
    float *const q = ptr_arg<float>(q_bits), *const k = ptr_arg<float>(k_bits);
    const float* const v = ptr_arg<const float>(v_bits);
    __shared__ __attribute__((aligned(16))) float2 sh_cs[kRopeThreads]; // (read two pairs at a time)
    const int tokens = (int)(unsigned)counts, n_heads = (int)(counts >> 32), n_q = (int)(unsigned)heads, n_k = (int)(heads >> 32);
    const int half = (int)(shape & 1023u), quads = (int)((shape >> 10) & 127u), block_tokens = (int)((shape >> 17) & 1023u);
    const int block_heads_log2 = (int)((shape >> 27) & 31u), head_dim = (int)(shape >> 32);
    const unsigned quads_magic = (unsigned)magic, half_magic = (unsigned)(magic >> 32);
    const int tid = threadIdx.x, token0 = (int)blockIdx.x * block_tokens, head0 = (int)blockIdx.y << block_heads_log2;
    const int o1 = NEOX ? half : 4;
    float4 lo, hi;
    const int rest = (int)((unsigned)tid * quads_magic >> 16), quad = tid - rest * quads;
    const int head = head0 + (rest & ((1 << block_heads_log2) - 1)), block_token = rest >> block_heads_log2, token = token0 + block_token;
    const bool live = block_token < block_tokens && token < tokens && head < n_heads;
    const bool is_q = head < n_q, is_k = !is_q && head < n_q + n_k;
    if (live) {
        const float* const row = is_q ? q + ((size_t)token * n_q + head) * head_dim
                                      : (is_k ? k : v) + ((size_t)token * n_k + (head - n_q - (is_k ? 0 : n_k))) * head_dim;
        const float* const p = row + quad * (NEOX ? 4 : 8);
        lo = *reinterpret_cast<const float4*>(p);
        hi = *reinterpret_cast<const float4*>(p + o1);
    }
    {
        const int t = (int)((unsigned)tid * half_magic >> 16), i = tid - t * half;
        if (t < block_tokens) {
            const float ang = (float)(a.d_pos ? *a.d_pos : a.n_past + token0 + t) * rope_freq_of_step(i, 2 * half, a);
            float s, c;
            sincosf(ang, &s, &c);
            sh_cs[tid] = float2{c, s};
        }
    }
    __syncthreads();
    if (!live) return;
    if (is_q || is_k) {
        const float4* const cs = reinterpret_cast<const float4*>(sh_cs + block_token * half + 4 * quad);
        const float4 c01 = cs[0], c23 = cs[1];
        if (NEOX) {
            rope_rotate(lo.x, hi.x, c01.x, c01.y);
            rope_rotate(lo.y, hi.y, c01.z, c01.w);
            rope_rotate(lo.z, hi.z, c23.x, c23.y);
            rope_rotate(lo.w, hi.w, c23.z, c23.w);
        } else {
            rope_rotate(lo.x, lo.y, c01.x, c01.y);
            rope_rotate(lo.z, lo.w, c01.z, c01.w);
            rope_rotate(hi.x, hi.y, c23.x, c23.y);
            rope_rotate(hi.z, hi.w, c23.z, c23.w);
        }
        float* const row = is_q ? q + ((size_t)token * n_q + head) * head_dim : k + ((size_t)token * n_k + (head - n_q)) * head_dim;
        float* const p = row + quad * (NEOX ? 4 : 8);
        store_stream(p, lo);
        store_stream(p + o1, hi);
    }
    if (!is_q && a.kc) {
        const int h = head - n_q - (is_k ? 0 : n_k);
        uint16_t* const p = (is_k ? a.kc : a.vc) + ((size_t)h * a.n_ctx + a.n_past + token) * head_dim + quad * (NEOX ? 4 : 8);
        half4_t l, m;
        l[0] = (_Float16)lo.x; l[1] = (_Float16)lo.y; l[2] = (_Float16)lo.z; l[3] = (_Float16)lo.w;
        m[0] = (_Float16)hi.x; m[1] = (_Float16)hi.y; m[2] = (_Float16)hi.z; m[3] = (_Float16)hi.w;
        *reinterpret_cast<half4_t*>(p) = l;
        *reinterpret_cast<half4_t*>(p + o1) = m;
    }
}

// n_k, n_v: heads behind the n_q ones that go to the cache (0: the rotation alone).
hipError_t pieces_launch(float* q, float* k, const float* v, RopeRest a, int tokens, int head_dim, int n_rot, float theta, int n_q, int n_k, int n_v,
                         bool neox, hipStream_t stream) {
    const RopeFreq f = rope_freq_plan(n_rot, theta);
    a.step = f.by_steps ? f.step[0] : 0.0;
    a.theta = theta;
    const int half = n_rot / 2, quads = n_rot / 8, n_heads = n_q + n_k + n_v;
    int block_tokens = kRopeThreads / half;
    if (block_tokens > tokens) block_tokens = tokens;
    // Heads of a block: as many as give every thread a piece.
    const int groups = (tokens + block_tokens - 1) / block_tokens, slots = block_tokens * quads;
    int log2 = 0;
    while ((slots << (log2 + 1)) <= kRopeThreads && (1 << log2) < n_heads) ++log2;
    const dim3 grid(groups, (n_heads + (1 << log2) - 1) >> log2);
    const uint64_t shape = arg_pair((unsigned)half | (unsigned)quads << 10 | (unsigned)block_tokens << 17 | (unsigned)log2 << 27, head_dim);
    auto go = [&](auto kernel) {
        return launch_lean(kernel, grid, kRopeThreads, 0, stream, arg_ptr(q), arg_ptr(k), arg_ptr(v), arg_pair(tokens, n_heads), arg_pair(n_q, n_k), shape,
                           arg_pair(65536u / quads + 1, 65536u / half + 1), RopeRest(a));
    };
    return neox ? go(rope_pieces_kernel<true>) : go(rope_pieces_kernel<false>);
}

// (cos, sin) of every pair at the position *d_pos: what each thread of rope_kernel forms for
// itself, written out once for callers that rotate several rows of one token (every layer of a
// decode step rotates by the same angles).
__global__ __launch_bounds__(64) void rope_angles_kernel(float* angles, RopeFreq f, const int* d_pos, const float* freq_factors) {
#pragma clang fp contract(off)
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i >= f.n_rot / 2) return;
    const float ang = (float)*d_pos * rope_freq(i, f, freq_factors);
    sincosf(ang, &angles[2 * i + 1], &angles[2 * i]);
}

} // namespace

hipError_t rope_angles_launch(float* angles, int n_rot, float theta, const int* d_pos, const float* freq_factors,
                              hipStream_t stream) {
    drop_stale_error();
    const unsigned grid = (unsigned)((n_rot / 2 + 63) / 64);
    if (grid == 0) return hipSuccess;
    hipLaunchKernelGGL(rope_angles_kernel, dim3(grid), dim3(64), 0, stream, angles, rope_freq_plan(n_rot, theta), d_pos, freq_factors);
    return hipGetLastError();
}

bool rope_store_fused_ok(const float* q, const float* k, const float* v, const uint16_t* kc, const uint16_t* vc,
                         long long heads, int head_dim, int n_rot) {
    const uintptr_t bits = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
                           reinterpret_cast<uintptr_t>(kc) | reinterpret_cast<uintptr_t>(vc);
    return n_rot == head_dim && head_dim % 8 == 0 && head_dim / 2 <= 256 && heads <= kRopePieceHeads && (bits & 15u) == 0;
}

hipError_t rope_store_launch(float* q, float* k, const float* v, uint16_t* kc, uint16_t* vc, int tokens, int n_head,
                             int n_kv, int head_dim, int n_ctx, int n_past, float theta, const float* freq_factors,
                             bool neox, hipStream_t stream) {
    if (tokens == 0) return hipSuccess;
    RopeRest a{};
    a.kc = kc; a.vc = vc; a.freq_factors = freq_factors; a.n_past = n_past; a.n_ctx = n_ctx;
    return pieces_launch(q, k, v, a, tokens, head_dim, head_dim, theta, n_head, n_kv, n_kv, neox, stream);
}

hipError_t rope_launch(float* x, int rows, int head_dim, int n_rot, float theta, int n_past, int heads,
                       const int* d_pos, const float* freq_factors, bool neox, hipStream_t stream) {
    // batch form: rows = tokens * heads; single-token form: every row belongs to the one token
    const int tokens = d_pos ? 1 : rows / heads;
    const int heads_per_token = d_pos ? rows : heads;
    if (tokens == 0 || heads_per_token == 0) return hipSuccess;
    if (n_rot % 8 == 0 && n_rot / 2 <= 256 && head_dim % 4 == 0 && heads_per_token <= kRopePieceHeads && (reinterpret_cast<uintptr_t>(x) & 15u) == 0) {
        RopeRest a{};
        a.d_pos = d_pos; a.freq_factors = freq_factors; a.n_past = n_past;
        return pieces_launch(x, nullptr, nullptr, a, tokens, head_dim, n_rot, theta, heads_per_token, 0, 0, neox, stream);
    }
    drop_stale_error();
    const int n_hgroups = (heads_per_token + kHeadsPerThread - 1) / kHeadsPerThread;
    const long long threads = (long long)tokens * n_hgroups * (n_rot / 2);
    const unsigned grid = (unsigned)((threads + 255) / 256);
    if (grid == 0) return hipSuccess;
#define ORIN_ROPE_LAUNCH(NEOX, IND) \
    hipLaunchKernelGGL((rope_kernel<NEOX, IND>), dim3(grid), dim3(256), 0, stream, x, tokens, heads_per_token, \
                       head_dim, rope_freq_plan(n_rot, theta), n_past, d_pos, freq_factors)
    if (neox) { if (d_pos) ORIN_ROPE_LAUNCH(true, true); else ORIN_ROPE_LAUNCH(true, false); }
    else      { if (d_pos) ORIN_ROPE_LAUNCH(false, true); else ORIN_ROPE_LAUNCH(false, false); }
#undef ORIN_ROPE_LAUNCH
    return hipGetLastError();
}

} // namespace orin_fa
