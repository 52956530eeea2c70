// The two mutators of the fp16 KV cache for gfx950 (MI355X): the fp32 -> fp16 row store that
// runs right before attention, and the rolling-window shift.
//
// Replaces the reference's kv_store_k / kv_shift_k and their wrappers (reference:
// src/kernels.cu:1659-1700, 2079-2093; CPU statement of the same operations:
// src/model_cpu.cpp:276-279, 321-338).  Cache layout as everywhere: element (head, pos, i) of
// one layer at (head * n_ctx + pos) * head_dim + i, fp16 bit patterns in uint16_t; the whole
// cache is n_layer such blocks for K, and the same again for V.
//
// Both are pure byte movers, bound by HBM:
//   * store: one thread converts 8 consecutive fp32 values (two 16-byte loads) with
//     round-to-nearest-even and writes one 16-byte piece of a cache row; K and V are handled
//     by the two halves of the grid.  The reference launches one 256-thread block per row with
//     2-byte stores.  The "ind" form reads the position on the device, so the launch can be
//     captured in a graph.
//   * shift: rows [n_keep + shift, n_ctx) move down by `shift` rows and the last `shift` rows are
//     cleared, in place.  Row p only ever takes the value of row p + shift, so the rows of one
//     residue class (p - n_keep) mod shift form a chain that one thread walks front to back
//     (load p + shift, store p), and different chains never touch the same bytes: the grid is
//     one thread per 16-byte piece of every chain head -- (layers x {K,V} x heads x shift rows x
//     head_dim/8) threads, every access a full coalesced row -- where the reference walks each
//     column of a head with a single thread.
#include "fa_common.hpp"

namespace orin_fa {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));

// VEC = 8: head_dim is a multiple of 8 (16-byte cache pieces); VEC = 1: any head_dim.  A launch has fewer than 2^31 threads, so
// that its divisions are 32-bit ones (64-bit: some 500 instructions ahead of the first load); its arguments are few (launch_lean())
// and in registers when a wave starts (kernel-argument preload).  Bound by the launch: 301 tokens of Llama-3.2-1B 2.25 -> 2.2 us.
//   shape   heads | head_dim << 32        rows   n_ctx | pos_base << 32        pos_or_batch   the position's address, or the tokens
template <int VEC, bool IND>
__global__ __launch_bounds__(256) void kv_store_kernel(const uint64_t kc_bits, const uint64_t vc_bits, const uint64_t k_bits, const uint64_t v_bits,
                                                       const uint64_t shape, const uint64_t rows, const uint64_t pos_or_batch) {
    uint16_t *const kc = ptr_arg<uint16_t>(kc_bits), *const vc = ptr_arg<uint16_t>(vc_bits);
    const float *const k = ptr_arg<const float>(k_bits), *const v = ptr_arg<const float>(v_bits);
    const int* const d_pos = ptr_arg<const int>(IND ? pos_or_batch : 0);
    const unsigned batch = IND ? 1u : (unsigned)pos_or_batch;
    const unsigned heads = (unsigned)shape, head_dim = (unsigned)(shape >> 32);
    const int n_ctx = (int)(unsigned)rows, pos_base = (int)(rows >> 32);
    const unsigned per_row = head_dim / VEC;                  // threads per (token, head) row
    const unsigned half = batch * heads * per_row;
    const unsigned idx = blockIdx.x * 256 + threadIdx.x;
    const bool is_v = idx >= half;                            // second half of the grid stores V
    const unsigned j = is_v ? idx - half : idx;
    if (j >= half) return;
    const unsigned row = j / per_row, piece = j - row * per_row; // row = token * heads + head
    const unsigned token = row / heads, head = row - token * heads;
    const int pos = IND ? *d_pos : pos_base + (int)token;
    if (pos < 0 || pos >= n_ctx) return;                      // (the reference would write out of bounds)
    const float* src = (is_v ? v : k) + (size_t)row * head_dim + piece * VEC;
    uint16_t* dst = (is_v ? vc : kc) + ((size_t)head * n_ctx + pos) * head_dim + piece * VEC;
    if constexpr (VEC == 8) {
        const float4 x0 = *reinterpret_cast<const float4*>(src);
        const float4 x1 = *reinterpret_cast<const float4*>(src + 4);
        half8 h;
        h[0] = (_Float16)x0.x; h[1] = (_Float16)x0.y; h[2] = (_Float16)x0.z; h[3] = (_Float16)x0.w;
        h[4] = (_Float16)x1.x; h[5] = (_Float16)x1.y; h[6] = (_Float16)x1.z; h[7] = (_Float16)x1.w;
        // (An ordinary store: the attention of the same chunk reads these rows next, once per query tile and head group, and
        // finds them in the last-level cache.  With streaming stores, this launch and the attention behind it: 45 tokens of
        // Llama-3-8B 6.5 us for 6.3, 512 of Qwen2.5-1.5B at the start of a sequence 10.6 for 9.8, at 4096 27.0 for 26.6;
        // 301 of Llama-3.2-1B at 1501 14.3 for 14.5.)
        *reinterpret_cast<half8*>(dst) = h;
    } else {
        const _Float16 h = (_Float16)src[0];
        dst[0] = __builtin_bit_cast(uint16_t, h);
    }
}

// One thread per 16-byte piece of a chain head.  PIECE = bytes per thread (16, or 2 when
// head_dim is not a multiple of 8).
template <int PIECE>
__global__ __launch_bounds__(256) void kv_shift_kernel(uint16_t* kc, uint16_t* vc, long long strips, int row_bytes,
                                                       int n_ctx, int n_keep, int shift) {
    typedef unsigned piece_t __attribute__((ext_vector_type(PIECE == 16 ? 4 : 1)));
    const int per_row = row_bytes / PIECE;
    const long long per_strip = (long long)shift * per_row;   // chain heads of one (layer, head) strip, times pieces
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
    const bool is_v = idx >= strips * per_strip;
    const long long j = is_v ? idx - strips * per_strip : idx;
    if (j >= strips * per_strip) return;
    const long long strip = j / per_strip;                    // = layer * n_kv + head
    const int rem = (int)(j % per_strip);
    const int residue = rem / per_row, piece = rem % per_row;
    unsigned char* base = reinterpret_cast<unsigned char*>(is_v ? vc : kc) + (size_t)strip * n_ctx * row_bytes +
                          (size_t)piece * PIECE;
    int p = n_keep + residue;
    if (p >= n_ctx) return;
    for (; p + shift < n_ctx; p += shift) {
        if constexpr (PIECE == 16) {
            const piece_t x = *reinterpret_cast<const piece_t*>(base + (size_t)(p + shift) * row_bytes);
            __builtin_nontemporal_store(x, reinterpret_cast<piece_t*>(base + (size_t)p * row_bytes));
        } else {
            const uint16_t x = *reinterpret_cast<const uint16_t*>(base + (size_t)(p + shift) * row_bytes);
            *reinterpret_cast<uint16_t*>(base + (size_t)p * row_bytes) = x;
        }
    }
    // p is now the chain's row in the last `shift` rows: cleared
    if constexpr (PIECE == 16) *reinterpret_cast<piece_t*>(base + (size_t)p * row_bytes) = piece_t{0u, 0u, 0u, 0u};
    else *reinterpret_cast<uint16_t*>(base + (size_t)p * row_bytes) = 0;
}

} // namespace

hipError_t kv_store_launch(uint16_t* kc, uint16_t* vc, const float* k, const float* v, int heads, int head_dim,
                           int n_ctx, int pos_base, int batch, const int* d_pos, hipStream_t stream) {
    const bool vec = head_dim % 8 == 0 &&
                     ((reinterpret_cast<uintptr_t>(kc) | reinterpret_cast<uintptr_t>(vc) |
                       reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v)) & 15u) == 0;
    const long long per_token = 2ll * heads * (head_dim / (vec ? 8 : 1)); // threads
    if (per_token > 0x7fffff00ll) return hipErrorInvalidValue;
    const int most = (int)(0x7fffff00ll / per_token); // tokens of a launch
    for (int t = 0; t < batch; t += most) { // (batch = 1 with a position on the device)
        const int n = batch - t < most ? batch - t : most;
        auto go = [&](auto kernel) {
            return launch_lean(kernel, dim3((unsigned)((per_token * n + 255) / 256)), 256, 0, stream, arg_ptr(kc), arg_ptr(vc), arg_ptr(k + (size_t)t * heads * head_dim),
                               arg_ptr(v + (size_t)t * heads * head_dim), arg_pair(heads, head_dim), arg_pair(n_ctx, pos_base + t), d_pos ? arg_ptr(d_pos) : (uint64_t)n);
        };
        const hipError_t e = vec ? (d_pos ? go(kv_store_kernel<8, true>) : go(kv_store_kernel<8, false>))
                                 : (d_pos ? go(kv_store_kernel<1, true>) : go(kv_store_kernel<1, false>));
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t kv_shift_launch(uint16_t* kc, uint16_t* vc, int n_layer, int n_kv, int head_dim, int n_ctx, int n_keep,
                           int shift, hipStream_t stream) {
    drop_stale_error();
    const int row_bytes = head_dim * 2;
    const bool vec = row_bytes % 16 == 0 &&
                     ((reinterpret_cast<uintptr_t>(kc) | reinterpret_cast<uintptr_t>(vc)) & 15u) == 0;
    const long long strips = (long long)n_layer * n_kv;
    const long long threads = 2ll * strips * shift * (row_bytes / (vec ? 16 : 2));
    const long long blocks = (threads + 255) / 256;
    if (blocks == 0) return hipSuccess;
    if (blocks > 0x7fffffffll) return hipErrorInvalidValue;
    if (vec) hipLaunchKernelGGL((kv_shift_kernel<16>), dim3((unsigned)blocks), dim3(256), 0, stream, kc, vc, strips, row_bytes, n_ctx, n_keep, shift);
    else hipLaunchKernelGGL((kv_shift_kernel<2>), dim3((unsigned)blocks), dim3(256), 0, stream, kc, vc, strips, row_bytes, n_ctx, n_keep, shift);
    return hipGetLastError();
}

} // namespace orin_fa
