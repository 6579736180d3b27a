// dequant.hip -- IQ4_XS super-blocks -> fp32 weights on gfx950.
//
// Semantics (kernels/demo_iq4xs_dequant/ref_cpu.cpp:6-27, impl.hip:14-48):
//   dl = fp16(d) * (float(ls) - 32)             (exact in fp32)
//   y[32*ib + j]      = dl * float(kvalues_iq4nl[qs[16*ib + j] & 15])
//   y[32*ib + j + 16] = dl * float(kvalues_iq4nl[qs[16*ib + j] >> 4])
// Two IEEE fp32 multiplies per output, no contraction possible, so the
// outputs are bit-identical to the reference's CPU dequantiser.
//
// MI355X mapping.  The op moves 136 bytes in and 1024 bytes out per
// super-block: it is bound by HBM writes, so every store instruction writes
// whole 128-byte lines.  8 lanes share a pair of sub-blocks (2g, 2g + 1): lane
// c (+ 4) takes qs dword c of both, the low (high) nibbles, so one 16-byte
// store of the 8 lanes is sub-block 2g in output order and the next 2g + 1;
// 32 threads share a super-block and read its 8-byte header.  (One lane for
// both nibbles wrote 16-byte pieces 32 bytes apart: 5120 x 17408 in 75.0 us,
// whole lines 68.7.)  Codes are decoded with the GEMV's v_perm tables
// (decode_codes_x), one nibble at a time.
//
// An output too large to stay in the 256 MB Infinity Cache is written with
// nontemporal stores: 56.0 us for 5120 x 17408 (340 MiB of output, the 45 MiB
// of weights in the cache between passes; a device fill of that size takes
// 53.1), 42.5 against 51.7 plain for 256 MiB.  Smaller ones are written with
// plain stores, which leave them in the cache for their reader and take as
// long where one buffer is written again and again (192 MiB 33.2 us plain,
// 32.8 nontemporal; 128 MiB 23.0, 23.3); over several buffers nontemporal ones
// would be faster on their own (192 MiB 39.7 plain, 32.4).
#include "dequant_plan.h"
#include "iq4xs_device.h"
#include "iq4xs_internal.h"

namespace iq4xs {

template <bool kStream>
__global__ __launch_bounds__(DEQUANT_WG) void dequant_iq4xs_kernel(const uint8_t* __restrict__ src, float* __restrict__ dst,
                                                            int64_t n_blocks) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    static_assert(DEQUANT_THREADS == 32, "t & 31 is the thread's part of its super-block");
    const int64_t b = t >> 5;
    if (b >= n_blocks) return;
    const int p = (int)(t & 31), g = p >> 3, c = p & 3, shift = p & 4;  // sub-block pair, qs dword, nibble
    const uint8_t* blk = src + b * BLOCK_BYTES;
    const v2u hd = *reinterpret_cast<const v2u*>(blk);
    const uint32_t q0 = *reinterpret_cast<const uint32_t*>(blk + 8 + 32 * g + 4 * c);
    const uint32_t q1 = *reinterpret_cast<const uint32_t*>(blk + 24 + 32 * g + 4 * c);
    const float d = half_bits_to_float(hd.x & 0xFFFFu);
    const float d0 = d * (float)(subblock_ls(hd.x, hd.y, 2 * g) - 32);
    const float d1 = d * (float)(subblock_ls(hd.x, hd.y, 2 * g + 1) - 32);
    const uint32_t k0 = decode_nibbles_x((q0 >> shift) & 0x0F0F0F0Fu);
    const uint32_t k1 = decode_nibbles_x((q1 >> shift) & 0x0F0F0F0Fu);
    v4f y0, y1;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        y0[k] = d0 * (float)(int8_t)(k0 >> (8 * k));
        y1[k] = d1 * (float)(int8_t)(k1 >> (8 * k));
    }
    v4f* y = reinterpret_cast<v4f*>(dst + b * QK_K + 64 * g) + (p & 7);
    if constexpr (kStream) {
        __builtin_nontemporal_store(y0, y);
        __builtin_nontemporal_store(y1, y + 8);
    } else {
        y[0] = y0;
        y[8] = y1;
    }
}

hipError_t launch_dequant(const uint8_t* src, float* dst, int64_t n_blocks, hipStream_t stream) {
    clear_launch_error();
    constexpr int64_t kCached = 192 * 1024;  // super-blocks of 1 KB of output: 192 MiB
    const bool stream_out = n_blocks > kCached;
    for (int64_t done = 0; done < n_blocks;) {
        const int64_t n = dequant_chunk(n_blocks - done);
        const dim3 grid((unsigned)((n * DEQUANT_THREADS + DEQUANT_WG - 1) / DEQUANT_WG)), block(DEQUANT_WG);
        const uint8_t* s = src + done * BLOCK_BYTES;
        float* d = dst + done * QK_K;
        if (stream_out)
            hipLaunchKernelGGL(dequant_iq4xs_kernel<true>, grid, block, 0, stream, s, d, n);
        else
            hipLaunchKernelGGL(dequant_iq4xs_kernel<false>, grid, block, 0, stream, s, d, n);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        done += n;
    }
    return hipSuccess;
}

}  // namespace iq4xs
