// Dequantised-weight dump: W[k,n] = bf16(float(q) * float(scale)) written to memory, through the device routines of the
// conversion (codes*_to_s8*, sbyte_to_f32, make_col_scale, pack_bf16_rne).  The GEMM kernels that make their weights by halves
// (bfaintb_device.hpp) come to the same weights but for the sign of a zero; products with one-hot rows hold them against this dump.
// Successor of the reference's ASM_PRINT channel (/root/reference/bfAintBGemm/bfAintBGemm.cc:113-118,
// 156-169; bf16gemm_kernel_gfx90a.s:2-16): the way to look at in-kernel dequantised values.
#include "bfaintb_device.hpp"

namespace bfaintb {

struct DequantParams {
    uint16_t* w;
    const uint8_t* b;
    const uint16_t* scale;
    uint32_t n, k, ldb_bytes, ldw, lds, group_size;
};

// One thread: 4 consecutive columns of 2 consecutive rows (so that cvt_pk pairs are rows, as in
// the GEMM kernels).
template <int BITS>
__global__ void __launch_bounds__(256) bfaintb_dequant_kernel(const DequantParams p)
{
    const uint32_t col = (blockIdx.x * 256u + threadIdx.x) * 4u;
    const uint32_t row = blockIdx.y * 2u;
    if (col >= p.n) return;
    uint32_t x[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const uint8_t* src = p.b + (size_t)(row + r) * p.ldb_bytes + (BITS == 8 ? col : col / 2);
        if constexpr (BITS == 8) x[r] = *reinterpret_cast<const uint32_t*>(src);
        else x[r] = *reinterpret_cast<const uint16_t*>(src);
    }
    uint32_t y[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        if constexpr (BITS == 8) {
            y[r] = codes8_to_s8(x[r]);
        } else {
            y[r] = codes4_quad_to_s8x16(x[r]);
        }
    }
    const uint32_t g = p.group_size ? row / p.group_size : 0u;  // group_size is even: both rows share a group
    const uint2 sr = *reinterpret_cast<const uint2*>(p.scale + (size_t)g * p.lds + col);
    const float cs[4] = {make_col_scale<BITS>(sr.x & 0xffffu), make_col_scale<BITS>(sr.x >> 16),
                         make_col_scale<BITS>(sr.y & 0xffffu), make_col_scale<BITS>(sr.y >> 16)};
    uint32_t pk[4];
    pk[0] = pack_bf16_rne(sbyte_to_f32<0>(y[0]) * cs[0], sbyte_to_f32<0>(y[1]) * cs[0]);
    pk[1] = pack_bf16_rne(sbyte_to_f32<1>(y[0]) * cs[1], sbyte_to_f32<1>(y[1]) * cs[1]);
    pk[2] = pack_bf16_rne(sbyte_to_f32<2>(y[0]) * cs[2], sbyte_to_f32<2>(y[1]) * cs[2]);
    pk[3] = pack_bf16_rne(sbyte_to_f32<3>(y[0]) * cs[3], sbyte_to_f32<3>(y[1]) * cs[3]);
    // row `row`: low halves; row+1: high halves
    uint2 o0, o1;
    o0.x = (pk[0] & 0xffffu) | (pk[1] << 16);
    o0.y = (pk[2] & 0xffffu) | (pk[3] << 16);
    o1.x = (pk[0] >> 16) | (pk[1] & 0xffff0000u);
    o1.y = (pk[2] >> 16) | (pk[3] & 0xffff0000u);
    *reinterpret_cast<uint2*>(p.w + (size_t)row * p.ldw + col) = o0;
    *reinterpret_cast<uint2*>(p.w + (size_t)(row + 1) * p.ldw + col) = o1;
}

hipError_t launch_dequant(uint16_t* w, const uint8_t* b, const uint16_t* scale, uint32_t n, uint32_t k, uint32_t ldb_bytes,
                          uint32_t ldw, int bits, uint32_t group_size, hipStream_t stream)
{
    DequantParams p{w, b, scale, n, k, ldb_bytes, ldw, n, group_size};
    const dim3 grid((n / 4u + 255u) / 256u, k / 2u, 1);
    if (bits == 8) return launch_kernel(bfaintb_dequant_kernel<8>, grid, dim3(256, 1, 1), 0, stream, p);
    return launch_kernel(bfaintb_dequant_kernel<4>, grid, dim3(256, 1, 1), 0, stream, p);
}

__global__ void __launch_bounds__(256) bfaintb_fill_u32_kernel(uint32_t* dst, uint32_t count, uint32_t value)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < count) dst[i] = value;
}

// Measurement aid: reads `n16` 16-byte words with the widest coalesced loads (a wave reads 8 KiB in
// 8 loads issued back to back) and throws them away.  Its time is what this GPU needs merely to
// fetch that many bytes in one kernel launch: the practical ceiling for a weight-streaming GEMV.
__global__ void __launch_bounds__(256) bfaintb_probe_read_kernel(const uint4* __restrict__ src, uint32_t* sink, size_t n16)
{
    const size_t wave = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const size_t base = wave * 512 + (threadIdx.x & 63);
    uint4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const size_t idx = base + (size_t)i * 64;
        v[i] = idx < n16 ? src[idx] : make_uint4(0, 0, 0, 0);
    }
    uint32_t x = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) x ^= v[i].x ^ v[i].y ^ v[i].z ^ v[i].w;
    if (x == 0x9e3779b9u && sink != nullptr) sink[threadIdx.x & 63] = x;  // practically never: keeps the loads alive
}

hipError_t launch_probe_read(const void* src, size_t bytes, void* sink, hipStream_t stream)
{
    const size_t n16 = bytes / 16;
    const size_t waves = (n16 + 511) / 512;
    const uint32_t grid = (uint32_t)((waves + 3) / 4);
    return launch_kernel(bfaintb_probe_read_kernel, dim3(grid, 1, 1), dim3(256, 1, 1), 0, stream, static_cast<const uint4*>(src),
                         static_cast<uint32_t*>(sink), n16);
}

hipError_t launch_fill_u32(uint32_t* dst, uint32_t count, uint32_t value, hipStream_t stream)
{
    return launch_kernel(bfaintb_fill_u32_kernel, dim3((count + 255u) / 256u, 1, 1), dim3(256, 1, 1), 0, stream, dst, count, value);
}

}  // namespace bfaintb
