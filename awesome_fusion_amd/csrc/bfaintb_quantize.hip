// Weight quantisation at load time: a float weight [n, k] (k contiguous, how a Linear keeps it) -> row-major codes
// [k, n * bits / 8] and bf16 scales [groups, n], the operands the GEMM kernels read.  Symmetric: scale = max|w| of the group
// times 1 / qmax, at least 1e-12, rounded to bf16; code = round-to-even(w / scale) clamped to [-qmax - 1, qmax], stored in
// excess form.  The reference generates its codes on the host and has no quantiser (bfAintBGemm.cc:88-103).
//
// Every weight read once (twice where a group is longer than a tile, the second time mostly from the 256 MB cache), every code written
// once.  Bound by its vector instructions, memory close behind: 11008 x 4096 bf16 -> 4-bit, groups of 128, 25 us = 4.5 TB/s (a copy
// reaches 5.2) with 0.85 of the CUs' vector issue slots used (profiles/counters_of_serving_calls.txt).  As a chain of framework operations the same work is 17 passes over fp32 copies:
// 11008 x 4096, groups of 128, 4-bit, quantised and packed: 1200 us; with this kernel and the packing one 33 us.
#include <type_traits>
#include "bfaintb_device.hpp"

namespace bfaintb {

namespace {

enum { kWeightBf16 = 0, kWeightF16 = 1, kWeightF32 = 2 };

// Eight consecutive weights of a row, as loaded.
template <int TYPE>
struct Raw8 {
    uint32_t w[TYPE == kWeightF32 ? 8 : 4];
};

template <int TYPE>
__device__ __forceinline__ Raw8<TYPE> load_raw8(const void* base, size_t element)
{
    Raw8<TYPE> r;
    const uint4* src = reinterpret_cast<const uint4*>(static_cast<const uint8_t*>(base) + element * (TYPE == kWeightF32 ? 4u : 2u));
    const uint4 a = src[0];
    r.w[0] = a.x, r.w[1] = a.y, r.w[2] = a.z, r.w[3] = a.w;
    if constexpr (TYPE == kWeightF32) {
        const uint4 b = src[1];
        r.w[4] = b.x, r.w[5] = b.y, r.w[6] = b.z, r.w[7] = b.w;
    }
    return r;
}

template <int TYPE>
__device__ __forceinline__ float raw_to_f32(const Raw8<TYPE>& r, int i)
{
    if constexpr (TYPE == kWeightF32) return __uint_as_float(r.w[i]);
    const uint32_t half = (i & 1) ? r.w[i >> 1] >> 16 : r.w[i >> 1] & 0xffffu;
    if constexpr (TYPE == kWeightBf16) return __uint_as_float(half << 16);
    return (float)__builtin_bit_cast(_Float16, (uint16_t)half);
}

typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));

// Bit pattern of the largest magnitude: with the sign cleared, the patterns of every float format are ordered as integers,
// NaNs above infinity — so a NaN weight makes its group's scale a NaN, as a floating-point maximum that keeps NaNs would.
template <int TYPE>
__device__ __forceinline__ uint32_t max_abs_bits(const Raw8<TYPE>& r)
{
    if constexpr (TYPE == kWeightF32) {
        uint32_t m = r.w[0] & 0x7fffffffu;
#pragma unroll
        for (int i = 1; i < 8; ++i) m = max(m, r.w[i] & 0x7fffffffu);
        return m;
    } else {
        u16x2_t m = __builtin_bit_cast(u16x2_t, r.w[0] & 0x7fff7fffu);
#pragma unroll
        for (int i = 1; i < 4; ++i) m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2_t, r.w[i] & 0x7fff7fffu));
        return max((uint32_t)m[0], (uint32_t)m[1]);
    }
}

template <int TYPE>
__device__ __forceinline__ float bits_to_f32(uint32_t bits)
{
    if constexpr (TYPE == kWeightF32) return __uint_as_float(bits);
    if constexpr (TYPE == kWeightBf16) return __uint_as_float(bits << 16);
    return (float)__builtin_bit_cast(_Float16, (uint16_t)bits);
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_max(uint32_t x)
{
    return max(x, (uint32_t)__builtin_amdgcn_update_dpp((int)x, (int)x, CTRL, 0xf, 0xf, false));
}

template <int BITS>
__device__ __forceinline__ uint32_t scale_bits(float max_abs)
{
    float s = max_abs * (1.0f / (BITS == 8 ? 127.0f : 7.0f));
    s = s < 1e-12f ? 1e-12f : s;  // (a NaN stays one)
    return pack_bf16_rne(s, 0.0f) & 0xffffu;
}

// w / s for 16-bit weights: the quotient by the refined reciprocal, corrected once by its own remainder.  Only where it
// rounds to matters: a quotient of an 8- or 11-bit significand by an 8-bit one is either exactly half-way between two codes
// — then the correction makes it exact — or at least 2^-20 of itself away, far more than the error left here.
__device__ __forceinline__ float quotient16(float w, float s, float r)
{
    const float q = w * r;
    return fmaf(fmaf(-q, s, w), r, q);
}

// The code is left in the low bits of 2^23 + code: adding 2^23 + excess (an even number) to the quotient rounds it to an integer, half to
// even, and puts it into the significand.  7 instructions a weight with the unpacking, where a rounding, two comparisons, a
// conversion and an addition made it 10.  (Clamped first, which changes no code: the bounds are whole numbers.  A NaN becomes the least
// code — v_med3_f32 gives the least of the other two — until the caller replaces it.)
constexpr uint32_t kMagic = 0x4b000000u;  // the bits of 2^23
template <int BITS, int TYPE>
__device__ __forceinline__ uint32_t code_in_float(float w, float s, float r)
{
    constexpr float kExcess = BITS == 8 ? 128.0f : 8.0f;
    const float q = TYPE == kWeightF32 ? w / s : quotient16(w, s, r);
    return __float_as_uint(__builtin_amdgcn_fmed3f(q, -kExcess, kExcess - 1.0f) + (8388608.0f + kExcess));
}

struct QuantizeParams {
    uint8_t* b;
    uint16_t* scale;
    const void* w;
    uint32_t n, k, ldw, ldb_bytes, group_size;  // group_size: of k rows; k itself without groups
};

constexpr uint32_t kTileK = 128, kTileBytes = 128;  // a workgroup's tile of codes: 128 rows of k, one cache line of each
constexpr uint32_t kTilePitch = kTileBytes / 4u + 1u;  // dwords: the 16 lanes that write 8 rows apart fall into different banks

// One workgroup: 128 k x 256 columns (4-bit; 128 columns for 8-bit codes), neighbours along k: they read whole rows of W between them,
// where neighbours along n would all read the same 256 bytes of rows that often lie a power of two apart, in few memory channels
// (28672 x 4096 4-bit g64 72 us so, 60 now; 11008 x 4096 4-bit g128 30.4 and 26.1, 4.3 TB/s; only 8-bit codes whose scales were made
// before, and whose weights come from the cache therefore, are 2 % faster along n: 11008 x 4096 41.5 / 42.4).  A lane holds 8 consecutive k of as many rows of
// W as a dword holds codes, so that it makes whole dwords of the output's rows; the tile is turned through LDS and leaves
// in full 128-byte lines.  FUSED: groups lie within the tile (32, 64 or 128 weights = 4, 8 or 16 lanes) and the scales
// are made here, over the row of lanes; otherwise they have been made by scale_kernel.
template <int BITS, int TYPE, bool FUSED>
__global__ void __launch_bounds__(512) bfaintb_quantize_kernel(const QuantizeParams p)
{
    constexpr uint32_t kRows = 32u / BITS;  // rows of W per lane
    constexpr uint32_t kCode0 = BITS == 8 ? 0x80808080u : 0x88888888u;  // a group without a finite scale (a NaN or an infinity among its weights)
    __shared__ uint32_t tile[kTileK * kTilePitch];
    constexpr bool kAlongK = FUSED || BITS == 4;
    const uint32_t fast = kAlongK ? (p.k + kTileK - 1u) / kTileK : (p.n + 32u * kRows - 1u) / (32u * kRows);  // tiles of the direction that neighbours walk
    const uint32_t slow_tile = blockIdx.x / fast, fast_tile = blockIdx.x - slow_tile * fast;
    const uint32_t tile_k = kAlongK ? fast_tile : slow_tile, tile_n = kAlongK ? slow_tile : fast_tile;
    const uint32_t kq = threadIdx.x & 15u, ng = threadIdx.x >> 4;
    const uint32_t k0 = tile_k * kTileK + 8u * kq, n0 = (tile_n * 32u + ng) * kRows;
    if (k0 < p.k && n0 < p.n) {  // (whole groups of lanes: n is a multiple of kRows, and k of 8 and of the group)
        Raw8<TYPE> raw[kRows];
#pragma unroll
        for (uint32_t r = 0; r < kRows; ++r) raw[r] = load_raw8<TYPE>(p.w, (size_t)(n0 + r) * p.ldw + k0);
        uint32_t sb[kRows];
        uint32_t* scales = reinterpret_cast<uint32_t*>(p.scale + (size_t)(k0 / p.group_size) * p.n + n0);
        if constexpr (FUSED) {
#pragma unroll
            for (uint32_t r = 0; r < kRows; ++r) {
                uint32_t m = max_abs_bits(raw[r]);
                m = dpp_max<0xB1>(m);   // quad_perm 1,0,3,2
                m = dpp_max<0x4E>(m);   // quad_perm 2,3,0,1
                if (p.group_size >= 64u) m = dpp_max<0x141>(m);   // row_half_mirror: the two quads of 8 lanes
                if (p.group_size >= 128u) m = dpp_max<0x140>(m);  // row_mirror: the two halves of 16
                sb[r] = scale_bits<BITS>(bits_to_f32<TYPE>(m));
            }
            if (k0 % p.group_size == 0u) {
#pragma unroll
                for (uint32_t r = 0; r < kRows; r += 2) scales[r >> 1] = sb[r] | (sb[r + 1] << 16);
            }
        } else {
#pragma unroll
            for (uint32_t r = 0; r < kRows; r += 2) {
                const uint32_t two = scales[r >> 1];
                sb[r] = two & 0xffffu, sb[r + 1] = two >> 16;
            }
        }
        uint32_t out[8], finite = 0u;  // (finite: all bits of the rows whose scale is)
        constexpr uint32_t kMagics = BITS == 8 ? kMagic : (uint32_t)(kMagic * 0x11111111ull);  // what the 2^23s of all rows add up to
#pragma unroll
        for (int i = 0; i < 8; ++i) out[i] = 0u - kMagics;
#pragma unroll
        for (uint32_t r = 0; r < kRows; ++r) {
            const float s = bf16_bits_to_f32(sb[r]);
            finite |= (sb[r] & 0x7f80u) != 0x7f80u ? ((1u << BITS) - 1u) << (BITS * r) : 0u;
            float rcp = __builtin_amdgcn_rcpf(s);
            rcp = fmaf(fmaf(-s, rcp, 1.0f), rcp, rcp);
#pragma unroll
            for (int i = 0; i < 8; ++i) out[i] += code_in_float<BITS, TYPE>(raw_to_f32(raw[r], i), s, rcp) << (BITS * r);
        }
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) tile[(8u * kq + i) * kTilePitch + ng] = (out[i] & finite) | (kCode0 & ~finite);
    }
    __syncthreads();
    // 16 lanes x 8 bytes = one row's line
    const uint32_t row_bytes = p.n * BITS / 8u, col = tile_n * kTileBytes + 8u * kq;
    if (col >= row_bytes) return;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t kr = 32u * i + ng, row = tile_k * kTileK + kr;
        if (row >= p.k) break;
        const uint32_t* src = tile + kr * kTilePitch + 2u * kq;
        *reinterpret_cast<uint2*>(p.b + (size_t)row * p.ldb_bytes + col) = make_uint2(src[0], src[1]);
    }
}

// One wave per row and group: the group's scale.  Four 16-byte loads in flight per lane.
template <int BITS, int TYPE>
__global__ void __launch_bounds__(256) bfaintb_scale_kernel(const QuantizeParams p)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t row = blockIdx.x * 4u + (threadIdx.x >> 6), g = blockIdx.y;
    if (row >= p.n) return;
    const size_t first = (size_t)row * p.ldw + (size_t)g * p.group_size;
    uint32_t m = 0;
    uint32_t i = 8u * lane;
    for (; i + 3u * 512u < p.group_size; i += 4u * 512u) {
        Raw8<TYPE> raw[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) raw[u] = load_raw8<TYPE>(p.w, first + i + 512u * u);
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) m = max(m, max_abs_bits(raw[u]));
    }
    for (; i < p.group_size; i += 512u) m = max(m, max_abs_bits(load_raw8<TYPE>(p.w, first + i)));
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, d));
    if (lane == 0u) p.scale[(size_t)g * p.n + row] = (uint16_t)scale_bits<BITS>(bits_to_f32<TYPE>(m));
}

template <int BITS, int TYPE>
hipError_t launch_quantize_t(const QuantizeParams& p, hipStream_t stream)
{
    constexpr uint32_t kCols = 32u * (32u / BITS);
    const dim3 grid(((p.k + kTileK - 1u) / kTileK) * ((p.n + kCols - 1u) / kCols), 1, 1);
    // groups of 32, 64 or 128 lie within one tile, and within one row of 16 lanes
    if (p.group_size == 32u || p.group_size == 64u || p.group_size == 128u)
        return launch_kernel(bfaintb_quantize_kernel<BITS, TYPE, true>, grid, dim3(512, 1, 1), 0, stream, p);
    const hipError_t e = launch_kernel(bfaintb_scale_kernel<BITS, TYPE>, dim3((p.n + 3u) / 4u, p.k / p.group_size, 1), dim3(256, 1, 1), 0, stream, p);
    if (e != hipSuccess) return e;
    return launch_kernel(bfaintb_quantize_kernel<BITS, TYPE, false>, grid, dim3(512, 1, 1), 0, stream, p);
}

template <int BITS>
hipError_t launch_quantize_b(const QuantizeParams& p, int type, hipStream_t stream)
{
    if (type == kWeightBf16) return launch_quantize_t<BITS, kWeightBf16>(p, stream);
    if (type == kWeightF16) return launch_quantize_t<BITS, kWeightF16>(p, stream);
    return launch_quantize_t<BITS, kWeightF32>(p, stream);
}

}  // namespace

hipError_t launch_quantize(uint8_t* b, uint16_t* scale, const void* w, int type, uint32_t n, uint32_t k, uint32_t ldw, uint32_t ldb_bytes,
                           int bits, uint32_t group_size, hipStream_t stream)
{
    const QuantizeParams p{b, scale, w, n, k, ldw, ldb_bytes, group_size ? group_size : k};
    return bits == 8 ? launch_quantize_b<8>(p, type, stream) : launch_quantize_b<4>(p, type, stream);
}

}  // namespace bfaintb
