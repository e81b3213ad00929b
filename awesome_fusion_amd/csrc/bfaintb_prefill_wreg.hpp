// Tiled variant, tiles of 128 to 256 rows x 256 columns, weights kept in registers: the prefill kernel, for row-major B and for B in the packed order
// (PACKED: what changes is said where the codes are fetched).
//
// Same job and the same reference kernel replaced as bfaintb_prefill_kernel
// (/root/reference/bfAintBGemm/bf16gemm_kernel_gfx90a.s:184-630).  That kernel stages both operands in LDS and is bound
// by LDS traffic as much as by the matrix pipe (per K-step a CU reads 192 KiB and writes 64 KiB of LDS).  Here W never is in LDS, only
// A and, of weights in rows, the codes:
//   256 threads = 4 waves side by side along n; a wave owns ALL 16 MT rows x 64 columns of the tile, i.e. MT x 4 accumulators of
//   v_mfma_f32_16x16x32_bf16 (MT = 16: 256 accumulator registers, one wave per SIMD, the whole register file).
//   Because a wave owns its 64 columns outright, it converts exactly the weights it multiplies by, straight into the
//   matrix instruction's operand registers: no W tile in LDS, no duplicate conversion, no LDS writes by the waves at all.
//   Lane (c16 = lane % 16, kq = lane / 16) has, per block of 32 k, rows 8 kq .. 8 kq + 7 of the wave's columns 16 j + c16, j = 0 .. 3: the layout
//   v_mfma_f32_16x16x32_bf16 wants.
//   A: global -> LDS directly (buffer_load ... lds), three stages of 16 MT rows x 64 k, rows of 128 bytes in 8
//   chunks of 16, chunk c of row r at position c ^ ((r >> 1) & 7); a fragment read is one ds_read_b128 (16 rows x 32 k).
//   Codes in rows: the same way, three stages, read by transposing reads (ds_read_b64_tr_b8 / _b4).  Packed codes lie as the lanes need them and
//   are loaded straight to registers.  Group scales: through LDS.
// Accumulator (mt, j), register r of lane (c16, q = lane / 16): row 16 mt + 4 q + r, column 64 w + 16 j + c16 of the tile.
//
// What bounds it: on a full machine the board's power (1.4 kW: the clock gives way to 1.9 GHz); below that what one wave a SIMD issues in order.
// Measured by switching parts off, cycles a step of 16 blocks (2048 of them the matrix pipe's): the bare loop 2110; LDS reads 70; one
// vector instruction in every slot some 1, a second one in a slot 8; a memory request 7 if the step's are spread evenly, 17 to 33 one behind the other
// (four waves make theirs at the same time, and a copy of 16 bytes a lane takes the memory path 16 cycles).  Hence
//   - few vector instructions, one a slot: the conversion by halves (128 a step for 8-bit codes, 168 for 4-bit ones with group scales; a
//     conversion, a multiplication and half a pack were 194 and 250), every one held in the slot it is written for;
//   - few requests, spread over the step: codes in rows through LDS, 4 or 2 copies a wave and step (16 loads of a dword or less before);
//   - waits that cover many registers at once.
// Cycles a step, 8-bit codes in rows, one scale a column / 4-bit, groups of 128: 2632 / 3070 with a conversion, a multiplication and half a pack; 2380
// to 2430 / 2585 to 2640 now with 16 blocks, 1790 to 1830 / 1930 to 1980 with 10, 1570 to 1600 / 1705 to 1745 with 8.  us, before / now, both on one
// card in turn, weights cold: 4096 x 4096 x 4096 8-bit in rows 103.7 / 101.7, packed 103.5 / 99.3, 4-bit g128 109.6 / 102.9, packed 111.0 / 102.5;
// 2048 x 28672 x 8192 4-bit g128 775 / 726, packed 742 / 714.
// Fewer blocks: rows spread evenly over the tiles (wide_tiles in bfaintb_capi.hip), so that no matrix instruction is spent on rows
// that do not exist and the tiles make whole rounds.  us, before there were fewer than 16 / now, as above: 384 x 22016 x 4096 4-bit g128 102.1 / 71.3, 8-bit
// 85.7 / 69.6; 300 x 28672 x 4096 4-bit 91.1 / 74.0, packed 84.4 / 74.3; 577 x 13824 x 5120 packed 4-bit 95.6 / 83.5, 8-bit 96.8 / 78.6; 768 rows
// packed 4-bit 116.2 / 96.6; 2560 x 4096 x 4096 4-bit g128 100.4 / 75.1.
// The thin last round of the 256x256 tiles runs as halves of 128 x 256, eight blocks, and not of 256 x 128 (bfaintb_prefill256x128_wreg_kernel): the same
// conversions and fragment reads for the same matrix instructions, but 24 KiB copied a step instead of 36 and no weight converted twice.  us, 256 x 128 / 128 x
// 256: 2048 x 28672 x 8192 4-bit g128 730 / 711, packed 719 / 712, 8-bit 713 / 699; 2727 x 31312 x 2816 packed 4-bit 406 / 402.
#pragma once
#include <utility>
#include "bfaintb_device.hpp"
#include "bfaintb_prefill_wreg_step.hpp"

namespace bfaintb {

namespace {
constexpr uint32_t kWrTile = 256, kWrK = 64;
constexpr uint32_t kWrCRowBytes = 256 * 2;     // epilogue staging row

__device__ __forceinline__ uint32_t wr_swz(uint32_t row, uint32_t chunk) { return row * 128u + ((chunk ^ ((row >> 1) & 7u)) << 4); }

// The accumulators are the accumulation registers a[0 : 16 MT - 1], by name: accumulator (mt, j) is the four from 16 mt + 4 j on.  The
// compiler knows of them only that the kernel uses them (acc_reserve, at the start and the end of every path), and has no other use for them as
// long as it does not run out of its 256 ordinary registers; tests/test_compiled_tiles.py looks whether it had.  Given to it as variables, it keeps part
// of 256 of them in ordinary registers and shuttles them back and forth around every matrix instruction, or, as in-out operands of the assembly, moves
// some where paths through the kernel meet.  What its hazard bookkeeping cannot see behind the assembly is kept safe by construction: the operands a and b are written
// (LDS reads, conversions) long before, under waits for LDS; the accumulators are read only in the epilogue, behind explicit idle cycles
// (acc_settle) that cover a matrix instruction's write latency.
template <int MT>
__device__ __forceinline__ void acc_reserve()
{
    if constexpr (MT > 0) asm volatile("" ::: "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", "a10", "a11", "a12", "a13", "a14", "a15", "a16", "a17", "a18", "a19", "a20", "a21", "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", "a30", "a31");
    if constexpr (MT > 2) asm volatile("" ::: "a32", "a33", "a34", "a35", "a36", "a37", "a38", "a39", "a40", "a41", "a42", "a43", "a44", "a45", "a46", "a47", "a48", "a49", "a50", "a51", "a52", "a53", "a54", "a55", "a56", "a57", "a58", "a59", "a60", "a61", "a62", "a63");
    if constexpr (MT > 4) asm volatile("" ::: "a64", "a65", "a66", "a67", "a68", "a69", "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79", "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", "a88", "a89", "a90", "a91", "a92", "a93", "a94", "a95");
    if constexpr (MT > 6) asm volatile("" ::: "a96", "a97", "a98", "a99", "a100", "a101", "a102", "a103", "a104", "a105", "a106", "a107", "a108", "a109", "a110", "a111", "a112", "a113", "a114", "a115", "a116", "a117", "a118", "a119", "a120", "a121", "a122", "a123", "a124", "a125", "a126", "a127");
    if constexpr (MT > 8) asm volatile("" ::: "a128", "a129", "a130", "a131", "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", "a140", "a141", "a142", "a143", "a144", "a145", "a146", "a147", "a148", "a149", "a150", "a151", "a152", "a153", "a154", "a155", "a156", "a157", "a158", "a159");
    if constexpr (MT > 10) asm volatile("" ::: "a160", "a161", "a162", "a163", "a164", "a165", "a166", "a167", "a168", "a169", "a170", "a171", "a172", "a173", "a174", "a175", "a176", "a177", "a178", "a179", "a180", "a181", "a182", "a183", "a184", "a185", "a186", "a187", "a188", "a189", "a190", "a191");
    if constexpr (MT > 12) asm volatile("" ::: "a192", "a193", "a194", "a195", "a196", "a197", "a198", "a199", "a200", "a201", "a202", "a203", "a204", "a205", "a206", "a207", "a208", "a209", "a210", "a211", "a212", "a213", "a214", "a215", "a216", "a217", "a218", "a219", "a220", "a221", "a222", "a223");
    if constexpr (MT > 14) asm volatile("" ::: "a224", "a225", "a226", "a227", "a228", "a229", "a230", "a231", "a232", "a233", "a234", "a235", "a236", "a237", "a238", "a239", "a240", "a241", "a242", "a243", "a244", "a245", "a246", "a247", "a248", "a249", "a250", "a251", "a252", "a253", "a254", "a255");
}
template <uint32_t ACC>
__device__ __forceinline__ void mfma16(const bf16x8_t& a, const bf16x8_t& b)
{
    asm volatile("v_mfma_f32_16x16x32_bf16 a[%2:%3], %0, %1, a[%2:%3]" ::"v"(a), "v"(b), "n"(4u * ACC), "n"(4u * ACC + 3u));
}
// The same where its operands have been written just before.
template <uint32_t ACC>
__device__ __forceinline__ void mfma16_settled(const bf16x8_t& a, const bf16x8_t& b)
{
    asm volatile("s_nop 7\n\tv_mfma_f32_16x16x32_bf16 a[%2:%3], %0, %1, a[%2:%3]" ::"v"(a), "v"(b), "n"(4u * ACC), "n"(4u * ACC + 3u));
}
template <uint32_t ACC>
__device__ __forceinline__ void acc_clear()
{
    asm volatile("v_accvgpr_write_b32 a[%0], 0\n\tv_accvgpr_write_b32 a[%1], 0\n\tv_accvgpr_write_b32 a[%2], 0\n\tv_accvgpr_write_b32 a[%3], 0" ::"n"(4u * ACC),
                 "n"(4u * ACC + 1u), "n"(4u * ACC + 2u), "n"(4u * ACC + 3u));
}
template <uint32_t ACC>
__device__ __forceinline__ f32x4_t acc_read()
{
    float v[4];
    asm volatile("v_accvgpr_read_b32 %0, a[%4]\n\tv_accvgpr_read_b32 %1, a[%5]\n\tv_accvgpr_read_b32 %2, a[%6]\n\tv_accvgpr_read_b32 %3, a[%7]"
                 : "=v"(v[0]), "=v"(v[1]), "=v"(v[2]), "=v"(v[3]) : "n"(4u * ACC), "n"(4u * ACC + 1u), "n"(4u * ACC + 2u), "n"(4u * ACC + 3u));
    return f32x4_t{v[0], v[1], v[2], v[3]};
}
__device__ __forceinline__ void acc_settle() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }

// Waits as instructions that the compiler sees: it adds none of its own for what they cover (where paths meet, only if every one of them has it covered).
template <uint32_t IN_FLIGHT>
__device__ __forceinline__ void wait_vm()
{
    static_assert(IN_FLIGHT < 64u, "six bits");
    __builtin_amdgcn_s_waitcnt((IN_FLIGHT & 15u) | 0x0f70u | (IN_FLIGHT >> 4) << 14);  // vmcnt
}
template <uint32_t IN_FLIGHT>
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xc07f | IN_FLIGHT << 8); }  // lgkmcnt

// The weight of the code in half PART of h: as assembly, which stays in the slot it is written in (and without the compiler's idle cycle behind it, see pair_of_halves).
template <uint32_t PART>
__device__ __forceinline__ void weight_in_place(float& w, uint32_t h, float s, float o)
{
    if constexpr (PART == 0u) asm volatile("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(w) : "v"(h), "v"(s), "v"(o));
    else asm volatile("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(w) : "v"(h), "v"(s), "v"(o));
}

// The order of a step's conversion instructions (see convert_op).
struct WregOp {
    static constexpr uint32_t kPrepare = 0, kFirst = 1, kSecond = 2, kPack = 3;
    uint32_t kind, quad, index;
};
template <uint32_t PREPARE>
struct WregSchedule {
    static constexpr uint32_t kOps = 8u * PREPARE + 32u * 3u;
    static constexpr WregOp op(uint32_t at)
    {
        if (at < PREPARE) return WregOp{WregOp::kPrepare, 0u, at};
        at -= PREPARE;
        for (uint32_t v = 0;; ++v) {
            const uint32_t quad = v >> 2, b = v & 3u, next = quad < 7u ? PREPARE : 0u;
            const uint32_t from = b * next / 4u, to = (b + 1u) * next / 4u;
            if (at < 2u) return WregOp{at == 0u ? WregOp::kFirst : WregOp::kSecond, quad, b};
            at -= 2u;
            if (at < to - from) return WregOp{WregOp::kPrepare, quad + 1u, from + at};
            at -= to - from;
            if (at == 0u) return WregOp{WregOp::kPack, quad, b};
            at -= 1u;
        }
    }
};

}  // namespace

template <int BITS, bool GROUPED, bool PACKED, int MT>
__global__ void __launch_bounds__(256) bfaintb_prefill_wreg_kernel(const GemmParams p)
{
    static_assert(MT >= 8 && MT <= 16 && MT % 2 == 0, "blocks of 16 rows, whole copies of 32 rows");
    constexpr uint32_t kRows = 16u * MT;          // rows of a tile
    constexpr uint32_t kACopies = MT / 2u;        // of A, per wave and step: 8 rows each
    constexpr uint32_t kStageBytes = kRows * 128u;
    constexpr uint32_t kCodeStageBytes = PACKED ? 0u : 64u * 256u * BITS / 8u;
    __shared__ __attribute__((aligned(1024))) uint8_t lds_a0[kStageBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t lds_a1[kStageBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t lds_a2[kStageBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t lds_w0[PACKED ? 1024u : kCodeStageBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t lds_w1[PACKED ? 1024u : kCodeStageBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t lds_w2[PACKED ? 1024u : kCodeStageBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t lds_s0[1024];
    __shared__ __attribute__((aligned(1024))) uint8_t lds_s1[1024];
    __shared__ __attribute__((aligned(1024))) uint8_t lds_s2[1024];
    // (separate arrays rather than one block: the compiler then knows that reads of one stage cannot alias
    // the asynchronous copies into another, and does not make them wait for those)
    auto a_tile = [&](auto stage_c) -> uint8_t* {
        constexpr uint32_t St = decltype(stage_c)::value % 3u;
        return St == 0 ? lds_a0 : St == 1 ? lds_a1 : lds_a2;
    };
    auto w_tile = [&](auto stage_c) -> uint8_t* {
        constexpr uint32_t St = decltype(stage_c)::value % 3u;
        return St == 0 ? lds_w0 : St == 1 ? lds_w1 : lds_w2;
    };
    auto s_tile = [&](auto stage_c) -> uint8_t* {
        constexpr uint32_t St = decltype(stage_c)::value % 3u;
        return St == 0 ? lds_s0 : St == 1 ? lds_s1 : lds_s2;
    };
    using C0 = std::integral_constant<uint32_t, 0>;
    using C1 = std::integral_constant<uint32_t, 1>;
    using C2 = std::integral_constant<uint32_t, 2>;

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // 0..3: the wave's 64 columns
    const uint32_t c16 = lane & 15u, kq = lane >> 4;

    // ---- tile of this workgroup: ids that share an XCD (id mod 8) cover consecutive logical ids, which walk groups of
    //      4 tile-rows column by column (as in bfaintb_prefill_kernel)
    //      (eight blocks: or, with p.tile_halves, the upper and the lower halves of tiles of 256 rows, the thin last round of those)
    const bool in_halves = MT == 8 && p.tile_halves != 0u;
    const uint32_t tile_rows = in_halves ? 2u * kRows : kRows;
    const uint32_t tiles_m = (p.m + tile_rows - 1) / tile_rows, tiles_n = (p.n + kWrTile - 1) / kWrTile;
    const uint32_t wgs = in_halves ? 2u * p.tile_count : p.tile_count;
    const uint32_t per_xcd = (wgs + 7u) / 8u;
    const uint32_t local = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
    if (local >= wgs) return;
    const uint32_t logical = p.tile_first + (in_halves ? local >> 1 : local);
    const uint32_t group = logical / (4u * tiles_n);
    const uint32_t first_m = group * 4u;
    const uint32_t group_rows = tiles_m - first_m < 4u ? tiles_m - first_m : 4u;
    const uint32_t in_group = logical - group * 4u * tiles_n;
    const uint32_t tm = first_m + in_group % group_rows;
    const uint32_t tn = in_group / group_rows;
    const uint32_t m0 = tm * tile_rows + (in_halves ? (local & 1u) * kRows : 0u), n0 = tn * kWrTile;
    if (in_halves && m0 >= p.m) return;  // the lower half of a last, flat tile

    const uint32_t rows_valid = p.m - m0 < kRows ? p.m - m0 : kRows;
    const uint32_t a_extent = ((rows_valid - 1u) * p.lda + p.k) * 2u;
    const __amdgpu_buffer_rsrc_t rsrc_a =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.a + (size_t)m0 * p.lda), 0, (int)a_extent, kBufferFlags);
    const uint32_t cols_valid = p.n - n0 < kWrTile ? p.n - n0 : kWrTile;
    // packed weights: a block of 16 columns is one run of k x 16 codes (chunks of 1024 bytes: 64 rows of 8-bit, 128 rows of
    // 4-bit codes); the tile's column blocks follow one another, and one past n reads as zero through the extent
    const uint32_t slab_bytes = p.k * (BITS == 8 ? 16u : 8u);
    const __amdgpu_buffer_rsrc_t rsrc_b =
        PACKED ? __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.b + (size_t)(n0 / 16u) * slab_bytes), 0,
                                                   (int)(cols_valid / 16u * slab_bytes), kBufferFlags)
               : __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.b + (BITS == 8 ? n0 : n0 / 2u)), 0,
                                                   (int)((p.k - 1u) * p.ldb_bytes + (BITS == 8 ? cols_valid : cols_valid / 2u)), kBufferFlags);

    const uint32_t ksteps = (p.k + kWrK - 1u) / kWrK;
    const uint32_t last_chunks = (p.k - (ksteps - 1u) * kWrK) / 8u;  // valid 16-byte chunks per row of A in the last step

    // A copy: instruction j of wave w fills rows 8 (kACopies w + j) .. + 7; lane l lands at row + l / 8, chunk position l % 8, so it
    // fetches chunk (l % 8) ^ ((row >> 1) & 7) = (l % 8) ^ (l / 16) for even kACopies w + j and that ^ 4 for odd ones: two lane
    // offsets, the row advance of j (and the K advance) in the scalar offset.
    const uint32_t a_block = kACopies * wave;  // the wave's first 8 rows
    const uint32_t a_row = 8u * a_block + (lane >> 3);
    const uint32_t chunk_e = (lane & 7u) ^ ((lane >> 4) & 7u) ^ (4u * (a_block & 1u)), chunk_o = chunk_e ^ 4u;
    const uint32_t a_voff_e = (a_row * p.lda + chunk_e * 8u) * 2u, a_voff_o = (a_row * p.lda + chunk_o * 8u) * 2u;
    // a chunk past the end of k (partial last step) is fetched from beyond the extent: it reads as zero
    const uint32_t a_last_e = chunk_e < last_chunks ? a_voff_e : a_extent, a_last_o = chunk_o < last_chunks ? a_voff_o : a_extent;
    auto copy_a = [&](auto stage_c, auto j_c, uint32_t ve, uint32_t vo, uint32_t soff) {
        constexpr uint32_t j = decltype(j_c)::value;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (__attribute__((address_space(3))) void*)(a_tile(stage_c) + a_block * 1024u + j * 1024u), 16, (j & 1u) ? vo : ve, soff, 0, 0);
    };
    auto copy_a_all = [&](auto stage_c, uint32_t kt) {
        const bool last = kt + 1u == ksteps;
        for_each_const<kACopies>([&](auto j_c) { copy_a(stage_c, j_c, last ? a_last_e : a_voff_e, last ? a_last_o : a_voff_o, kt * kWrK * 2u + decltype(j_c)::value * 16u * p.lda); });
    };

    // Codes in rows.  Copy: instruction i of a wave and step fills 1024 bytes = 8 rows of 128 bytes of the stage, lane l row l / 8 of them, position
    // l % 8, from the 16 bytes that belong there: position = 16 bytes' index ^ turn(row), chosen so that the transposing reads below
    // find 16 rows of a column block in 16 different groups of banks.
    //   8-bit: the stage is two halves of 128 columns, 64 rows of 128 bytes each; wave w copies rows 16 w .. + 15 of both, instruction i rows
    //     8 (i / 2) of them, half i % 2;
    //   4-bit: 64 rows of 256 columns; wave w copies rows 16 w .. + 15, instruction i rows 8 i of them.
    // Rows of B past k read as zero codes, finite weights, and multiply zeros of A.
    constexpr uint32_t kCodeCopies = PACKED ? 0u : BITS / 2u;
    auto turn = [](uint32_t row) { return BITS == 8 ? (row ^ (row >> 3)) & 7u : (row >> 1) & 7u; };
    const uint32_t w_row0 = 16u * wave + (lane >> 3);  // (rows 8 further on: the other lane offset)
    const uint32_t w_voff0 = PACKED ? 0u : w_row0 * p.ldb_bytes + (((lane & 7u) ^ turn(w_row0)) << 4);
    const uint32_t w_voff1 = PACKED ? 0u : (w_row0 + 8u) * p.ldb_bytes + (((lane & 7u) ^ turn(w_row0 + 8u)) << 4);
    auto copy_codes = [&](auto stage_c, auto i_c, uint32_t kt) {
        constexpr uint32_t i = decltype(i_c)::value, eight = BITS == 8 ? i >> 1 : i, half = BITS == 8 ? i & 1u : 0u;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (__attribute__((address_space(3))) void*)(w_tile(stage_c) + half * 8192u + wave * 2048u + eight * 1024u), 16,
                                                 eight ? w_voff1 : w_voff0, kt * kWrK * p.ldb_bytes + half * 128u, 0, 0);
    };
    // Group scales: the tile's 256 for each of a step's two blocks of 32 k, 4 bytes a lane; wave w copies columns 128 (w % 2) .. + 127 of block w / 2.
    const uint32_t scale_rows = GROUPED ? p.k / p.group_size : 1u;
    const __amdgpu_buffer_rsrc_t rsrc_s = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(p.scale), 0, (int)(((scale_rows - 1u) * p.lds + p.n) * 2u), kBufferFlags);
    auto group_at = [&](uint32_t row) -> uint32_t {
        const uint32_t g = GROUPED ? group_of_row(p, row) : 0u;
        return g < scale_rows ? g : scale_rows - 1u;  // rows past k in a partial last step: any scale will do
    };
    auto copy_scales = [&](auto stage_c, uint32_t kt) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_s, (__attribute__((address_space(3))) void*)(s_tile(stage_c) + wave * 256u), 4,
                                                 (n0 + 128u * (wave & 1u)) * 2u + lane * 4u, group_at(kt * kWrK + 32u * (wave >> 1)) * p.lds * 2u, 0, 0);
    };
    // Packed codes: a lane's 16 bytes of a chunk of a column block are, in order, its 8-row operands for the chunk's blocks of 32 k: two for 8-bit codes
    // = a step; four for 4-bit codes, of which a step takes 8 bytes.
    struct Raw {
        uint32_t d[4][4];  // [column block j]: 8-bit: rows 0 .. 3 and 4 .. 7 of block 0, of block 1; 4-bit: the 8 rows of block 0, of block 1
    };
    auto load_codes = [&](Raw& raw, uint32_t kt, auto j_c) {
        constexpr uint32_t j = decltype(j_c)::value;
        const uint32_t soff = (4u * wave + j) * slab_bytes + (BITS == 8 ? kt * 1024u : (kt >> 1) * 1024u + (kt & 1u) * 8u);
        if constexpr (BITS == 8) {
            const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(rsrc_b, lane * 16u, soff, 0);
            raw.d[j][0] = v[0], raw.d[j][1] = v[1], raw.d[j][2] = v[2], raw.d[j][3] = v[3];
        } else {
            const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(rsrc_b, lane * 16u, soff, 0);
            raw.d[j][0] = v[0], raw.d[j][1] = v[1];
        }
    };

    const uint32_t wcol = 64u * wave + c16;  // the lane's column j of the tile: wcol + 16 j
    auto col_ok = [&](uint32_t j) { return n0 + wcol + 16u * j < p.n; };

    // ---- Conversion by halves (bfaintb_device.hpp has the argument).
    constexpr int kUpper = BITS == 8 ? 1024 : 64;
    typedef HalfMultipliers<BITS, kUpper> Multiplier;
    HalfConstants<BITS, kUpper> half_k;
    half_k.keep();
    float most = 0.f;  // 8-bit codes: the largest magnitude among the lane's scales
    Multiplier fixed[4];
    if constexpr (!GROUPED) {
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) fixed[j] = Multiplier(bf16_bits_to_f32(__builtin_amdgcn_raw_buffer_load_b16(rsrc_s, (n0 + wcol) * 2u, 32u * j, 0)));
        if constexpr (BITS == 8) largest_scale(most, fixed[0].s, fixed[1].s), largest_scale(most, fixed[2].s, fixed[3].s);
    }
    struct Ops {
        uint32_t w[2][4][4];  // [block of 32 k][column j]: the 8-element operand as 4 packed pairs of rows
    };
    // A step's weights are made as 8 quads, quad q column q % 4 of block q / 4, of 4 pairs of rows (4-bit codes: pairs 0, 2, 1, 3, as the halves lie).
    struct Quad {
        uint32_t d[2];  // codes: 8-bit: rows 0 .. 3, 4 .. 7; 4-bit: 8 rows
        uint32_t s;     // group scale, bf16
    };
    Quad codes[4];             // by the quad, mod 4
    struct Conversion {
        uint32_t h[2][4];      // halves, by the quad's parity
        uint32_t x[4];         // 4-bit codes: shifted
        Multiplier mu[2];      // group scales, by the quad's parity
        float w0, w1;          // a pair's weights
    };
    // What a quad needs from LDS.  Rows: lane (c16, kq) addresses, of the 8 rows of its kq,
    //   8-bit (ds_read_b64_tr_b8): 8 bytes, half c16 % 2 of row c16 / 2, and receives byte c16 of each row;
    //   4-bit (ds_read_b64_tr_b4): 8 bytes, 16 codes, of row c16 % 8, and receives code c16 of all: eight rows of one column block from lanes 0 .. 7,
    //     the same rows of the next from the others: two quads.
    uint32_t w_rd[2][4];       // [block of 32 k][column block (4-bit: pair of column blocks)]
    const uint32_t s_rd0 = (64u * wave + c16) * 2u;
    // (The stages lie one behind the other, and an instruction's 16 offset bits reach 64 KiB: indexes that far on, which the compiler cannot take
    // apart again, save an addition for each read of the stages there.)
    constexpr uint32_t kFarA = 2u * kStageBytes, kFarW = 3u * kStageBytes, kFarS = kFarW + 3u * (PACKED ? 1024u : kCodeStageBytes);
#pragma unroll
    for (uint32_t blk = 0; blk < 2; ++blk) {
        const uint32_t row = 32u * blk + 8u * kq + (BITS == 8 ? c16 >> 1 : c16 & 7u);
#pragma unroll
        for (uint32_t j = 0; j < (BITS == 8 ? 4u : 2u); ++j) {
            w_rd[blk][j] = kFarW + (BITS == 8 ? (wave >> 1) * 8192u + row * 128u + (((4u * (wave & 1u) + j) ^ turn(row)) << 4) + 8u * (c16 & 1u)
                                              : row * 128u + (((2u * wave + j) ^ turn(row)) << 4) + (c16 & 8u));
            if constexpr (!PACKED) asm("" : "+v"(w_rd[blk][j]));
        }
    }
    uint32_t s_rd = s_rd0 + kFarS;
    if constexpr (GROUPED) asm("" : "+v"(s_rd));
    auto read_quad = [&](auto stage_c, auto quad_c) {
        constexpr uint32_t quad = decltype(quad_c)::value, blk = quad >> 2, j = quad & 3u;
        typedef int v2i __attribute__((ext_vector_type(2)));
        typedef __attribute__((address_space(3))) v2i* lds_v2i;
        if constexpr (!PACKED && BITS == 8) {
            const v2i v = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i)(w_tile(stage_c) + (w_rd[blk][j] - kFarW)));
            codes[quad & 3u].d[0] = (uint32_t)v[0], codes[quad & 3u].d[1] = (uint32_t)v[1];
        } else if constexpr (!PACKED && (quad & 1u) == 0u) {
            const v2i v = __builtin_amdgcn_ds_read_tr4_b64_v2i32((lds_v2i)(w_tile(stage_c) + (w_rd[blk][j >> 1] - kFarW)));
            codes[quad & 3u].d[0] = (uint32_t)v[0], codes[(quad + 1u) & 3u].d[0] = (uint32_t)v[1];
        }
        if constexpr (GROUPED) codes[quad & 3u].s = *reinterpret_cast<const uint16_t*>(s_tile(stage_c) + (s_rd - kFarS) + blk * 512u + 32u * j);
    };

    // One vector instruction of what a quad needs before its products.  Each is held where it is written, in an order in which none
    // reads what the one before has made (the compiler would put an idle cycle between).
    constexpr uint32_t kPrepareOps = (BITS == 8 ? 4u : 7u) + (GROUPED ? (BITS == 8 ? 3u : 2u) : 0u);
    auto prepare = [&](Conversion& w, const Raw& raw, auto quad_c, auto op_c) {
        constexpr uint32_t quad = decltype(quad_c)::value, blk = quad >> 2, j = quad & 3u;
        constexpr uint32_t kWiden = 100u, kOffset = 101u, kLargest = 102u;
        constexpr uint32_t order8g[7] = {kWiden, 0u, 1u, kOffset, 2u, kLargest, 3u}, order4g[9] = {kWiden, 0u, 1u, kOffset, 2u, 3u, 4u, 5u, 6u};
        constexpr uint32_t op = !GROUPED ? decltype(op_c)::value : BITS == 8 ? order8g[decltype(op_c)::value % 7u] : order4g[decltype(op_c)::value];
        uint32_t (&h)[4] = w.h[quad & 1u];
        Multiplier& mu = w.mu[quad & 1u];
        if constexpr (op == kWiden) {
            uint32_t bits = codes[quad & 3u].s;
            hold(bits);  // (or the widening moves up to the read)
            mu.s = bf16_bits_to_f32(bits), hold(mu.s);
        } else if constexpr (op == kOffset) {
            mu.o = Multiplier(mu.s).o, hold(mu.o);
        } else if constexpr (op == kLargest) {
            largest_scale(most, mu.s, mu.s);
        } else if constexpr (BITS == 8) {  // rows 0 and 2, 1 and 3, 4 and 6, 5 and 7
            const uint32_t d = PACKED ? raw.d[j][2u * blk + (op >> 1)] : codes[quad & 3u].d[op >> 1];
            h[op] = (op & 1u) == 0u ? halves<0>(d, half_k) : halves<1>(d, half_k);
            hold(h[op]);
        } else {                           // rows 0 and 4, 1 and 5, 2 and 6, 3 and 7
            const uint32_t x = PACKED ? raw.d[j][blk] : codes[quad & 3u].d[0];
            if constexpr (op == 0u) w.x[1] = x << 4, hold(w.x[1]);
            if constexpr (op == 1u) w.x[2] = x >> 4, hold(w.x[2]);
            if constexpr (op == 2u) h[0] = halves<1>(w.x[1], half_k), hold(h[0]);
            if constexpr (op == 3u) w.x[3] = x >> 8, hold(w.x[3]);
            if constexpr (op == 4u) h[1] = halves<1>(x, half_k), hold(h[1]);
            if constexpr (op == 5u) h[2] = halves<1>(w.x[2], half_k), hold(h[2]);
            if constexpr (op == 6u) h[3] = halves<1>(w.x[3], half_k), hold(h[3]);
        }
    };
    auto multiply = [&](Conversion& w, auto quad_c, auto b_c, auto second_c) {
        constexpr uint32_t quad = decltype(quad_c)::value, b = decltype(b_c)::value, second = decltype(second_c)::value;
        const Multiplier& mu = GROUPED ? w.mu[quad & 1u] : fixed[quad & 3u];
        weight_in_place<(b & 1u)>(second ? w.w1 : w.w0, w.h[quad & 1u][(b & 2u) + second], mu.s, mu.o);
    };
    auto pack = [&](Ops& ops, const Conversion& w, auto quad_c, auto b_c) {
        constexpr uint32_t quad = decltype(quad_c)::value, b = decltype(b_c)::value;
        uint32_t& to = ops.w[quad >> 2][quad & 3u][BITS == 8 ? b : (b & 1u) * 2u + (b >> 1)];
        to = pack_bf16_rne(w.w0, w.w1);
        hold(to);
    };
    // The instructions in order: what the first quad needs; then for each pair its two products, a quarter of what the next quad needs, the pack.
    typedef WregSchedule<kPrepareOps> Schedule;
    auto convert_op = [&](Ops& ops, Conversion& w, const Raw& raw, auto at_c) {
        constexpr WregOp o = Schedule::op(decltype(at_c)::value);
        using QuadC = std::integral_constant<uint32_t, o.quad>;
        using Index = std::integral_constant<uint32_t, o.index>;
        if constexpr (o.kind == WregOp::kPrepare) prepare(w, raw, QuadC{}, Index{});
        else if constexpr (o.kind == WregOp::kFirst) multiply(w, QuadC{}, Index{}, C0{});
        else if constexpr (o.kind == WregOp::kSecond) multiply(w, QuadC{}, Index{}, C1{});
        else pack(ops, w, QuadC{}, Index{});
    };

    acc_reserve<MT>();
    for_each_const<4u * MT>([](auto acc_c) { acc_clear<decltype(acc_c)::value>(); });

    // fragment (mt, blk): row 16 mt + c16 of the tile, chunk 4 blk + kq
    uint32_t a_rd[2], a_rd_far[2];
#pragma unroll
    for (uint32_t blk = 0; blk < 2; ++blk) {
        a_rd[blk] = wr_swz(c16, 4u * blk + kq);  // + mt * 2048 (16 rows; the swizzle repeats every 16 rows)
        a_rd_far[blk] = a_rd[blk] + kFarA;
        asm("" : "+v"(a_rd_far[blk]));
    }
    auto read_frag = [&](auto stage_c, uint32_t blk, uint32_t mt) -> bf16x8_t {
        constexpr bool kFar = decltype(stage_c)::value % 3u == 2u;
        return *reinterpret_cast<const bf16x8_t*>(a_tile(stage_c) + (kFar ? a_rd_far[blk] - kFarA : a_rd[blk]) + mt * 2048u);
    };

    // One K-step: stage S and `cur` hold this step; `nxt` receives the operands of step kt + 1, from `raw1` (packed codes, loaded one
    // step ago) or from the code stage S + 1; `raw2` receives the packed codes of step kt + 2.
    // With one wave per SIMD nothing overlaps by itself: the wave issues in order, and the matrix pipe idles whenever the
    // wave is busy issuing something else for longer than a matrix instruction runs (16 cycles).  One vector instruction and one LDS read fit
    // beside a matrix instruction, a second vector instruction costs some 8 cycles, a memory request 7 or more (four waves make theirs at
    // the same time).  So the step is written as 8 MT fenced slots of one matrix instruction, with everything else spread evenly over them: slot
    // 4 u + j is unit u (row block u % MT of the block of 32 k u / MT), column block j.
    //   fragments of A: a group of four units waits once, for its own, and reads those of the group after the next, one in each unit;
    //   quads: read a quarter of a step before they are prepared, the first two at the end of the step before;
    //   conversion: one instruction after the other (Schedule);
    //   memory: codes (in rows of step kt + 3, packed of kt + 2), group scales of kt + 3 and the copies of A of kt + 2, evenly over the step, packed codes first.
    // The step's one barrier stands 24 slots before its end, where the next step's first fragments and the codes after it are about to be read: before
    // it the wave makes sure that its part of them has landed (requested in the step before: what may still be in flight then is this step's
    // own) and that it has everything it reads of this step's A and the next one's codes and scales.  Behind it every wave's part has landed, and
    // nobody reads this step's A or the next one's codes any more: copies requested from there on go to their places.
    using Step = WregStep<BITS, GROUPED, PACKED, MT>;
    static_assert(Step::quad_slot(6u) < Step::quad_slot(7u) && Step::quad_slot(7u) < Step::kBarrierSlot && Step::frag_slot(Step::kUnits - 1u) < Step::kBarrierSlot,
                  "a step's reads of its own A and the next step's codes stand before its barrier");
    constexpr uint32_t kUnits = Step::kUnits, kSlots = Step::kSlots, kBarrierSlot = Step::kBarrierSlot;
    bf16x8_t af[12];
    auto step = [&](auto at_c, uint32_t kt, const Ops& cur, Ops& nxt, const Raw& raw1, Raw& raw2) {
        constexpr uint32_t S = decltype(at_c)::value, kTurn = S * kUnits;
        using Now = std::integral_constant<uint32_t, S % 3u>;
        using Next = std::integral_constant<uint32_t, (S + 1u) % 3u>;
        using After = std::integral_constant<uint32_t, (S + 2u) % 3u>;
        const uint32_t kt2 = kt + 2 < ksteps ? kt + 2 : ksteps - 1, kt3 = kt + 3 < ksteps ? kt + 3 : ksteps - 1;
        const bool last = kt2 + 1u == ksteps;
        const uint32_t a_ve = last ? a_last_e : a_voff_e, a_vo = last ? a_last_o : a_voff_o;
        uint32_t a_soff = kt2 * kWrK * 2u;
        Conversion w;
        if constexpr (PACKED) wait_vm<Step::behind_codes()>();  // raw1's
        __builtin_amdgcn_sched_barrier(0);
        for_each_const<kSlots>([&](auto slot_c) {
            constexpr uint32_t slot = decltype(slot_c)::value;
            constexpr uint32_t u = slot >> 2, j = slot & 3u, blk = u / MT, mt = u % MT;
            if constexpr (slot % 16u == 0u) wait_lds<Step::in_flight(slot / 16u)>();
            mfma16<4u * mt + j>(af[(u + kTurn) % 12u],
                                __builtin_bit_cast(bf16x8_t, make_uint4(cur.w[blk][j][0], cur.w[blk][j][1], cur.w[blk][j][2], cur.w[blk][j][3])));
            if constexpr (slot == kBarrierSlot) {
                wait_vm<Step::requests_before(kBarrierSlot)>();
                wait_lds<0>();
                barrier_no_fence();  // (a fenced barrier would also wait for the copies this step has just started)
            }
            for_each_const<2u>([&](auto next_c) {  // a fragment: of the unit two groups on; behind the barrier the next step's first
                constexpr bool next = decltype(next_c)::value != 0u;
                constexpr uint32_t un = next ? (slot - kBarrierSlot) / 3u : slot / 4u + 8u;
                if constexpr (next ? slot >= kBarrierSlot && un < 8u && Step::frag_slot(un) == slot : un < kUnits && Step::frag_slot(un) == slot) {
                    if constexpr (next) af[(un + kUnits + kTurn) % 12u] = read_frag(Next{}, 0, un);
                    else af[(un + kTurn) % 12u] = read_frag(Now{}, un / MT, un % MT);
                }
            });
            for_each_const<8u>([&](auto quad_c) {
                if constexpr (Step::quad_slot(decltype(quad_c)::value) == slot) {
                    if constexpr (decltype(quad_c)::value < 2u) read_quad(After{}, quad_c);
                    else read_quad(Next{}, quad_c);
                }
            });
            constexpr uint32_t from = slot * Schedule::kOps / kSlots, to = (slot + 1u) * Schedule::kOps / kSlots;
            for_each_const<to - from>([&](auto i_c) { convert_op(nxt, w, raw1, std::integral_constant<uint32_t, from + decltype(i_c)::value>{}); });
            constexpr uint32_t r = Step::requests_before(slot);
            if constexpr (Step::requests_before(slot + 1u) != r) {
                constexpr uint32_t c = Step::copies_before(r), q = r - c;
                if constexpr (Step::copies_before(r + 1u) != c) {
                    copy_a(After{}, std::integral_constant<uint32_t, c>{}, a_ve, a_vo, a_soff);
                    a_soff += 16u * p.lda;
                    asm("" : "+s"(a_soff));  // (or each request gets a multiplication of its own)
                } else if constexpr (GROUPED && q == 0u) {
                    copy_scales(Now{}, kt3);
                } else if constexpr (PACKED) {
                    load_codes(raw2, kt2, std::integral_constant<uint32_t, q - (GROUPED ? 1u : 0u)>{});
                } else {
                    copy_codes(Now{}, std::integral_constant<uint32_t, q - (GROUPED ? 1u : 0u)>{}, kt3);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    };

    // ---- prologue: A tiles 0 and 1, codes and group scales of steps 0 to 2 on their way; operands of step 0; the first fragments and quads
    Ops ops0, ops1;
    Raw rawa, rawb;
    const uint32_t kt1 = ksteps > 1 ? 1 : 0, kt2 = ksteps > 2 ? 2 : ksteps - 1;
    copy_a_all(C0{}, 0);
    if constexpr (PACKED) {
        for_each_const<4u>([&](auto j_c) { load_codes(rawb, 0, j_c); });
        for_each_const<4u>([&](auto j_c) { load_codes(rawa, kt1, j_c); });
    } else {
        for_each_const<kCodeCopies>([&](auto i_c) { copy_codes(C0{}, i_c, 0); });
        for_each_const<kCodeCopies>([&](auto i_c) { copy_codes(C1{}, i_c, kt1); });
        for_each_const<kCodeCopies>([&](auto i_c) { copy_codes(C2{}, i_c, kt2); });
    }
    if constexpr (GROUPED) copy_scales(C0{}, 0), copy_scales(C1{}, kt1), copy_scales(C2{}, kt2);
    __builtin_amdgcn_sched_barrier(0);
    copy_a_all(C1{}, kt1);
    __builtin_amdgcn_sched_barrier(0);
    wait_vm<kACopies>();
    barrier_no_fence();
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) af[i] = read_frag(C0{}, 0, i);
    {
        Conversion w;
        for_each_const<2u>([&](auto blk_c) {
            constexpr uint32_t blk = decltype(blk_c)::value;
            for_each_const<4u>([&](auto j_c) { read_quad(C0{}, std::integral_constant<uint32_t, 4u * blk + decltype(j_c)::value>{}); });
            for_each_const<4u>([&](auto j_c) {
                using QuadC = std::integral_constant<uint32_t, 4u * blk + decltype(j_c)::value>;
                for_each_const<kPrepareOps>([&](auto op_c) { prepare(w, rawb, QuadC{}, op_c); });
                for_each_const<4u>([&](auto b_c) { multiply(w, QuadC{}, b_c, C0{}), multiply(w, QuadC{}, b_c, C1{}), pack(ops0, w, QuadC{}, b_c); });
            });
        });
    }
    // (the first step's copies of codes and scales go to stage 0: every wave has read it)
    if constexpr (!PACKED || GROUPED) barrier_no_fence();
    read_quad(C1{}, C0{}), read_quad(C1{}, C1{});

#ifdef BFAINTB_TRACE
    const long long tr_c0 = clock64(), tr_w0 = wall_clock64();
#endif
    using C3 = std::integral_constant<uint32_t, 3>;
    using C4 = std::integral_constant<uint32_t, 4>;
    using C5 = std::integral_constant<uint32_t, 5>;
    // Six at a time (stages by threes, operands by twos), in a loop that is left at its end only, and the last one to six behind it.  With an exit
    // behind each step the compiler led all of them round by the loop's head, took what every step's end has in flight for what the head has, and waited
    // there for all of a wave's copies, those of a dozen slots ago included.  us, so / now: 2684 x 3888 x 8832 4-bit g32 163.0 / 160.0, 2670 x 3104 x 4864
    // packed 8-bit 78.4 / 75.5, 3128 x 9280 x 2304 packed 8-bit g128 124.7 / 121.1; up to a k of 768 level (the loop over whole sixes, with up to five
    // behind it, loses up to 2 % there: its last steps' code is a workgroup's first).
    uint32_t kt = 0;
    for (; kt + 6 < ksteps; kt += 6) {
        step(C0{}, kt, ops0, ops1, rawa, rawb);
        step(C1{}, kt + 1, ops1, ops0, rawb, rawa);
        step(C2{}, kt + 2, ops0, ops1, rawa, rawb);
        step(C3{}, kt + 3, ops1, ops0, rawb, rawa);
        step(C4{}, kt + 4, ops0, ops1, rawa, rawb);
        step(C5{}, kt + 5, ops1, ops0, rawb, rawa);
    }
    step(C0{}, kt, ops0, ops1, rawa, rawb);
    if (kt + 1 < ksteps) {
        step(C1{}, kt + 1, ops1, ops0, rawb, rawa);
        if (kt + 2 < ksteps) {
            step(C2{}, kt + 2, ops0, ops1, rawa, rawb);
            if (kt + 3 < ksteps) {
                step(C3{}, kt + 3, ops1, ops0, rawb, rawa);
                if (kt + 4 < ksteps) {
                    step(C4{}, kt + 4, ops0, ops1, rawa, rawb);
                    if (kt + 5 < ksteps) step(C5{}, kt + 5, ops1, ops0, rawb, rawa);
                }
            }
        }
    }
#ifdef BFAINTB_TRACE
    {   // shader cycles and 100 MHz ticks the K loop took, per wave: words 0, 1 of the wave's 8
        const long long tr_c1 = clock64(), tr_w1 = wall_clock64();
        if (lane == 0 && p.trace != nullptr) {
            unsigned long long* t = p.trace + (size_t)(blockIdx.x * 4u + wave) * 8u;
            t[0] = (unsigned long long)(tr_c1 - tr_c0);
            t[1] = (unsigned long long)(tr_w1 - tr_w0);
            t[2] = (unsigned long long)tr_w0;
            t[3] = (unsigned long long)tr_w1;
        }
    }
#endif

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing asynchronous may still be writing LDS
    // ---- 8-bit codes, a scale beyond the conversion by halves: the wave's sums once more, in the same order, by the other conversion,
    // everything straight from memory (the other waves wait at the epilogue's first barrier)
    if constexpr (BITS == 8) {
        if (__builtin_expect(beyond_halves(most), 0)) {
            acc_settle();
            for_each_const<4u * MT>([](auto acc_c) { acc_clear<decltype(acc_c)::value>(); });
#pragma unroll 1
            for (uint32_t block = 0; block < 2u * ksteps; ++block) {
                const uint32_t kt = block >> 1, blk = block & 1u, row0 = 32u * block;
                const uint32_t s_off = group_at(row0) * p.lds * 2u;
                bf16x8_t w[4];
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) {
                    const float s = bf16_bits_to_f32(__builtin_amdgcn_raw_buffer_load_b16(rsrc_s, (n0 + wcol) * 2u, s_off + 32u * j, 0));
                    uint32_t c[2] = {0u, 0u};
                    if constexpr (PACKED) {
                        const uint32_t off = (4u * wave + j) * slab_bytes + kt * 1024u + 8u * blk;
                        c[0] = __builtin_amdgcn_raw_buffer_load_b32(rsrc_b, lane * 16u, off, 0);
                        c[1] = __builtin_amdgcn_raw_buffer_load_b32(rsrc_b, lane * 16u + 4u, off, 0);
                    } else {
#pragma unroll
                        for (uint32_t r = 0; r < 8; ++r)
                            c[r >> 2] |= (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(rsrc_b, (row0 + 8u * kq + r) * p.ldb_bytes + wcol + 16u * j, 0, 0) << (8u * (r & 3u));
                    }
                    w[j] = __builtin_bit_cast(bf16x8_t, weights8(c[0], c[1], s));
                }
                const bool past_k = kt + 1u == ksteps && 4u * blk + kq >= last_chunks;
                for_each_const<(uint32_t)MT>([&](auto mt_c) {
                    constexpr uint32_t mt = decltype(mt_c)::value;
                    const uint32_t off = past_k ? a_extent : ((16u * mt + c16) * p.lda + row0 + 8u * kq) * 2u;
                    const bf16x8_t a = __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, off, 0, 0));
                    mfma16_settled<4u * mt>(a, w[0]), mfma16_settled<4u * mt + 1u>(a, w[1]), mfma16_settled<4u * mt + 2u>(a, w[2]), mfma16_settled<4u * mt + 3u>(a, w[3]);
                });
            }
        }
    }

    // ---- epilogue: the tile through LDS (the stages of A) in [m][n] order, a part of its rows at a time, then 16-byte row-contiguous stores
    acc_settle();  // the last matrix instructions have written their accumulators
    __syncthreads();
    // where four rows of the staged part start, rows4 = the first one / 4, with `per_array` such rows in each array
    auto c_rows4 = [&](uint32_t rows4, uint32_t per_array, uint32_t row_bytes) -> uint8_t* {
        const uint32_t q = rows4 / per_array;
        return (q == 0u ? lds_a0 : q == 1u ? lds_a1 : lds_a2) + (rows4 - q * per_array) * 4u * row_bytes;
    };
    const bool gated = p.activation == kActSiluGate;
    if (p.residual == nullptr && !gated) {
        // the bare sums, or sums + bias: rounded in registers, staged as bf16, half the rows (in the first two arrays) at a time
        float bias[4] = {0.f, 0.f, 0.f, 0.f};
        const bool has_bias = p.bias != nullptr;
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j)
            if (has_bias && col_ok(j)) bias[j] = bf16_bits_to_f32(p.bias[n0 + wcol + 16u * j]);
        // A lane's four columns are 16 apart, so it stages four single values per row, and the four
        // k-groups of a wave (rows 4 apart: the same banks) would collide; the 32-byte groups of a row are therefore
        // stored at position (group ^ ((row >> 2) & 3)), which the readers below undo.
        uint32_t at[4];
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) at[j] = (((4u * wave + j) ^ kq) << 5) + c16 * 2u;
        for_each_const<2u>([&](auto half_c) {
            constexpr uint32_t half = decltype(half_c)::value;
            for_each_const<MT / 2u>([&](auto mh_c) {
                constexpr uint32_t mh = decltype(mh_c)::value, mt = MT / 2u * half + mh;
                uint8_t* base = c_rows4(4u * mh + kq, MT, kWrCRowBytes);
                const f32x4_t acc[4] = {acc_read<4u * mt>(), acc_read<4u * mt + 1u>(), acc_read<4u * mt + 2u>(), acc_read<4u * mt + 3u>()};
#pragma unroll
                for (uint32_t r = 0; r < 4; ++r) {
                    uint2 o;
                    // without a bias the sums are stored as they are (adding +0 would turn a -0 sum into +0)
                    if (has_bias) {
                        o.x = pack_bf16_rne(acc[0][r] + bias[0], acc[1][r] + bias[1]);
                        o.y = pack_bf16_rne(acc[2][r] + bias[2], acc[3][r] + bias[3]);
                    } else {
                        o.x = pack_bf16_rne(acc[0][r], acc[1][r]);
                        o.y = pack_bf16_rne(acc[2][r], acc[3][r]);
                    }
                    *reinterpret_cast<uint16_t*>(base + r * kWrCRowBytes + at[0]) = (uint16_t)(o.x & 0xffffu);
                    *reinterpret_cast<uint16_t*>(base + r * kWrCRowBytes + at[1]) = (uint16_t)(o.x >> 16);
                    *reinterpret_cast<uint16_t*>(base + r * kWrCRowBytes + at[2]) = (uint16_t)(o.y & 0xffffu);
                    *reinterpret_cast<uint16_t*>(base + r * kWrCRowBytes + at[3]) = (uint16_t)(o.y >> 16);
                }
            });
            __syncthreads();
#pragma unroll 4
            for (uint32_t pass = 0; pass < (uint32_t)MT; ++pass) {
                const uint32_t row = pass * 8u + (tid >> 5);  // within the half
                const uint32_t ch = tid & 31u;
                const uint32_t gm = m0 + 8u * MT * half + row, gn = n0 + ch * 8u;
                if (gm < p.m && gn < p.n) {
                    const uint4 v = *reinterpret_cast<const uint4*>(c_rows4(row >> 2, MT, kWrCRowBytes) + (row & 3u) * kWrCRowBytes +
                                                                    (((ch >> 1) ^ ((row >> 2) & 3u)) << 5) + (ch & 1u) * 16u);
                    *reinterpret_cast<uint4*>(p.c + (size_t)gm * p.ldc + gn) = v;
                }
            }
            if constexpr (half == 0u) __syncthreads();  // the second half overwrites the staging area
        });
        acc_reserve<MT>();
        return;
    }
    // Residual and / or the SiLU gate: the fp32 sums are staged, as many blocks of 16 rows as the arrays hold at a time, and each thread
    // finishes 8 neighbouring columns of a row — bias, gate, residual, the one rounding — as the small-tile kernels do.
    const uint32_t ch = tid & 31u;  // 8 columns: 8 ch .. 8 ch + 7 of the tile
    const uint32_t gn = n0 + 8u * ch;
    float bias8[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) bias8[i] = 0.f;
    if (p.bias != nullptr && gn < p.n) {
        const uint4 raw = *reinterpret_cast<const uint4*>(p.bias + gn);
        const uint32_t d[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            bias8[2 * i] = bf16_bits_to_f32(d[i] & 0xffffu);
            bias8[2 * i + 1] = bf16_bits_to_f32(d[i] >> 16);
        }
    }
    // The residual's rows of a part are requested together, a part ahead of their use: row by row, each behind the store of the row before,
    // their trips to memory stood one behind the other with nothing else on the CU.  What bounds the part behind the loop is the residual's and
    // the outputs' bytes (us, row by row / so: 4096 x 4096 x 4096 8-bit 111.8 / 106.6, 2048 x 22016 x 4096 8-bit 334 / 297, 577 x 13824 x 5120 packed 4-bit
    // 91.8 / 88.2).  The staged rows are not turned against their bank conflicts: it is level or slower (768 x 28672 x 1024 packed 4-bit 60.8 turned, 60.0 so;
    // 4-bit 1500 x 16384 x 1024 behind a gate 58.1 / 57.7).
    constexpr uint32_t kBlocksHeld = 6u * MT / 16u, kParts = (MT + kBlocksHeld - 1u) / kBlocksHeld;
    uint4 residual[2][2u * kBlocksHeld];
    auto request_part = [&](auto part_c) {
        constexpr uint32_t first = decltype(part_c)::value * kBlocksHeld, blocks = MT - first < kBlocksHeld ? MT - first : kBlocksHeld;
        if (p.residual == nullptr) return;
#pragma unroll
        for (uint32_t pass = 0; pass < 2u * blocks; ++pass) {
            const uint32_t gm = m0 + 16u * first + pass * 8u + (tid >> 5);
            uint4& r = residual[decltype(part_c)::value & 1u][pass];
            r = make_uint4(0u, 0u, 0u, 0u);
            if (gm < p.m && gn < p.n) r = request_residual8(p, gm, gn, gated);
        }
    };
    request_part(std::integral_constant<uint32_t, 0u>{});
    for_each_const<kParts>([&](auto part_c) {
        constexpr uint32_t first = decltype(part_c)::value * kBlocksHeld, blocks = MT - first < kBlocksHeld ? MT - first : kBlocksHeld;
        for_each_const<blocks>([&](auto mh_c) {
            constexpr uint32_t mh = decltype(mh_c)::value, mt = first + mh;
            const f32x4_t acc[4] = {acc_read<4u * mt>(), acc_read<4u * mt + 1u>(), acc_read<4u * mt + 2u>(), acc_read<4u * mt + 3u>()};
            float* base = reinterpret_cast<float*>(c_rows4(4u * mh + kq, MT / 2u, kWrTile * 4u));
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r)
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) base[r * kWrTile + wcol + 16u * j] = acc[j][r];
        });
        if constexpr (decltype(part_c)::value + 1u < kParts) request_part(std::integral_constant<uint32_t, decltype(part_c)::value + 1u>{});
        __syncthreads();
        auto finish = [&](uint32_t pass, const uint4& r, auto added_c) {
            const uint32_t row = pass * 8u + (tid >> 5);  // within the part
            const uint32_t gm = m0 + 16u * first + row;
            if (gm >= p.m || gn >= p.n) return;
            const float* src = reinterpret_cast<const float*>(c_rows4(row >> 2, MT / 2u, kWrTile * 4u)) + (row & 3u) * kWrTile + 8u * ch;
            const float4 lo = *reinterpret_cast<const float4*>(src), hi = *reinterpret_cast<const float4*>(src + 4);
            float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] += bias8[i];
            if (gated) {
                float o[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = silu_gate(v[2 * i], v[2 * i + 1]);
                if constexpr (decltype(added_c)::value) {
#pragma clang fp contract(off)  // (added to the rounded product, as by every other kernel)
                    o[0] += bf16_bits_to_f32(r.x & 0xffffu);
                    o[1] += bf16_bits_to_f32(r.x >> 16);
                    o[2] += bf16_bits_to_f32(r.y & 0xffffu);
                    o[3] += bf16_bits_to_f32(r.y >> 16);
                }
                *reinterpret_cast<uint2*>(p.c + (size_t)gm * p.ldc + gn / 2u) = make_uint2(pack_bf16_rne(o[0], o[1]), pack_bf16_rne(o[2], o[3]));
            } else {
                const uint32_t d[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    v[2 * i] += bf16_bits_to_f32(d[i] & 0xffffu);
                    v[2 * i + 1] += bf16_bits_to_f32(d[i] >> 16);
                }
                *reinterpret_cast<uint4*>(p.c + (size_t)gm * p.ldc + gn) =
                    make_uint4(pack_bf16_rne(v[0], v[1]), pack_bf16_rne(v[2], v[3]), pack_bf16_rne(v[4], v[5]), pack_bf16_rne(v[6], v[7]));
            }
        };
        // (Unrolled, the residual's registers have their places.  A gate alone has none and stays a loop: unrolled and turned / so, us, 1500 x 16384 x 1024 4-bit
        // g64 58.9 / 57.7, 768 x 28672 x 1024 packed 4-bit 57.2 / 56.2, 2048 x 12288 x 1024 4-bit 61.8 / 59.3; 8-bit 60.9 / 60.0.)
        if (p.residual != nullptr) {
#pragma unroll
            for (uint32_t pass = 0; pass < 2u * blocks; ++pass) finish(pass, residual[decltype(part_c)::value & 1u][pass], std::true_type{});
        } else {
#pragma unroll 4
            for (uint32_t pass = 0; pass < 2u * blocks; ++pass) finish(pass, make_uint4(0u, 0u, 0u, 0u), std::false_type{});
        }
        __syncthreads();  // the next part overwrites the staging area
    });
    acc_reserve<MT>();
}

// Runs `tile_count` tiles of 16 x tile_blocks (0: 16) rows from `tile_first` on; with tile_halves (eight blocks), so many tiles of 256 rows as two of 128 each.
template <int BITS, bool GROUPED, bool PACKED, int MT>
static hipError_t launch_wreg_t(const GemmParams& p, hipStream_t stream)
{
    const uint32_t grid = ((p.tile_halves ? 2u : 1u) * p.tile_count + 7u) / 8u * 8u;  // a whole number of workgroups per XCD; ids past the last tile exit at once
    void (*kernel)(const GemmParams) = bfaintb_prefill_wreg_kernel<BITS, GROUPED, PACKED, MT>;
    return launch_kernel(kernel, dim3(grid, 1, 1), dim3(256, 1, 1), 0, stream, p);
}

template <int BITS, bool GROUPED, bool PACKED>
static hipError_t launch_wreg_rows(const GemmParams& p, hipStream_t stream)
{
    switch (p.tile_blocks) {
        case 8: return launch_wreg_t<BITS, GROUPED, PACKED, 8>(p, stream);
        case 10: return launch_wreg_t<BITS, GROUPED, PACKED, 10>(p, stream);
        case 12: return launch_wreg_t<BITS, GROUPED, PACKED, 12>(p, stream);
        case 14: return launch_wreg_t<BITS, GROUPED, PACKED, 14>(p, stream);
        default: return launch_wreg_t<BITS, GROUPED, PACKED, 16>(p, stream);
    }
}

template <int BITS, bool PACKED>
static hipError_t launch_wreg_scales(const GemmParams& p, hipStream_t stream)
{
    return p.group_size != 0 ? launch_wreg_rows<BITS, true, PACKED>(p, stream) : launch_wreg_rows<BITS, false, PACKED>(p, stream);
}

}  // namespace bfaintb
