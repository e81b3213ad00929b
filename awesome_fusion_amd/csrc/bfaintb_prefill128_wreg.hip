// Tiled variant, tiles of 128 columns and 32 to 256 rows, weights kept in registers: the small-tile and the tall-tile kernel, for
// row-major B and for B in the packed order (PACKED).
//
// Same job and the same reference kernel replaced as bfaintb_prefill128_kernel
// (/root/reference/bfAintBGemm/bf16gemm_kernel_gfx90a.s:184-630; the reference's own tile is 32 x 64,
// /root/reference/bfAintBGemm/bfAintBGemm.cc:105-109).  That kernel converts W into LDS and every wave reads both
// operands back: a K-step takes 0.75 us whatever the load on the machine, three times its matrix-instruction time.
// Here, as in bfaintb_prefill_wreg_kernel, only A goes through LDS:
//   4 column groups of 32 columns side by side along n, two waves each (512 threads, two waves per SIMD); a wave owns all 16 MT
//   rows x 32 columns of the tile = MT x 2 accumulators of v_mfma_f32_16x16x32_bf16, converts exactly the weights it multiplies by,
//   straight into the instruction's operand registers, and each weight of the tile is converted once.  The two waves of a column group
//   share a K-step of 64 by its blocks of 32 k (wave kh takes block kh of every step) and the epilogue adds their sums, first blocks +
//   second blocks: an output is the sum of two chains of matrix instructions, not of one as in the other tiled kernels, so it agrees
//   with them to rounding, not bit for bit (it is reproducible run to run: nothing depends on timing).
//   A and the codes come in by the asynchronous copy, 16 bytes a lane, into NS stages of LDS each, the copies of step kt + NS - 1
//   behind the barrier of step kt.  (Codes fetched by each wave itself, 16 two-byte loads a step, made a step 0.80 us: the
//   vector-memory path takes about 20 cycles for a wave's instruction whatever it moves.)
//
// What bounds a step: the instructions that a SIMD issues.  Measured with chains of independent instructions, two waves per SIMD: a
// matrix instruction holds the issue for 8 of its 16 cycles, any vector instruction beside it takes some 4.2, an LDS read some 5.  So a
// step of MT row blocks costs 64 MT cycles of matrix instructions, in whose shadow 2 vector instructions each are free, and, when there are
// too few of those, what the conversion (36 to 46 vector instructions a wave) and the reads add.  Hence
//   - the tall tiles: 16 blocks share one conversion.  us, 4 waves of 128 x 64 (bfaintb_prefill256x128_wreg_kernel) / this: 2048 x 4096 x
//     4096 8-bit 70.8 / 63.0; 512 x 11008 x 4096 8-bit 63.0 / 52.1, 4-bit 71.6 / 53.9; 512 x 13824 x 5120 packed 4-bit 85.4 / 73.1.
//   - no row blocks that do not exist: MT = 2, 4, 6, 8, 10, 12, 16, the rows spread evenly over the tiles (96 x 20480 x 4096 packed 8-bit 32.9
//     with eight blocks / 29.1 with six).
//   - the conversion by half-precision magic numbers (bfaintb_device.hpp) and codes by transposing reads: 42 vector and 16 LDS instructions a
//     wave and step of eight blocks before, 34 and 10 now, counted in the compiled loop for 8-bit codes and a scale for each column (64 x 4096 x
//     11008 8-bit unsplit, codes in the last-level cache: 55.9 -> 49.2); 38 to 43 vector ones with group scales, whose multipliers are new every step.
//   - the conversion spread over the slots an instruction or a pair of weights at a time, each where the schedule below puts it, and none
//     where the codes are still on their way: a pair's two products and its rounding pack are one piece of assembly, so that the compiler, which
//     fenced them with idle cycles (8 to 11 a step, each of the next instruction's time), sees one result; 2 to 4 are left.  The copies'
//     requests are spread likewise.  us before / after: 128 x 20480 x 4096 packed 4-bit g128 31.7 / 29.7, 192 x 16384 x 4096 32.6 / 31.5, 64 x
//     20480 x 4096 packed 4-bit 22.6 / 21.5; over 40000 random shapes of 17 to 700 rows 1.3 % on average, 2.2 % for 33 to 64 rows.
//   - more stages the fewer rows there are, since such launches read their codes from memory and wait for it: 64 x 4096 x 11008 8-bit
//     unsplit, codes cold, 4 / 8 stages 69.2 / 63.1; 96 rows 4-bit g128, 4 / 6 stages 88.9 / 78.6.
//   - for 17 to 32 rows, whose calls read every code once, from memory: the copying wave and eight stages whatever the codes (32 x 22016 x
//     4096, one row of 172 tiles, us with / without: 4-bit g128 in rows 21.5 / 23.9; 8-bit in rows 24.3 / 24.1), and a walk over k that each
//     tile of packed 8-bit codes starts at a step of its own, so that the column blocks, a power of two apart, are not all read at the
//     same place at once (22016 x 4096 22.5 without / 21.3, 28672 x 8192 44.6 / 43.5; 4-bit codes lose by it, 38.6 / 39.9).  A step of
//     two row blocks takes 0.25 to 0.3 us: 16 waves in two halves of k, each with stages of its own, were no faster (32 x 22016 x 4096 8-bit
//     in rows 27.1, 28672 x 8192 packed 4-bit 41.9 against 38.9): the vector instructions of the conversion bound it, not a wait.
// With a workgroup on every CU the clock gives way to the board's power on top (16 blocks: 0.60 us a step on 96 CUs, 0.82 on 256).
// Accumulator (mt, j), register r of lane (c16 = lane % 16, q = lane / 16): row 16 mt + 4 q + r, column 32 w + 16 j + c16 of the tile.
// Epilogue: as bfaintb_prefill128_kernel — fp32 sums staged in LDS in [m][n] order, each thread finishes 8 neighbouring
// columns of a row (bias, SiLU gate, residual, the one rounding) and stores them with one 16-byte write.
#include <utility>
#include "bfaintb_device.hpp"

namespace bfaintb {

namespace {
constexpr uint32_t kTw = 128, kTwK = 64;

__device__ __forceinline__ uint32_t tw_swz(uint32_t row, uint32_t chunk) { return row * 128u + ((chunk ^ ((row >> 1) & 7u)) << 4); }

// acc += a x b with the accumulator pinned to the accumulation registers and updated in place: written as assembly
// because the compiler gives some of the kernel's matrix instructions a destination other than their source and copies
// the sums back (21 of 224 instructions, 150 accumulator moves).  Behind the assembly its hazard bookkeeping sees
// nothing, so: the operands are written long before (LDS reads and conversions, under wait counts the compiler does
// insert for assembly operands); the accumulators are written by ordinary instructions only at the very start, with the
// whole prologue between that and the first matrix instruction, and read by them only in the epilogue, behind explicit
// idle cycles (tw_settle).
__device__ __forceinline__ void tw_mfma(f32x4_t& acc, const bf16x8_t& a, const bf16x8_t& b)
{
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
// The idle cycles, and behind them every accumulator as an operand: with the idle cycles alone nothing keeps the compiler from
// moving an accumulator to an ordinary register ahead of them (it did so for the last one of sixteen row blocks).
template <int MT>
__device__ __forceinline__ void tw_settle(f32x4_t (&acc)[MT][2])
{
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int j = 0; j < 2; ++j) asm volatile("" : "+a"(acc[mt][j]));
}
}  // namespace

// The order of a step's conversion: what column 0 needs, then its pairs with the instructions that column 1 needs between them, then column 1's pairs.
struct TwOp {
    bool pair;  // three instructions, or one
    uint32_t column, index;
};
template <uint32_t PREPARE>
struct TwSchedule {
    static constexpr uint32_t kCount = 2u * PREPARE + 8u, kInstructions = 2u * PREPARE + 24u;
    static constexpr TwOp op(uint32_t at)
    {
        if (at < PREPARE) return TwOp{false, 0u, at};
        at -= PREPARE;
        for (uint32_t b = 0; b < 4u; ++b) {
            const uint32_t from = b * PREPARE / 4u, to = (b + 1u) * PREPARE / 4u;
            if (at == 0u) return TwOp{true, 0u, b};
            at -= 1u;
            if (at < to - from) return TwOp{false, 1u, from + at};
            at -= to - from;
        }
        return TwOp{true, 1u, at};
    }
    static constexpr uint32_t before(uint32_t at)  // instructions
    {
        uint32_t n = 0;
        for (uint32_t i = 0; i < at; ++i) n += op(i).pair ? 3u : 1u;
        return n;
    }
};

// The LDS of a workgroup, one array for each stage and kind (A, codes, scales): the compiler then sees that a stage's reads do not
// depend on the copies into the others.
template <uint32_t BYTES, char KIND, uint32_t STAGE>
__shared__ __attribute__((aligned(1024))) uint8_t tw_lds[BYTES];

// One tile: 16 MT rows from row m0, 128 columns from column n0, the K-steps of split ks.  NS: stages; SCALES: group scales go through
// LDS.
template <int BITS, bool GROUPED, bool PACKED, bool SCALES, int MT, int NS, bool COPIER>
__device__ __forceinline__ void tw_tile(const GemmParams& p, const uint32_t m0, const uint32_t n0, const uint32_t ks)
{
    static_assert(MT >= 2 && MT <= 16, "blocks of 16 rows");
    constexpr uint32_t kAhead = MT < 4 ? MT : 4;       // units that the fragments of A are read ahead
    static_assert((NS == 4 || NS == 6 || NS == 8) && NS * MT % kAhead == 0, "the fragments' rotation comes round with the stages");
    constexpr uint32_t kRows = 16u * MT;               // rows of a tile
    constexpr uint32_t kACopies = (MT + 3u) / 4u;      // of A, per wave and step: 8 rows each
    constexpr uint32_t kStageRows = MT < 4 ? kRows : 64u * kACopies;  // rows of a stage of A (those past the tile's are zero and not read)
    constexpr uint32_t kRowBytes = 128u * BITS / 8u;   // a tile row of codes
    constexpr bool kScalesInLds = GROUPED && SCALES;   // group scales come by the copy engine as well
    using C0 = std::integral_constant<uint32_t, 0>;
    using C1 = std::integral_constant<uint32_t, 1>;
    using C2 = std::integral_constant<uint32_t, 2>;
    using C3 = std::integral_constant<uint32_t, 3>;
    using C4 = std::integral_constant<uint32_t, 4>;
    using C5 = std::integral_constant<uint32_t, 5>;
    using C6 = std::integral_constant<uint32_t, 6>;
    using C7 = std::integral_constant<uint32_t, 7>;
    constexpr uint32_t kDepth = NS - 1u;  // steps ahead that the copies run
    auto s_tile = [&](auto stage_c) -> uint8_t* { return tw_lds<512u, 's', decltype(stage_c)::value>; };
    auto w_tile = [&](auto stage_c) -> uint8_t* { return tw_lds<8192u, 'w', decltype(stage_c)::value>; };
    auto a_tile = [&](auto stage_c) -> uint8_t* { return tw_lds<kStageRows * 128u, 'a', decltype(stage_c)::value>; };
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wc = wave & 3u;                  // the wave's 32 columns
    const uint32_t kh = wave >> 2;                  // two waves per column group: the block of 32 k this one multiplies
    const uint32_t c16 = lane & 15u, kq = lane >> 4;

    const uint32_t rows_valid = p.m - m0 < kRows ? p.m - m0 : kRows;
    const uint32_t a_extent = ((rows_valid - 1u) * p.lda + p.k) * 2u;
    const __amdgpu_buffer_rsrc_t rsrc_a =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.a + (size_t)m0 * p.lda), 0, (int)a_extent, kBufferFlags);
    const uint32_t cols_valid = p.n - n0 < kTw ? p.n - n0 : kTw;
    // packed weights: a block of 16 columns is one run of k x 16 codes in chunks of 1024 bytes (64 rows of 8-bit, 128 rows
    // of 4-bit codes); the tile's 8 column blocks follow one another, and one past n reads as zero through the extent
    const uint32_t slab_bytes = p.k * (BITS == 8 ? 16u : 8u);
    const uint32_t b_extent = PACKED ? cols_valid / 16u * slab_bytes : (p.k - 1u) * p.ldb_bytes + (BITS == 8 ? cols_valid : cols_valid / 2u);
    const __amdgpu_buffer_rsrc_t rsrc_b =
        PACKED ? __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.b + (size_t)(n0 / 16u) * slab_bytes), 0,
                                                   (int)b_extent, kBufferFlags)
               : __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.b + (BITS == 8 ? n0 : n0 / 2u)), 0,
                                                   (int)b_extent, kBufferFlags);

    // K-steps of this workgroup: all of them, or the share of split ks (p.k_per_wg rows each; the host makes sure
    // every split has at least one).  kt below counts within the share; kbase + kt is the step of the whole matrix.
    const uint32_t ksteps_all = (p.k + kTwK - 1u) / kTwK;
    const uint32_t kbase = ks * (p.k_per_wg / kTwK);
    const uint32_t ksteps = p.k_per_wg / kTwK < ksteps_all - kbase ? p.k_per_wg / kTwK : ksteps_all - kbase;
    const uint32_t last_chunks = (p.k - (ksteps_all - 1u) * kTwK) / 8u;  // valid 16-byte chunks per row of A in the last step
    auto clamp = [&](uint32_t t) { return t < ksteps ? t : ksteps - 1u; };
    // The K-step of the whole matrix that step t of the share is.  Few rows of packed 8-bit codes: each tile starts its walk at a step of its
    // own (see the head of the file).
    const uint32_t rotate = PACKED && BITS == 8 && MT < 4 ? (n0 / kTw) % ksteps : 0u;
    auto at_step = [&](uint32_t t) -> uint32_t {
        if constexpr (PACKED && BITS == 8 && MT < 4) {
            const uint32_t r = t + rotate;
            return kbase + (r < ksteps ? r : r - ksteps);
        } else {
            return kbase + t;
        }
    };

    // A copy: instruction j of wave w fills rows 8 (kACopies w + j) .. + 7; lane l lands at row + l / 8, chunk position l % 8, so
    // it fetches chunk (l % 8) ^ ((row >> 1) & 7) = (l % 8) ^ (l / 16) for even kACopies w + j and that ^ 4 for odd ones; the row
    // advance of j and the K advance sit in the scalar offset.  A chunk past the end of k (partial last step) is fetched from
    // beyond the extent and reads as zero; rows of B past k read as zero codes, finite weights, and multiply those zeros.
    // (a stage of fewer than 64 rows: several waves copy the same 8 rows to the same place, so that all have as many requests in flight)
    const uint32_t a_block = kStageRows < 64u ? wave & (kStageRows / 8u - 1u) : kACopies * wave;  // the wave's first 8 rows
    const uint32_t a_row = 8u * a_block + (lane >> 3);
    const uint32_t chunk_e = (lane & 7u) ^ ((lane >> 4) & 7u) ^ (4u * (a_block & 1u)), chunk_o = chunk_e ^ 4u;
    const uint32_t a_voff_e = (a_row * p.lda + chunk_e * 8u) * 2u, a_voff_o = (a_row * p.lda + chunk_o * 8u) * 2u;
    const uint32_t a_last_e = chunk_e < last_chunks ? a_voff_e : a_extent, a_last_o = chunk_o < last_chunks ? a_voff_o : a_extent;
    auto dma_a = [&](auto stage_c, uint32_t kt) {
        uint8_t* base = a_tile(stage_c) + a_block * 1024u;
        const bool last = at_step(kt) + 1u == ksteps_all;
        const uint32_t ve = last ? a_last_e : a_voff_e, vo = last ? a_last_o : a_voff_o;
#pragma unroll
        for (uint32_t j = 0; j < kACopies; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (__attribute__((address_space(3))) void*)(base + j * 1024u), 16,
                                                     (j & 1u) ? vo : ve, at_step(kt) * kTwK * 2u + j * 16u * p.lda, 0, 0);
    };

    // W codes.  Copy: a 16-byte-per-lane instruction fills 1024 bytes = kRowsPerCopy rows of the stage; the step's 64
    // rows take kCopies instructions, kCopiesPerWave for each wave.  Lane l lands at row l / kChunks of its block, chunk
    // position l % kChunks, and fetches the chunk that belongs there: position = chunk ^ turn(row), chosen so that the
    // transposing reads below find 16 rows of a column block in 16 different groups of banks.
    //
    // Packed weights: the chunk of a column block that holds the step (1024 bytes: all of it for 8-bit codes; for 4-bit
    // codes it spans two steps and is copied for each) is one instruction and lies in LDS as it lies in memory: piece
    // 16 kg + nl of 16 bytes = rows 8 kg .. + 7 of both K-blocks (4-bit: of four), column nl; wave w copies column block w.
    constexpr uint32_t kChunks = kRowBytes / 16u;        // 8 or 4 chunks per row
    // One instruction a wave and step (4-bit codes in rows: 8 rows, half of it — the other lanes fetch from beyond the extent, and
    // the stage has a gap of 512 bytes behind every 8 rows — so that every wave has the same number of requests in flight for the
    // one wait count at the top of a step and none fetches what another does).
    auto row_at = [](uint32_t row) { return BITS == 8 ? row * 128u : (row >> 3) * 1024u + (row & 7u) * 64u; };
    auto turn = [](uint32_t row) { return BITS == 8 ? (row ^ (row >> 3)) & 7u : (row >> 2) & 3u; };
    uint32_t w_voff;
    if constexpr (PACKED) {
        w_voff = wave * slab_bytes + lane * 16u;
    } else {
        const uint32_t row = 8u * wave + (lane / kChunks & 7u);  // within the step
        w_voff = BITS == 8 || lane < 32u ? row * p.ldb_bytes + ((lane % kChunks) ^ turn(row)) * 16u : b_extent;
    }
    // where step kt's codes start, beyond the lane's offset: w_step * (kbase + kt >> w_shift)
    const uint32_t w_step = PACKED ? 1024u : kTwK * p.ldb_bytes;
    constexpr uint32_t w_shift = (PACKED && BITS == 4) ? 1u : 0u;
    auto dma_w = [&](uint8_t* stage, uint32_t kt) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (__attribute__((address_space(3))) void*)(stage + wave * 1024u), 16, w_voff,
                                                 (at_step(kt) >> w_shift) * w_step, 0, 0);
    };
    // Read: lane (c16, kq) of the wave takes, of its block of 32 k, rows 8 kq .. 8 kq + 7 of columns 16 j + c16, j = 0, 1, of the
    // wave's 32: 8 bytes (8-bit codes) or 4 for each.
    //   rows, 8-bit: one transposing read for each j (ds_read_b64_tr_b8: the 16 lanes of a kq address 8 rows x 16 bytes, lane 2 r + h
    //     the half h of row r, and lane i receives byte i of each of the 8 rows);
    //   rows, 4-bit: one for both (ds_read_b64_tr_b4: lane r addresses 8 bytes, 16 codes, of its own, and lane i receives code i of all
    //     16: eight rows of column block 0 by lanes 0 .. 7, the same rows of block 1 by the others);
    //   packed: the lane's own piece.
    // As 16 rows of 2-byte reads (8 a wave) these were a fifth of the step's LDS instructions, which hold a SIMD's issue for some 5
    // cycles each.
    const uint32_t w_row = 32u * kh + 8u * kq + (BITS == 8 ? c16 >> 1 : c16 & 7u);
    auto w_at = [&](uint32_t j) -> uint32_t {
        if constexpr (PACKED) return (2u * wc + j) * 1024u + lane * 16u + (BITS == 8 ? 8u : 4u) * kh;
        else if constexpr (BITS == 8) return row_at(w_row) + (((2u * wc + j) ^ turn(w_row)) << 4) + 8u * (c16 & 1u);
        else return row_at(w_row) + ((wc ^ turn(w_row)) << 4) + (c16 & 8u);
    };
    const uint32_t w_rd[2] = {w_at(0), w_at(1)};
    struct Codes {
        uint32_t d[2][BITS / 4];  // [column j]: 8-bit: rows 0 .. 3 and 4 .. 7 in the bytes of a dword; 4-bit: 8 rows in the nibbles of one
    };
    auto read_codes = [&](Codes& c, const uint8_t* stage, uint32_t kt) {
        typedef int v2i __attribute__((ext_vector_type(2)));
        typedef __attribute__((address_space(3))) v2i* lds_v2i;
        if constexpr (BITS == 8) {
#pragma unroll
            for (uint32_t j = 0; j < 2; ++j) {
                if constexpr (PACKED) {
                    const u32x2_t v = *reinterpret_cast<const u32x2_t*>(stage + w_rd[j]);
                    c.d[j][0] = v[0], c.d[j][1] = v[1];
                } else {
                    const v2i v = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i)(const_cast<uint8_t*>(stage) + w_rd[j]));
                    c.d[j][0] = (uint32_t)v[0], c.d[j][1] = (uint32_t)v[1];
                }
            }
        } else if constexpr (PACKED) {
#pragma unroll
            for (uint32_t j = 0; j < 2; ++j) c.d[j][0] = *reinterpret_cast<const uint32_t*>(stage + w_rd[j] + 8u * (at_step(kt) & 1u));
        } else {
            const v2i v = __builtin_amdgcn_ds_read_tr4_b64_v2i32((lds_v2i)(const_cast<uint8_t*>(stage) + w_rd[0]));
            c.d[0][0] = (uint32_t)v[0], c.d[1][0] = (uint32_t)v[1];
        }
    };
    // Scales go through a buffer resource so that the load is issued whatever the lane's column (the wait counts
    // below count requests): columns past n read other columns' scales, or zero beyond the array; their results are
    // never stored.
    const uint32_t scale_rows = GROUPED ? p.k / p.group_size : 1u;
    const __amdgpu_buffer_rsrc_t rsrc_s = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(p.scale), 0, (int)(((scale_rows - 1u) * p.lds + p.n) * 2u), kBufferFlags);
    const uint32_t wcol = 32u * wc + c16;  // the lane's column j of the tile: wcol + 16 j
    const uint32_t s_voff = (n0 + wcol) * 2u;
    struct Scales {
        uint32_t s[2];  // bf16
    };
    auto load_scales = [&](Scales& sr, uint32_t row_off) {
#pragma unroll
        for (uint32_t j = 0; j < 2; ++j) sr.s[j] = __builtin_amdgcn_raw_buffer_load_b16(rsrc_s, s_voff + 32u * j, row_off, 0);
    };
    auto group_offset = [&](uint32_t kt, uint32_t block) {  // of the scale row of a block of 32 k of step kt
        uint32_t g = group_of_row(p, at_step(kt) * kTwK + 32u * block);
        if (g >= scale_rows) g = scale_rows - 1u;  // rows past k in a partial last step: any scale will do
        return g * p.lds * 2u;
    };
    // Group scales by the copy engine: the tile's 128 scales for each of a step's two blocks of 32 k, 4 bytes a lane, wave w the block
    // w % 2 (four waves the same bytes to the same place: every wave has the same number of requests).  Fetched by every wave into
    // registers, two gathers a step, they hold up the memory path for longer (some 16 cycles each) than one copy does.
    auto dma_s = [&](uint8_t* stage, uint32_t kt) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_s, (__attribute__((address_space(3))) void*)(stage + (wave & 1u) * 256u), 4, n0 * 2u + lane * 4u,
                                                 group_offset(kt, wave & 1u), 0, 0);
    };
    auto read_scales = [&](Scales& sr, const uint8_t* stage) {
#pragma unroll
        for (uint32_t j = 0; j < 2; ++j) sr.s[j] = *reinterpret_cast<const uint16_t*>(stage + kh * 256u + (wcol + 16u * j) * 2u);
    };

    // The copying wave (COPIER: one wave more than those that compute): every copy of the K loop is its request; the computing waves,
    // which issue in order, are spared four instructions a step of the memory path and the scalar ones that prepare them.
    if (COPIER && wave == 8u) {
        const uint32_t pc_e = (lane & 7u) ^ ((lane >> 4) & 7u), pc_o = pc_e ^ 4u;
        const uint32_t pa_e = ((lane >> 3) * p.lda + pc_e * 8u) * 2u, pa_o = ((lane >> 3) * p.lda + pc_o * 8u) * 2u;
        const uint32_t pl_e = pc_e < last_chunks ? pa_e : a_extent, pl_o = pc_o < last_chunks ? pa_o : a_extent;
        constexpr uint32_t kCodeCopies = 8u;
        uint32_t pw[kCodeCopies];
#pragma unroll
        for (uint32_t j = 0; j < kCodeCopies; ++j) {
            const uint32_t row = 8u * j + (lane / kChunks & 7u);
            pw[j] = PACKED ? j * slab_bytes + lane * 16u : BITS == 8 || lane < 32u ? row * p.ldb_bytes + ((lane % kChunks) ^ turn(row)) * 16u : b_extent;
        }
        constexpr uint32_t kStepCopies = kStageRows / 8u + kCodeCopies + (kScalesInLds ? 2u : 0u);
        auto copy_step = [&](auto stage_c, uint32_t kt) {
            const bool last = at_step(kt) + 1u == ksteps_all;
            const uint32_t ve = last ? pl_e : pa_e, vo = last ? pl_o : pa_o;
#pragma unroll
            for (uint32_t j = 0; j < kCodeCopies; ++j)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (__attribute__((address_space(3))) void*)(w_tile(stage_c) + j * 1024u), 16, pw[j],
                                                         (at_step(kt) >> w_shift) * w_step, 0, 0);
            if constexpr (kScalesInLds) {
#pragma unroll
                for (uint32_t h = 0; h < 2; ++h)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_s, (__attribute__((address_space(3))) void*)(s_tile(stage_c) + h * 256u), 4, n0 * 2u + lane * 4u,
                                                             group_offset(kt, h), 0, 0);
            }
#pragma unroll
            for (uint32_t j = 0; j < kStageRows / 8u; ++j)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (__attribute__((address_space(3))) void*)(a_tile(stage_c) + j * 1024u), 16, (j & 1u) ? vo : ve,
                                                         at_step(kt) * kTwK * 2u + j * 16u * p.lda, 0, 0);
        };
        // The first two steps' copies are shared out over the computing waves, which wait for them before they start; those of the steps behind
        // them are this wave's, in flight meanwhile and counted by its own waits.  (Shared out as well and waited for at the start, a machine's
        // whole pipeline had to land first.  us before / now: 32 x 22016 x 4096 4-bit g128 23.4 / 22.4, 32 x 28672 x 4096 packed 8-bit 24.5 / 23.1, 26 x
        // 23392 x 3584 packed 4-bit 17.3 / 16.2, 54 x 22192 x 1152 packed 4-bit 10.0 / 9.3; four stages or many steps level.)
        auto ahead = [&](auto stage_c) {
            if constexpr (decltype(stage_c)::value < kDepth) copy_step(stage_c, clamp(decltype(stage_c)::value));
        };
        ahead(C2{}), ahead(C3{}), ahead(C4{}), ahead(C5{}), ahead(C6{});
        barrier_no_fence();
        uint32_t kt = 0;
        auto turn_of = [&](auto stage_c) {  // step kt + stage
            constexpr uint32_t St = decltype(stage_c)::value;
            if constexpr (St < (uint32_t)NS) {
                if (kt + St >= ksteps) return;
                // the computing waves start this step behind this barrier: the copies of it and of the next have landed when at most
                // those of the steps behind are in flight (a wait counts 63 at most).  Steps 0 and 1 are not among this wave's: the computing waves'
                // wait for all of theirs and the prologue's barrier cover them, and the count here begins with steps 2 .. kDepth - 1 in flight
                constexpr uint32_t kAllowed = (kDepth - 2u) * kStepCopies;
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kAllowed < 63u ? kAllowed : 63u) : "memory");
                barrier_no_fence();
                copy_step(std::integral_constant<uint32_t, (St + kDepth) % NS>{}, clamp(kt + St + kDepth));  // a stage that every wave has left
            }
        };
        for (; kt < ksteps; kt += NS) turn_of(C0{}), turn_of(C1{}), turn_of(C2{}), turn_of(C3{}), turn_of(C4{}), turn_of(C5{}), turn_of(C6{}), turn_of(C7{});
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();  // the epilogue's first barrier: nothing is writing LDS any more
        return;           // (a wave that has ended no longer counts at the barriers that follow)
    }

    // ---- Conversion by halves (bfaintb_device.hpp has the argument): 4 (8-bit) and 4.25 (4-bit) instructions for two weights, where a
    // conversion, a multiplication and the pack take 5 to 7; the step is bound by the instructions a SIMD issues, some 4 cycles each
    // beside its matrix instructions.
    // (4-bit codes with group scales, whose multipliers are new every step: two of them and two shifts more, good for every scale of the format)
    constexpr int kUpper = BITS == 4 && GROUPED ? 64 : 1024;
    constexpr bool kLimited = kUpper == 1024;  // scales beyond the conversion go a second way along k
    typedef HalfMultipliers<BITS, kUpper> Multiplier;
    struct Multipliers {
        Multiplier h[2];
    };
    float most = 0.f;  // the largest magnitude among the lane's scales
    auto multipliers = [&](Multipliers& mu, const Scales& sr) {
#pragma unroll
        for (uint32_t j = 0; j < 2; ++j) mu.h[j] = Multiplier(bf16_bits_to_f32(sr.s[j]));
        if constexpr (kLimited) largest_scale(most, mu.h[0].s, mu.h[1].s);
    };
    HalfConstants<BITS, kUpper> half_k;
    half_k.keep();
    struct Ops {
        uint32_t w[2][4];  // [column j][dword]: the 8-element operand as 4 packed pairs
    };
    Multipliers fixed;  // one scale per column
    if constexpr (!GROUPED) {
        Scales sr;
        load_scales(sr, 0);
        multipliers(fixed, sr);
    }
    auto convert_all = [&](Ops& ops, const Codes& c, const Scales& sr) {
        Multipliers mu = fixed;
        if constexpr (GROUPED) multipliers(mu, sr);
#pragma unroll
        for (uint32_t j = 0; j < 2; ++j) {
            if constexpr (BITS == 4) {
                const uint4 w = weights4_by_halves(c.d[j][0], half_k, mu.h[j]);
                ops.w[j][0] = w.x, ops.w[j][1] = w.y, ops.w[j][2] = w.z, ops.w[j][3] = w.w;
            } else {
#pragma unroll
                for (uint32_t pr = 0; pr < 4u; ++pr)
                    ops.w[j][pr] = pack_bf16_rne(weight_of_half<0>(halves<0>(c.d[j][pr >> 1], half_k), pr & 1u, mu.h[j]),
                                                 weight_of_half<1>(halves<1>(c.d[j][pr >> 1], half_k), pr & 1u, mu.h[j]));
            }
        }
    };
    // In a step: what a column needs before its products, one vector instruction at a time, each held where it is written, and its four pairs of
    // rows (4-bit codes: pairs 0, 2, 1, 3, as the halves lie).
    struct Conversion {
        uint32_t h[2][4], x[3];
        Multiplier mu[2];
    };
    constexpr uint32_t kHalvesOps = BITS == 8 ? 4u : kUpper == 64 ? 7u : 5u, kPrepareOps = kHalvesOps + (GROUPED ? 2u : 0u);
    auto prepare = [&](Conversion& w, const Codes& c, const Scales& sr, auto j_c, auto op_c) {
        constexpr uint32_t j = decltype(j_c)::value, at = decltype(op_c)::value;
        // (group scales: the widening first, the offset three instructions on)
        constexpr uint32_t kWiden = 100u, kOffset = 101u;
        constexpr uint32_t op = !GROUPED ? at : at == 0u ? kWiden : at == 3u ? kOffset : at < 3u ? at - 1u : at - 2u;
        uint32_t (&h)[4] = w.h[j];
        if constexpr (op == kWiden) {
            uint32_t bits = sr.s[j];
            hold(bits);  // (or the widening moves up to the load, a step's wait with it)
            w.mu[j].s = bf16_bits_to_f32(bits), hold(w.mu[j].s);
        } else if constexpr (op == kOffset) {
            w.mu[j].o = Multiplier(w.mu[j].s).o, hold(w.mu[j].o);
            if constexpr (kLimited && j == 1u) largest_scale(most, w.mu[0].s, w.mu[1].s);
        } else if constexpr (BITS == 8) {
            h[op] = (op & 1u) == 0u ? halves<0>(c.d[j][op >> 1], half_k) : halves<1>(c.d[j][op >> 1], half_k);
            hold(h[op]);
        } else if constexpr (kUpper == 64) {
            if constexpr (op == 0u) w.x[0] = c.d[j][0] << 4, hold(w.x[0]);
            if constexpr (op == 1u) w.x[1] = c.d[j][0] >> 4, hold(w.x[1]);
            if constexpr (op == 2u) h[0] = halves<1>(w.x[0], half_k), hold(h[0]);
            if constexpr (op == 3u) w.x[2] = c.d[j][0] >> 8, hold(w.x[2]);
            if constexpr (op == 4u) h[1] = halves<1>(c.d[j][0], half_k), hold(h[1]);
            if constexpr (op == 5u) h[2] = halves<1>(w.x[1], half_k), hold(h[2]);
            if constexpr (op == 6u) h[3] = halves<1>(w.x[2], half_k), hold(h[3]);
        } else {
            if constexpr (op == 0u) w.x[0] = c.d[j][0] >> 8, hold(w.x[0]);
            if constexpr (op == 1u) h[0] = halves<0>(c.d[j][0], half_k), hold(h[0]);
            if constexpr (op == 2u) h[1] = halves<1>(c.d[j][0], half_k), hold(h[1]);
            if constexpr (op == 3u) h[2] = halves<0>(w.x[0], half_k), hold(h[2]);
            if constexpr (op == 4u) h[3] = halves<1>(w.x[0], half_k), hold(h[3]);
        }
    };
    auto make_pair = [&](Ops& ops, const Conversion& w, auto j_c, auto b_c) {
        constexpr uint32_t j = decltype(j_c)::value, b = decltype(b_c)::value;
        const Multiplier& mu = GROUPED ? w.mu[j] : fixed.h[j];
        uint32_t& to = ops.w[j][BITS == 8 ? b : (b & 1u) * 2u + (b >> 1)];
        if constexpr (BITS == 4 && kUpper == 1024) to = pair_of_halves<(b & 1u)>(w.h[j][b & 2u], w.h[j][(b & 2u) + 1u], mu.s, mu.o, mu.s4, mu.o4);
        else to = pair_of_halves<(b & 1u)>(w.h[j][b & 2u], w.h[j][(b & 2u) + 1u], mu.s, mu.o, mu.s, mu.o);
    };

    f32x4_t acc[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[mt][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // fragment mt: row 16 mt + c16 of the tile, chunk 4 kh + kq (the swizzle repeats every 16 rows)
    bf16x8_t af[kAhead];  // the fragments of the next few units, carried from step to step
    const uint32_t a_rd = tw_swz(c16, 4u * kh + kq);

    // One K-step.  `cur`: the operands of this step; `nxt` receives those of step kt + 1, converted from the codes in stage
    // S + 1; stage S holds this step's A; the copies of step kt + kDepth go into stage S - 1, which every wave finished
    // reading (A during step kt - 1, the codes during step kt - 2) before the barrier at the top.
    // The step is written as 2 MT fenced slots of one matrix instruction plus a few others: unit u = row block u has two slots (the
    // wave's two column groups);
    //   slot 0 of unit u: the A fragment of unit u + kAhead (the last kAhead units fetch the next step's first
    //          fragments: its stage is complete, see the wait below)
    //   slot 1 of unit u: one memory request (with group scales: those first, in unit 0; then the copies)
    // The conversion's instructions and the requests are spread evenly over the slots (several waves' requests behind one another hold all of
    // them up).
    // (fragments rotate through af[]: MT units leave the rotation MT % 4 further on, and four steps bring it back)
    constexpr uint32_t kSlots = 2u * MT;
    Scales ring[NS];  // group scales that do not go through LDS: those of step kt in ring[kt % NS]
    constexpr bool kRing = GROUPED && !kScalesInLds;
    constexpr uint32_t kRequests = kACopies + 1u + (kScalesInLds ? 1u : 0u);  // copies of a wave and step
    typedef TwSchedule<kPrepareOps> Schedule;
    // The first slots are left to the codes' read: five of six blocks' twelve, where two of them waited for it (284 x 10624 x 2560 packed 4-bit, us
    // with 2 / 3 / 5 / 6: 21.2 / 20.0 / 19.6 / 19.4; 259 x 4960 x 14208 packed 8-bit g128 59.0 / 56.4 / 56.0 / 55.6; sixteen blocks don't mind).
    // With fewer blocks there are none to spare: three where the multipliers or the packed order's reads come first, none for 8-bit codes in
    // rows (64 x 4096 x 11008 20.5 with none, 20.9 with three; packed 4-bit 64 x 20480 x 4096 21.7 / 21.5).
    constexpr uint32_t kFree = MT >= 6 ? 5u : MT >= 4 ? (GROUPED || PACKED || BITS == 4 ? 3u : 0u) : 1u;
    auto op_slot = [](uint32_t i) constexpr -> uint32_t { return kFree + Schedule::before(i) * (kSlots - kFree) / Schedule::kInstructions; };
    // (few blocks: as early as they can be, since those launches wait for memory: 40 x 4096 x 11008 8-bit 19.2 spread / 18.7)
    auto request_unit = [](uint32_t q) constexpr -> uint32_t {
        constexpr uint32_t first = kRing ? 1u : 0u, units = (uint32_t)MT - first;
        return first + (MT >= 6 ? q * units / kRequests : q < units ? q : units - 1u);
    };
    auto step = [&](auto stage_c, uint32_t kt, const Ops& cur, Ops& nxt) {
        constexpr uint32_t S = decltype(stage_c)::value;
        constexpr uint32_t kTurn = S * (uint32_t)MT % kAhead;
        using Next = std::integral_constant<uint32_t, (S + 1u) % NS>;
        using Target = std::integral_constant<uint32_t, (S + kDepth) % NS>;
        // At most the copies of the steps kt + 2 .. kt + kDepth - 1 may still be in flight: then this wave's part of this step's
        // AND the next step's A and codes has landed.  Behind the barrier every wave's has.  (Group scales in registers: two
        // requests a step, of which only the last step's are sure to be younger than those copies while the first steps' are still among them.)
        if constexpr (!COPIER) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kDepth - 2u) * kRequests + (kRing ? 2u : 0u)) : "memory");
        barrier_no_fence();  // (a fenced barrier would also wait for the copies of the steps ahead)
        const uint32_t kt3 = clamp(kt + kDepth);
        const bool last3 = at_step(kt3) + 1u == ksteps_all;
        const uint32_t ve = last3 ? a_last_e : a_voff_e, vo = last3 ? a_last_o : a_voff_o;
        uint8_t* const a_dst = a_tile(Target{}) + a_block * 1024u;
        const uint8_t* const a_src = a_tile(stage_c) + a_rd;
        const uint8_t* const a_nxt = a_tile(Next{}) + a_rd;
        const uint8_t* const w_src = w_tile(Next{});
        Codes code;  // of step kt + 1
        Conversion conv;
        Scales sr;
        if constexpr (kScalesInLds) read_scales(sr, s_tile(Next{}));
        else sr = ring[(S + 1u) % NS];
        read_codes(code, w_src, kt + 1u);
        __builtin_amdgcn_sched_barrier(0);
        const bf16x8_t wf0 = __builtin_bit_cast(bf16x8_t, make_uint4(cur.w[0][0], cur.w[0][1], cur.w[0][2], cur.w[0][3]));
        const bf16x8_t wf1 = __builtin_bit_cast(bf16x8_t, make_uint4(cur.w[1][0], cur.w[1][1], cur.w[1][2], cur.w[1][3]));
        bf16x8_t a_now;
        for_each_const<kSlots>([&](auto slot_c) {
            constexpr uint32_t slot = decltype(slot_c)::value, u = slot >> 1;
            if constexpr ((slot & 1u) == 0u) {
                constexpr uint32_t at = (u + kTurn) % kAhead;
                a_now = af[at];
                tw_mfma(acc[u][0], a_now, wf0);
                if constexpr (u + kAhead < (uint32_t)MT) af[at] = *reinterpret_cast<const bf16x8_t*>(a_src + (u + kAhead) * 2048u);
                else af[at] = *reinterpret_cast<const bf16x8_t*>(a_nxt + (u + kAhead - (uint32_t)MT) * 2048u);
            } else {
                tw_mfma(acc[u][1], a_now, wf1);
                if constexpr (kRing && u == 0u) load_scales(ring[S], group_offset(clamp(kt + NS), kh));
                constexpr uint32_t from = COPIER ? 0u : first_at_least<kRequests>(request_unit, u), to = COPIER ? 0u : first_at_least<kRequests>(request_unit, u + 1u);
                for_each_const<to - from>([&](auto i_c) {
                    constexpr uint32_t q = from + decltype(i_c)::value;
                    if constexpr (q < kACopies)
                        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (__attribute__((address_space(3))) void*)(a_dst + q * 1024u), 16, (q & 1u) ? vo : ve,
                                                                 at_step(kt3) * kTwK * 2u + q * 16u * p.lda, 0, 0);
                    else if constexpr (q == kACopies) dma_w(w_tile(Target{}), kt3);
                    else dma_s(s_tile(Target{}), kt3);
                });
            }
            constexpr uint32_t from = first_at_least<Schedule::kCount>(op_slot, slot), to = first_at_least<Schedule::kCount>(op_slot, slot + 1u);
            for_each_const<to - from>([&](auto i_c) {
                constexpr TwOp o = Schedule::op(from + decltype(i_c)::value);
                using Column = std::integral_constant<uint32_t, o.column>;
                using Index = std::integral_constant<uint32_t, o.index>;
                if constexpr (o.pair) make_pair(nxt, conv, Column{}, Index{});
                else prepare(conv, code, sr, Column{}, Index{});
            });
            __builtin_amdgcn_sched_barrier(0);
        });
    };

    // ---- prologue: A tiles and codes of the first steps -> their stages; operands of step 0.  Without the copying wave the computing waves request all of
    // them, steps 0, 1 and 2 ahead of the first barrier.  With it they request steps 0 and 1 only, and it has requested the rest (see there).
    Ops ops0, ops1;
    if constexpr (kRing) {
#pragma unroll
        for (uint32_t t = 0; t < (uint32_t)NS; ++t) load_scales(ring[t], group_offset(clamp(t), kh));
    }
    auto fetch = [&](auto stage_c) {
        constexpr uint32_t St = decltype(stage_c)::value;
        if constexpr (St < kDepth) {
            dma_w(w_tile(stage_c), clamp(St));
            if constexpr (kScalesInLds) dma_s(s_tile(stage_c), clamp(St));
            dma_a(stage_c, clamp(St));
        }
    };
    // (The first two steps' copies have to land before anything else happens.  Without the copying wave those of the last stages are issued behind that
    // wait, a microsecond's work of the memory path; with it they are under way meanwhile.)
    fetch(C0{}), fetch(C1{});
    if constexpr (COPIER) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    } else {
        fetch(C2{});
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kRequests) : "memory");
    }
    barrier_no_fence();
    if constexpr (!COPIER) fetch(C3{}), fetch(C4{}), fetch(C5{}), fetch(C6{});
    {
        Codes code;
        Scales sr = ring[0];
        if constexpr (kScalesInLds) read_scales(sr, s_tile(C0{}));
        read_codes(code, w_tile(C0{}), 0);
        convert_all(ops0, code, sr);
    }
#pragma unroll
    for (uint32_t u = 0; u < kAhead; ++u) af[u] = *reinterpret_cast<const bf16x8_t*>(a_tile(C0{}) + a_rd + u * 2048u);

    uint32_t kt = 0;
    auto run = [&](auto stage_c) {
        constexpr uint32_t St = decltype(stage_c)::value;
        if constexpr (St < (uint32_t)NS) {
            if constexpr ((St & 1u) == 0u) step(stage_c, kt + St, ops0, ops1);
            else step(stage_c, kt + St, ops1, ops0);
        }
    };
    for (; kt + NS - 1u < ksteps; kt += NS) {
        run(C0{}), run(C1{}), run(C2{}), run(C3{}), run(C4{}), run(C5{}), run(C6{}), run(C7{});
    }
    auto run_rest = [&](auto stage_c) {
        if constexpr (decltype(stage_c)::value + 1u < (uint32_t)NS) {
            if (kt + decltype(stage_c)::value < ksteps) run(stage_c);
        }
    };
    run_rest(C0{}), run_rest(C1{}), run_rest(C2{}), run_rest(C3{}), run_rest(C4{}), run_rest(C5{}), run_rest(C6{});

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing asynchronous may still be writing LDS
    // ---- a scale beyond the conversion by halves: the wave's sums once more, in the same order, by the other conversion, everything straight
    // from memory (the other waves wait at the epilogue's first barrier)
    if (kLimited && __builtin_expect(beyond_halves(most), 0)) {
        tw_settle(acc);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[mt][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (uint32_t t = 0; t < ksteps; ++t) {
            const uint32_t at = at_step(t), row0 = at * kTwK + 32u * kh + 8u * kq;  // the lane's 8 rows of B
            Scales sr;
            load_scales(sr, GROUPED ? group_offset(t, kh) : 0u);
            bf16x8_t wf[2];
#pragma unroll
            for (uint32_t j = 0; j < 2; ++j) {
                uint32_t c[2] = {0u, 0u};
                if constexpr (PACKED) {
                    const uint32_t off = (2u * wc + j) * slab_bytes + (at >> w_shift) * w_step + lane * 16u + (BITS == 8 ? 8u * kh : 8u * (at & 1u) + 4u * kh);
                    c[0] = __builtin_amdgcn_raw_buffer_load_b32(rsrc_b, off, 0, 0);
                    if constexpr (BITS == 8) c[1] = __builtin_amdgcn_raw_buffer_load_b32(rsrc_b, off + 4u, 0, 0);
                } else {
                    const uint32_t col = wcol + 16u * j;
#pragma unroll
                    for (uint32_t r = 0; r < 8; ++r) {
                        const uint32_t byte = __builtin_amdgcn_raw_buffer_load_b8(rsrc_b, (row0 + r) * p.ldb_bytes + (BITS == 8 ? col : col / 2u), 0, 0);
                        if constexpr (BITS == 8) c[r >> 2] |= byte << (8u * (r & 3u));
                        else c[0] |= (byte >> (4u * (col & 1u)) & 15u) << (4u * r);
                    }
                }
                const float s = bf16_bits_to_f32(sr.s[j]);
                wf[j] = __builtin_bit_cast(bf16x8_t, BITS == 8 ? weights8(c[0], c[1], s) : weights4(c[0], 16.0f * s));
            }
            const bool past_k = at + 1u == ksteps_all && 4u * kh + kq >= last_chunks;
#pragma unroll
            for (uint32_t mt = 0; mt < (uint32_t)MT; ++mt) {
                const uint32_t off = past_k ? a_extent : ((16u * mt + c16) * p.lda + row0) * 2u;
                const bf16x8_t a = __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, off, 0, 0));
                // (the compiler's own instruction: its operands are written just before, which tw_mfma is not made for)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[mt][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, wf[j], acc[mt][j], 0, 0, 0);
            }
        }
    }

    // ---- epilogue: fp32 sums -> LDS in [m][n] order (a quarter of a stage's rows in each array), then finish row-wise
    tw_settle(acc);                                       // the last matrix instructions have written their sums
    __syncthreads();                                   // ... and every wave is done reading the stages
    constexpr uint32_t kArrayRows = kStageRows / 4u;
    auto c_row = [&](uint32_t row) -> float* {  // tile row `row`
        const uint32_t q = row / kArrayRows;
        return reinterpret_cast<float*>(q == 0 ? a_tile(C0{}) : q == 1 ? a_tile(C1{}) : q == 2 ? a_tile(C2{}) : a_tile(C3{})) + (row - q * kArrayRows) * kTw;
    };
    // Columns are turned by the row, 16 at a time: the four kq of a wave write rows 4 apart, a multiple of the banks' width.
    auto c_at = [&](uint32_t row, uint32_t col) -> float* { return c_row(row) + (col ^ (((row >> 2) & 3u) << 4)); };
    // The two waves of a column group add their sums (first blocks of 32 k + second blocks, whatever the timing), each for half of
    // the row blocks: it stages the other half's for its partner, then adds the partner's to its own and leaves the total.
    constexpr uint32_t kLower = (MT + 1) / 2;  // row blocks that the wave of the first blocks finishes
    auto stage_block = [&](uint32_t mt, bool add) {
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) {
#pragma unroll
            for (uint32_t j = 0; j < 2; ++j) {
                float* at = c_at(16u * mt + 4u * kq + r, wcol + 16u * j);
                *at = add ? acc[mt][j][r] + *at : acc[mt][j][r];
            }
        }
    };
    if (kh == 1u) {
#pragma unroll
        for (uint32_t mt = 0; mt < kLower; ++mt) stage_block(mt, false);
    } else {
#pragma unroll
        for (uint32_t mt = kLower; mt < (uint32_t)MT; ++mt) stage_block(mt, false);
    }
    __syncthreads();
    if (kh == 0u) {
#pragma unroll
        for (uint32_t mt = 0; mt < kLower; ++mt) stage_block(mt, true);
    } else {
#pragma unroll
        for (uint32_t mt = kLower; mt < (uint32_t)MT; ++mt) stage_block(mt, true);
    }
    __syncthreads();
    const bool gated = p.activation == kActSiluGate;
    const uint32_t ch = tid & 15u;  // 8 columns: 8 ch .. 8 ch + 7 of the tile
    const uint32_t gn = n0 + 8u * ch;
    float bias[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) bias[i] = 0.f;
    if (p.bias != nullptr && gn < p.n) {
        const uint4 raw = *reinterpret_cast<const uint4*>(p.bias + gn);
        const uint32_t d[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            bias[2 * i] = bf16_bits_to_f32(d[i] & 0xffffu);
            bias[2 * i + 1] = bf16_bits_to_f32(d[i] >> 16);
        }
    }
    const bool plain = p.bias == nullptr && p.residual == nullptr && !gated;  // the bare sums keep a -0 as it is
    // the thread's 8 sums of tile row `row`, as staged
    auto staged = [&](uint32_t row, float (&v)[8]) {
        const float* src = c_at(row, 8u * ch);
        const float4 lo = *reinterpret_cast<const float4*>(src), hi = *reinterpret_cast<const float4*>(src + 4);
        v[0] = lo.x, v[1] = lo.y, v[2] = lo.z, v[3] = lo.w, v[4] = hi.x, v[5] = hi.y, v[6] = hi.z, v[7] = hi.w;
    };
    // bias, gate, residual, rounding and the store of 8 finished sums of global row gm
    auto finish = [&](uint32_t gm, float (&v)[8], const uint4& r) {
        if (!plain) {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] += bias[i];
        }
        if (gated) {
            float o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = silu_gate(v[2 * i], v[2 * i + 1]);
            if (p.residual != nullptr) {
                o[0] += bf16_bits_to_f32(r.x & 0xffffu);
                o[1] += bf16_bits_to_f32(r.x >> 16);
                o[2] += bf16_bits_to_f32(r.y & 0xffffu);
                o[3] += bf16_bits_to_f32(r.y >> 16);
            }
            *reinterpret_cast<uint2*>(p.c + (size_t)gm * p.ldc + gn / 2u) = make_uint2(pack_bf16_rne(o[0], o[1]), pack_bf16_rne(o[2], o[3]));
        } else {
            if (p.residual != nullptr) {
                const uint32_t d[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    v[2 * i] += bf16_bits_to_f32(d[i] & 0xffffu);
                    v[2 * i + 1] += bf16_bits_to_f32(d[i] >> 16);
                }
            }
            *reinterpret_cast<uint4*>(p.c + (size_t)gm * p.ldc + gn) =
                make_uint4(pack_bf16_rne(v[0], v[1]), pack_bf16_rne(v[2], v[3]), pack_bf16_rne(v[4], v[5]), pack_bf16_rne(v[6], v[7]));
        }
    };
    // The residual of all of a thread's rows is requested at once, and before the other splits' sums: row by row, each behind the store of the
    // row before, the rows' trips to memory stood one behind the other at the end of the tile (us, with a residual: 400 x 2560 x 2560 8-bit
    // g64 19.7 -> 18.6, 256 x 4096 x 4096 25.9 -> 24.9).
    constexpr uint32_t kPasses = (MT + 1u) / 2u;  // rows tid / 16, + 32, ...
    uint4 residual[kPasses];                      // (nobody looks at what is not there)
    auto request_residual = [&]() {
        if (p.residual == nullptr || gn >= p.n) return;
#pragma unroll
        for (uint32_t pass = 0; pass < kPasses; ++pass) {
            const uint32_t row = 32u * pass + (tid >> 4);
            if (row < rows_valid) residual[pass] = request_residual8(p, m0 + row, gn, gated);
        }
    };
    auto finish_tile = [&]() {
#pragma unroll
        for (uint32_t pass = 0; pass < kPasses; ++pass) {
            const uint32_t row = 32u * pass + (tid >> 4);
            if (row >= rows_valid || gn >= p.n) continue;
            float v[8];
            staged(row, v);
            finish(m0 + row, v, residual[pass]);
        }
    };
    if (p.splits == 1u) {
        request_residual();
        finish_tile();
        return;
    }
    // ---- split-K: the protocol of the decode kernels.  The workspace holds one fp32 word per (split but the last, row,
    // column), kEmptyWord at rest.  Producers write their sums with device-scope stores and are done; the workgroup of the
    // last split (dispatched after them: blockIdx.y is the slow index) fetches them, again while any word is still empty,
    // adds them in split order with its own sums last, finishes the outputs and leaves the words empty.  Only it waits, and
    // only on workgroups that wait for nothing; the wait is bounded all the same.
    // Who moves what: thread t has the four columns 4 (t % 32) .. + 3 of tile rows t / 32 + kHStride i, i = 0 .. kHeld - 1, so that one
    // instruction of a wave covers two whole rows of the tile (512 contiguous bytes each): whole cache lines go out and come
    // in.  What the hand-over costs all the same is the reducing workgroup's fetch: 64 KiB per split through one CU, which
    // draws some 15-20 GB/s from beyond its L2 (3-5 us per split; measured with the fetch, the producers' stores and the
    // emptying switched off in turn), plus about 6 us for the producers' stores to arrive.
    const __amdgpu_buffer_rsrc_t ws = __builtin_amdgcn_make_buffer_rsrc(p.partials, 0, (int)p.partial_bytes, kBufferFlags);
    const uint32_t split_bytes = p.m * p.n * 4u;
    constexpr uint32_t kHStride = 16u;
    constexpr uint32_t kHeld = MT < 8 ? MT : 8;  // rows of a thread that are fetched together (a tile of more goes in two parts)
    const uint32_t hrow = tid >> 5, hcol = 4u * (tid & 31u);
    const uint32_t mine = (n0 + hcol < p.n && hrow < rows_valid) ? (rows_valid - hrow + kHStride - 1u) / kHStride : 0u;  // the thread's rows
    auto word_off = [&](uint32_t i) { return ((m0 + hrow + kHStride * i) * p.n + n0 + hcol) * 4u; };
    auto held = [&](uint32_t i) -> float4* { return reinterpret_cast<float4*>(c_at(hrow + kHStride * i, hcol)); };
    if (ks != p.splits - 1u || p.finish_launch) {
        if (p.debug_flags & kDebugWithholdPartials) return;  // test hook: lets the reducer's wait run out
#pragma unroll
        for (uint32_t i = 0; i < (uint32_t)MT; ++i) {
            if (i >= mine) continue;
            const float4 v = *held(i);
            const u32x4_t w4 = {__float_as_uint(v.x), __float_as_uint(v.y), __float_as_uint(v.z), __float_as_uint(v.w)};
            __builtin_amdgcn_raw_buffer_store_b128(w4, ws, (int)word_off(i), (int)(ks * split_bytes), kAuxDeviceScope);
        }
        return;
    }
    // First wait, at the price of one word per thread and split, until the producers' last stores show: a fetch of whole
    // tiles that comes too early moves 64 KiB per split of nothing through this CU.  (What a thread stored last is not
    // bound to arrive last: the fetch below checks every word on its own.)
    uint32_t fetch_limit = p.split_wait_limit;
    request_residual();
    if (mine != 0u) {
        bool there = false;
        for (uint32_t tries = 0; !there && tries < p.split_wait_limit; ++tries) {
            if (tries) __builtin_amdgcn_s_sleep(2);
            asm volatile("" ::: "memory");
            there = true;
            for (uint32_t sp = 0; sp + 1u < p.splits; ++sp) {
                const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(ws, (int)word_off(mine - 1u), (int)(sp * split_bytes), kAuxDeviceScope);
                if (v[3] == kEmptyWord) there = false;
            }
        }
        if (!there) fetch_limit = 1u;  // the wait has run out: one fetch of what there is, no second wait of that length
    }
    for (uint32_t i0 = 0; i0 < (uint32_t)MT; i0 += kHeld) {  // rows i0 .. i0 + kHeld - 1 of the thread's
        const uint32_t here = mine > i0 ? (mine - i0 < kHeld ? mine - i0 : kHeld) : 0u;
        float4 total[kHeld];
#pragma unroll
        for (uint32_t i = 0; i < kHeld; ++i) total[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        for (uint32_t sp = 0; sp + 1u < p.splits; sp += 2u) {
            // two splits' words of all these rows are fetched together (more bytes in flight per CU, fewer round trips),
            // and fetched again together while any is empty
            const bool pair = sp + 2u < p.splits;  // the same for every thread
            u32x4_t w[2][kHeld];
            // bit 16 j + i: words (j, i) are wanted and have not been seen complete yet; only those are fetched again
            uint32_t missing = 0u;
#pragma unroll
            for (uint32_t i = 0; i < kHeld; ++i)
                if (i < here) missing |= (1u << i) | (pair ? 1u << (16u + i) : 0u);
            for (uint32_t tries = 0; missing != 0u && tries < fetch_limit; ++tries) {
                if (tries) __builtin_amdgcn_s_sleep(2);
                asm volatile("" ::: "memory");  // other workgroups write these words: every attempt really loads
#pragma unroll
                for (uint32_t j = 0; j < 2; ++j)
#pragma unroll
                    for (uint32_t i = 0; i < kHeld; ++i)
                        if (missing & (1u << (16u * j + i)))
                            w[j][i] = __builtin_amdgcn_raw_buffer_load_b128(ws, (int)word_off(i0 + i), (int)((sp + j) * split_bytes), kAuxDeviceScope);
#pragma unroll
                for (uint32_t j = 0; j < 2; ++j)
#pragma unroll
                    for (uint32_t i = 0; i < kHeld; ++i)
                        if ((missing & (1u << (16u * j + i))) && w[j][i][0] != kEmptyWord && w[j][i][1] != kEmptyWord && w[j][i][2] != kEmptyWord &&
                            w[j][i][3] != kEmptyWord)
                            missing &= ~(1u << (16u * j + i));
            }
            // a word that never arrived is still the empty pattern, a NaN, and turns its sum into one; the workspace's header
            // remembers that it happened
            if (missing != 0u) __hip_atomic_store(p.ws_header, kWorkspaceGaveUp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (uint32_t j = 0; j < 2; ++j)  // in split order
#pragma unroll
                for (uint32_t i = 0; i < kHeld; ++i) {
                    if (i >= here || (j == 1u && !pair)) continue;
                    total[i].x += __uint_as_float(w[j][i][0]);
                    total[i].y += __uint_as_float(w[j][i][1]);
                    total[i].z += __uint_as_float(w[j][i][2]);
                    total[i].w += __uint_as_float(w[j][i][3]);
                }
        }
        // the other splits' sums plus this workgroup's own, back where the finishing pass takes them from
#pragma unroll
        for (uint32_t i = 0; i < kHeld; ++i) {
            if (i >= here) continue;
            float4* own = held(i0 + i);
            const float4 o = *own;
            *own = make_float4(total[i].x + o.x, total[i].y + o.y, total[i].z + o.z, total[i].w + o.w);
        }
    }
    __syncthreads();
    finish_tile();
    // the words this workgroup consumed are empty again for the next launch (last: nothing waits for these stores)
    const u32x4_t empty4 = {kEmptyWord, kEmptyWord, kEmptyWord, kEmptyWord};
    for (uint32_t sp = 0; sp + 1u < p.splits; ++sp) {
#pragma unroll
        for (uint32_t i = 0; i < (uint32_t)MT; ++i)
            if (i < mine) __builtin_amdgcn_raw_buffer_store_b128(empty4, ws, (int)word_off(i), (int)(sp * split_bytes), kAuxDeviceScope);
    }
}

// Which tiles: 16 MT rows by 128 columns (the order of bfaintb_prefill128_kernel: the ids an XCD receives cover consecutive logical
// ids, which walk groups of 8 tile-rows column by column).
template <int BITS, bool GROUPED, bool PACKED, int MT, int NS, bool COPIER>
__global__ void __launch_bounds__(COPIER ? 576 : 512) __attribute__((amdgpu_waves_per_eu(COPIER ? 3 : 2, COPIER ? 3 : 2)))
bfaintb_prefill128_wreg_kernel(const u32x4_t addresses, const u32x4_t sizes, const u32x4_t strides, const u32x2_t in_splits, const GemmParams rest)
{
    GemmParams p = with_words(rest, addresses, sizes, strides);
    p.splits = in_splits[0], p.finish_launch = in_splits[1];
    constexpr bool kScales = GROUPED && MT <= 12;  // (a larger tile leaves no room in LDS)
    const uint32_t tiles_m = (p.m + 16u * MT - 1u) / (16u * MT), tiles_n = (p.n + kTw - 1u) / kTw;
    const uint32_t wgs = tiles_m * tiles_n;
    // (with a second launch no workgroup waits for another, so tiles x splits are dealt out as one run: 42 tiles x 6 splits
    // dealt split by split are 36 workgroups on each of seven XCDs of 32 CUs and none on the eighth; 139 x 1072
    // x 15488, 18 tiles x 14 splits: 32.0 us so, 19.8 as one run; 82 x 5296 x 10240 4-bit, 42 x 6: 37.4 and 23.9)
    const uint32_t items = p.finish_launch ? wgs * p.splits : wgs;
    const uint32_t per_xcd = (items + 7u) / 8u;
    uint32_t logical = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
    if (logical >= items) return;
    uint32_t ks = blockIdx.y;
    if (p.finish_launch) {
        ks = logical / wgs;
        logical -= ks * wgs;
    }
    uint32_t tm = 0u, tn = logical;
    if (tiles_m > 1u) {  // (one row of tiles: no divisions ahead of the first copies)
        const uint32_t group = logical / (8u * tiles_n);
        const uint32_t first_m = group * 8u;
        const uint32_t group_rows = tiles_m - first_m < 8u ? tiles_m - first_m : 8u;
        const uint32_t in_group = logical - group * 8u * tiles_n;
        tm = first_m + in_group % group_rows;
        tn = in_group / group_rows;
    }
    tw_tile<BITS, GROUPED, PACKED, kScales, MT, NS, COPIER>(p, tm * 16u * MT, tn * kTw, ks);
}

// The second launch of a product whose k is split many ways (p.finish_launch): adds the splits' sums of four columns of a row in
// split order, finishes the outputs and leaves the words empty, as every launch that uses the workspace expects them.  A
// word that is still empty was never produced: its sum stays the NaN it is and the header remembers it.
//
// Bound by the latency of one fetch past the L2s and by splits x m x n words read and written.  Within the one launch, the
// workgroup of a tile's last split draws all of it through its CU, two splits per round trip (15 - 20 GB/s); a launch of its
// own spreads it over the machine: 8-bit, 64 x 4096 x 11008, k split 8 ways: 19.7 us (4 ways in one launch: 29.0), 96 rows,
// 7 ways: 24.8 (32.9).  Device-scope accesses on both sides, as in the one launch: 64 x 4096 x 4096 14.1 us; with ordinary
// ones here 16.2 (every emptied word is still in an L2 when the kernel ends), with ordinary stores by the producers 16.9.
constexpr uint32_t kFinishBatch = 8;  // splits whose words a thread fetches together
__global__ void __launch_bounds__(256) bfaintb_split_finish_kernel(const GemmParams p)
{
    const uint32_t quads = p.n / 4u;
    const uint32_t id = blockIdx.x * 256u + threadIdx.x;
    if (id >= p.m * quads) return;
    const uint32_t row = id / quads, col = 4u * (id - row * quads);
    // (the sums of all splits fit 16 MiB: 32-bit offsets)
    const __amdgpu_buffer_rsrc_t ws = __builtin_amdgcn_make_buffer_rsrc(p.partials, 0, (int)p.partial_bytes, kBufferFlags);
    const uint32_t off = (row * p.n + col) * 4u, split_bytes = p.m * p.n * 4u;
    const u32x4_t empty4 = {kEmptyWord, kEmptyWord, kEmptyWord, kEmptyWord};
    float4 total = make_float4(0.f, 0.f, 0.f, 0.f);
    bool complete = true;
    for (uint32_t sp0 = 0; sp0 < p.splits; sp0 += kFinishBatch) {
        u32x4_t w[kFinishBatch];
#pragma unroll
        for (uint32_t j = 0; j < kFinishBatch; ++j)  // (the bound is the same for every thread)
            if (sp0 + j < p.splits) w[j] = __builtin_amdgcn_raw_buffer_load_b128(ws, (int)off, (int)((sp0 + j) * split_bytes), kAuxDeviceScope);
#pragma unroll
        for (uint32_t j = 0; j < kFinishBatch; ++j) {
            if (sp0 + j >= p.splits) continue;
            __builtin_amdgcn_raw_buffer_store_b128(empty4, ws, (int)off, (int)((sp0 + j) * split_bytes), kAuxDeviceScope);
            complete = complete && w[j][0] != kEmptyWord && w[j][1] != kEmptyWord && w[j][2] != kEmptyWord && w[j][3] != kEmptyWord;
            total.x += __uint_as_float(w[j][0]);
            total.y += __uint_as_float(w[j][1]);
            total.z += __uint_as_float(w[j][2]);
            total.w += __uint_as_float(w[j][3]);
        }
    }
    if (!complete) __hip_atomic_store(p.ws_header, kWorkspaceGaveUp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    finish_row4(p, total, row, col);
}

template <int BITS, bool GROUPED, bool PACKED, int MT, int NS, bool COPIER = false>
static hipError_t launch_prefill128_wreg_t(const GemmParams& p, hipStream_t stream)
{
    const uint32_t tiles = ((p.m + 16u * MT - 1u) / (16u * MT)) * ((p.n + kTw - 1u) / kTw);
    // a whole number of workgroups per XCD; ids past the last tile exit at once
    const uint32_t grid = (p.finish_launch ? tiles * p.splits + 7u : tiles + 7u) / 8u * 8u;
    auto kernel = bfaintb_prefill128_wreg_kernel<BITS, GROUPED, PACKED, MT, NS, COPIER>;
    const hipError_t e = launch_kernel(kernel, dim3(grid, p.finish_launch ? 1u : p.splits, 1), dim3(COPIER ? 576 : 512, 1, 1), 0, stream, words_of_addresses(p),
                                       words_of_sizes(p), words_of_strides(p), u32x2_t{p.splits, p.finish_launch}, p);
    if (e != hipSuccess || !p.finish_launch) return e;
    return launch_kernel(bfaintb_split_finish_kernel, dim3((p.m * (p.n / 4u) + 255u) / 256u, 1, 1), dim3(256, 1, 1), 0, stream, p);
}

// Whether a launch has the copying wave (p: the tile's blocks, the rows, the split and its share of k, the group size).  Always with two
// blocks (see the head of the file), never with more than eight.  Otherwise, and with the fewer stages that its wait counts reach:
// Over packed weights with grouped scales or 4-bit codes (us, without / with, both with the start as it is now: 128 x 20480 x 4096 4-bit g128 33.9 / 29.0,
// 64 rows 24.4 / 22.4; 8-bit g64 35.5 / 33.3 and 26.2 / 24.8; 4-bit, one scale per column, 29.6 / 27.6 and 21.6 / 20.0; not 8-bit, one scale per column:
// 31.5 / 32.2 and 24.5 / 23.6, nor codes in rows: 8-bit 39.1 / 38.6 and 31.1 / 30.3, 4-bit 37.9 / 38.0 and 29.3 / 29.4).
// Codes in rows with grouped scales: where several rows of tiles split k into shares of up to 64 steps (without / with: 785 x 1440 x 4480
// 8-bit 25.8 / 23.6, 4-bit 26.2 / 24.1; 400 x 2560 x 2560 19.4 / 17.9 and 19.4 / 18.3; 900 x 2048 x 8192 43.2 / 40.7 and 43.0 / 40.0; longer
// shares lose what the start gains, 384 x 4096 x 11008 52.9 / 54.7 and 51.4 / 54.7, and so do most unsplit ones, 640 x 4096 x 4096 8-bit 33.8 /
// 35.4, and one row of eight blocks, 128 x 11008 x 4096 8-bit 26.3 / 27.7).  The line was drawn before the wave had its own first copies; beyond it there
// is now something to gain with four and six blocks of 8-bit codes in rows (64 x 8192 x 8192 26.4 / 25.0, 96 x 4096 x 11008 23.2 / 22.0, 64 x 11008 x 4096 g128 19.9 /
// 18.9) and at 640 x 4096 x 4096 4-bit g128, 32.3 / 28.5.
bool prefill128_wreg_copier(const GemmParams& p, int bits, bool packed)
{
    const bool grouped = p.group_size != 0u;
    if (p.tile_blocks == 2u || p.tile_blocks > 8u) return p.tile_blocks == 2u;
    return packed ? grouped || bits == 4 : grouped && p.splits > 1u && p.m > 256u && p.k_per_wg <= 64u * kTwK;
}

template <int BITS, bool GROUPED, bool PACKED>
static hipError_t launch_prefill128_wreg_rows(const GemmParams& p, hipStream_t stream)
{
    constexpr bool kCopierOnly = PACKED && (GROUPED || BITS == 4), kCopierToo = !PACKED && GROUPED;
    if (prefill128_wreg_copier(p, BITS, PACKED)) {
        if constexpr (kCopierOnly || kCopierToo) {
            switch (p.tile_blocks) {
                case 4: return launch_prefill128_wreg_t<BITS, GROUPED, PACKED, 4, 6, true>(p, stream);
                case 6: return launch_prefill128_wreg_t<BITS, GROUPED, PACKED, 6, 4, true>(p, stream);
                case 8: return launch_prefill128_wreg_t<BITS, GROUPED, PACKED, 8, 4, true>(p, stream);
                default: break;
            }
        }
    } else if constexpr (!kCopierOnly) {
        switch (p.tile_blocks) {
            case 4: return launch_prefill128_wreg_t<BITS, GROUPED, PACKED, 4, 8>(p, stream);
            case 6: return launch_prefill128_wreg_t<BITS, GROUPED, PACKED, 6, 6>(p, stream);
            case 8: return launch_prefill128_wreg_t<BITS, GROUPED, PACKED, 8, 6>(p, stream);
            default: break;
        }
    }
    switch (p.tile_blocks) {
        case 2: return launch_prefill128_wreg_t<BITS, GROUPED, PACKED, 2, 8, true>(p, stream);  // (see the head of the file)
        case 10: return launch_prefill128_wreg_t<BITS, GROUPED, PACKED, 10, 4>(p, stream);
        case 12: return launch_prefill128_wreg_t<BITS, GROUPED, PACKED, 12, 4>(p, stream);
        case 16: return launch_prefill128_wreg_t<BITS, GROUPED, PACKED, 16, 4>(p, stream);
        default: return hipErrorInvalidValue;
    }
}

// Whether this kernel can serve a launch: this library's own arithmetic (either order of the weights).
bool prefill128_wreg_serves(const GemmParams& p) { return !p.reference_arith; }

template <bool PACKED>
static hipError_t launch_prefill128_wreg_order(const GemmParams& p, int bits, hipStream_t stream)
{
    const bool grouped = p.group_size != 0;
    if (bits == 8) return grouped ? launch_prefill128_wreg_rows<8, true, PACKED>(p, stream) : launch_prefill128_wreg_rows<8, false, PACKED>(p, stream);
    return grouped ? launch_prefill128_wreg_rows<4, true, PACKED>(p, stream) : launch_prefill128_wreg_rows<4, false, PACKED>(p, stream);
}

// packed: p.b is the buffer in the packed order (p.ldb_bytes is unused)
hipError_t launch_prefill128_wreg(const GemmParams& p, int bits, bool packed, hipStream_t stream)
{
    return packed ? launch_prefill128_wreg_order<true>(p, bits, stream) : launch_prefill128_wreg_order<false>(p, bits, stream);
}

}  // namespace bfaintb
