// C ABI of the library: argument validation, kernel-family choice, split-K sizing, launches.
// Stands where the reference driver packs its kernarg block and calls hipModuleLaunchKernel
// (/root/reference/bfAintBGemm/bfAintBGemm.cc:107-152); unlike GPU_CHECK_ERROR
// (gpu_utils.hpp:5-11, print and exit(0)) every failure is returned to the caller.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <mutex>

#include "bfaintb_device.hpp"
#include "../../include/bfaintb_gemm.h"

namespace bfaintb {
hipError_t launch_decode(const GemmParams& p, int bits, hipStream_t stream);
hipError_t launch_prefill(const GemmParams& p, int bits, hipStream_t stream, bool wreg);
hipError_t launch_dequant(uint16_t* w, const uint8_t* b, const uint16_t* scale, uint32_t n, uint32_t k, uint32_t ldb_bytes,
                          uint32_t ldw, int bits, uint32_t group_size, hipStream_t stream);
hipError_t launch_fill_u32(uint32_t* dst, uint32_t count, uint32_t value, hipStream_t stream);
hipError_t launch_probe_read(const void* src, size_t bytes, void* sink, hipStream_t stream);
hipError_t launch_pack_colmajor(uint8_t* dst, const uint8_t* src, uint32_t n, uint32_t k, uint32_t ldb_bytes, int bits, hipStream_t stream);
hipError_t launch_pack(uint8_t* dst, const uint8_t* src, uint32_t n, uint32_t k, uint32_t ldb_bytes, int bits, bool unpack,
                       hipStream_t stream);
hipError_t launch_quantize(uint8_t* b, uint16_t* scale, const void* w, int type, uint32_t n, uint32_t k, uint32_t ldw, uint32_t ldb_bytes,
                           int bits, uint32_t group_size, hipStream_t stream);
hipError_t launch_decode_packed(const GemmParams& p, int bits, hipStream_t stream);
hipError_t launch_prefill_packed(const GemmParams& p, int bits, hipStream_t stream, bool wreg);
hipError_t launch_prefill128(const GemmParams& p, int bits, bool packed, hipStream_t stream);
hipError_t launch_prefill128_wreg(const GemmParams& p, int bits, bool packed, hipStream_t stream);
bool prefill128_wreg_serves(const GemmParams& p);
bool prefill128_wreg_copier(const GemmParams& p, int bits, bool packed);
hipError_t launch_prefill256x128_wreg(const GemmParams& p, int bits, bool packed, hipStream_t stream);
hipError_t launch_decode_family_packed(const GemmParams& p, int bits, hipStream_t stream);
hipError_t decode_prepare_device();
}  // namespace bfaintb

// Split-K scratch of bfaintb_gemm_static: one array per GPU the library runs on, held until the process ends.  In host
// code this name is only a handle for hipGetSymbolAddress; device_state() resolves it once per device and everything
// else uses the resolved pointer.
#define BFAINTB_STATIC_SCRATCH_BYTES (16u << 20)
static __device__ __align__(256) unsigned char scratch[BFAINTB_STATIC_SCRATCH_BYTES];

namespace {

using bfaintb::GemmParams;
using bfaintb::kEmptyWord;

constexpr uint32_t kDecodeAutoMaxM = 32;       // AUTO always runs the decode family up to this m
constexpr uint32_t kDecodeFamilyAutoMaxM = 4096;  // ... and never beyond this one
constexpr uint32_t kDecodeMaxM = 32768;        // what the decode family accepts when forced
// Compute units the plans are made for: those of the device that is current when the first plan is made (256 where there
// is no device to ask: the part the estimates were fitted on), or what the tuning hook says.  One count per process:
// workspace sizes and launches must agree, whichever device a later call runs on (a plan for another count is still a
// correct launch, only not the fastest one).
std::atomic<uint32_t> g_plan_cus_override{0};
uint32_t machine_cus()
{
    static const uint32_t device_cus = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0)
            return (uint32_t)n;
        (void)hipGetLastError();
        return 256u;
    }();
    const uint32_t forced = g_plan_cus_override.load(std::memory_order_relaxed);
    return forced ? forced : device_cus;
}
// workgroups the decode launches aim at: 8-wave workgroups run one per CU; 4-wave ones a little under two per CU
uint32_t decode_target_wgs_narrow() { return machine_cus(); }
uint32_t decode_target_wgs() { return machine_cus() * 15u / 8u; }
constexpr uint32_t kMaxSplits = 64;

int check_format(uint32_t k, int bits, uint32_t group_size)
{
    if (bits != 8 && bits != 4) return BFAINTB_ERR_UNSUPPORTED;
    if (group_size != 0 && (group_size % 32u != 0 || k % group_size != 0)) return BFAINTB_ERR_UNSUPPORTED;
    return BFAINTB_OK;
}

// Row-major weights: n a multiple of 8 (of 16 for 4-bit codes: a lane reads 16 of them per row), k a multiple of 8 (one
// 16-byte chunk of activations).  The kernels run a partial last step for the rest of k (the reference kernel needs
// n % 64 == 0 and k % 64 == 0: bf16gemm_kernel_gfx90a.s:341-343, :402-408).
int check_shape(uint32_t m, uint32_t n, uint32_t k, int bits = 8)
{
    if (k == 0 || n % (bits == 4 ? 16u : 8u) != 0 || k % 8u != 0) return BFAINTB_ERR_BAD_SHAPE;
    if (m >= (1u << 31) || n >= (1u << 31) || k >= (1u << 31)) return BFAINTB_ERR_BAD_SHAPE;
    return BFAINTB_OK;
}

// tuning hook (bfaintb_debug_control): the only row-block size, in units of 16 rows, decode_plan_row_blocks may pick; 0 = free
std::atomic<uint32_t> g_force_row_block{0};

// Launch shape of the decode variant: columns and waves per workgroup, blocks of 16 rows of A per workgroup,
// rows of k per workgroup, workgroups along k.
struct DecodePlan {
    uint32_t cols, waves, mb, k_per_wg, splits;
    uint32_t unit_bits = 0;  // width of the codes where it is not the `bits` the plan is made with (4-bit codes planned as 8-bit ones)
};

// Rows of k per workgroup and the number of splits that results, for `splits` wanted.
static void set_splits(DecodePlan& pl, uint32_t k, int bits, uint32_t splits, bool packed = false)
{
    // rows one workgroup covers per pipeline step of its waves
    const uint32_t unit = 32u * (uint32_t)bfaintb::decode_blocks_per_step(pl.unit_bits ? (int)pl.unit_bits : bits, (int)pl.cols / 16, packed, (int)pl.mb) * pl.waves;
    if (splits > kMaxSplits) splits = kMaxSplits;
    if (splits < 1) splits = 1;
    uint32_t per = (k + splits - 1) / splits;
    per = (per + unit - 1) / unit * unit;
    pl.k_per_wg = per;
    pl.splits = (k + per - 1) / per;
}

// Rough time, in microseconds, of the decode family for more than 32 rows of A (fitted on a 256-CU part).
// Every block of 16*mb rows streams and dequantises all weights again: measured 16, 22 and 35 cycles per
// weight and lane for mb = 1, 2, 4 (the dequantisation plus mb matrix instructions per 8 weights, less well
// overlapped the fewer waves a SIMD holds); repeats of the stream mostly hit in cache; split-K partial sums
// are written, read and cleared, and cost two more trips to memory; with fewer than one wave per SIMD both the
// arithmetic and the stream slow down in proportion.  Fitted to measurements at N = 4096, 11008 and 28672.
struct FamilyEstimate {
    double core, partial;  // the stream or the arithmetic, whichever is longer; the split's hand-over
    double serial;         // what the ranking adds for the reducing workgroup's own fetches (not part of the time estimates)
};
static double decode_family_estimate_us(uint32_t m, uint32_t n, uint32_t k, int bits, const DecodePlan& pl, FamilyEstimate* parts = nullptr)
{
    const double weights = (double)n * k;
    const double row_blocks = (double)((m + 16u * pl.mb - 1u) / (16u * pl.mb));
    const double col_blocks = (double)((n + pl.cols - 1u) / pl.cols);
    const double waves = row_blocks * col_blocks * pl.splits * pl.waves;
    const double cus = (double)machine_cus();
    const double busy = waves >= 4.0 * cus ? 1.0 : waves / (4.0 * cus);
    // 8-bit codes, refitted to a scan over row-block size x split factor at m = 40 .. 512 on 4096 x 4096, 11008 x 4096,
    // 4096 x 11008 and 2048 x 8192 (the choice of row block then lands within 0.5 % of the best on all 27 points; the
    // constants before it picked 16-row blocks where 32-row blocks with twice the splits run 6-24 % faster): larger row
    // blocks cost a little less per weight than first fitted, every further row block re-streams half of B from beyond
    // the caches, and the stream slows with idle CUs, not with idle wave slots.
    const double cycles_per_weight = bits == 8 ? 10.0 + 5.0 * pl.mb : 10.0 + 6.25 * pl.mb;
    // workgroups beyond one per CU share a CU's arithmetic: the last, partly filled round costs a whole one
    // (measured at n = k = 4096, 64-row blocks: m = 512 -> 256 workgroups, 35 us; m = 640 -> 320 workgroups, 61 us)
    const double wgs = row_blocks * col_blocks * pl.splits;
    const double ragged = wgs > cus ? (double)(uint64_t)((wgs + cus - 1.0) / cus) * cus / wgs : 1.0;
    const double compute = row_blocks * weights * cycles_per_weight / (256.0 * cus) / 2000.0 / busy * ragged;  // 4 SIMDs x 64 lanes per CU at 2 GHz
    const double stream_busy = bits == 8 ? (wgs >= cus ? 1.0 : wgs / cus) : busy;
    const double stream = weights * bits / 8.0 * (1.0 + (bits == 8 ? 0.5 : 0.3) * (row_blocks - 1.0)) / 3.5e6 / stream_busy;
    const double partial = pl.splits > 1 ? 3.0 + 12.0 * (pl.splits - 1.0) * m * n / 1.5e6 : 0.0;
    // (for the ranking only: the reducing workgroup fetches the other splits' sums of its block one after the other through
    // its one CU — the larger the block and the more the splits, the longer.  48 x 2560 x 16384: 64-row blocks with k split
    // 12 ways 27.0 us, 32-row blocks split 6 ways, the same number of workgroups, 20.6)
    const double serial = pl.splits > 1 ? 0.0075 * (pl.splits - 1.0) * pl.mb * pl.mb * pl.mb : 0.0;
    if (parts != nullptr) *parts = FamilyEstimate{compute > stream ? compute : stream, partial, serial};
    return 5.0 + (compute > stream ? compute : stream) + partial + serial;
}

// The same estimate, corrected to what the family's own plan takes in absolute terms: the estimate above ranks the
// family's plans among themselves (row-block size x split factor) and is left as fitted for that; against the tiles
// its absolute value decides, and there it is 1.3 - 1.75 times the measured time wherever k is split (the hand-over
// term is several times too large for row blocks of up to 32 rows, about 1.5 times for 64-row blocks) and within 8 %
// without a split.  Corrections fitted on 62 shapes (m = 48 .. 1024 over 4096 x 4096, 11008 x 4096, 4096 x 11008,
// 8192 x 8192, 2048 x 8192, 28672 x 8192, both code widths: the pick is then the faster form on 58 of them, within 10 %
// on the other four); 4-bit codes: 0.76 of the whole estimate, which dates from before their conversion got cheaper.
static double decode_family_time_us(uint32_t m, uint32_t n, uint32_t k, int bits, const DecodePlan& pl)
{
    FamilyEstimate e;
    const double ranked = decode_family_estimate_us(m, n, k, bits, pl, &e) - e.serial;
    if (bits == 4) {
        // (one row block that is not full costs less, a full one a little more than the 0.76 says: 64-row blocks of the
        // 128-column form at m = 40 / 48 / 64 against the tiles, us: 11008 x 8192 32.4 / 36.3, 33.6 / 36.5, 36.5 / 36.8;
        // 32000 x 4096 31.1 / 32.6, 32.1 / 32.6, 34.9 / 33.1; 16384 x 8192 34.4 / 36.8, 37.0 / 37.0, 40.6 / 38.8)
        const double block_rows = 16.0 * pl.mb;
        if (m <= block_rows && pl.cols <= 128u) {
            // (and CUs left idle slow the stream less than in proportion, as over packed weights: 86 column blocks x 2 splits)
            const double wgs = (double)((n + pl.cols - 1u) / pl.cols) * pl.splits, cus = (double)machine_cus();
            // (not below 0.65 of a round: 144 and 160 column blocks, unsplit, take all the estimate says and more — 18432 x 6144,
            // m = 40 / 64: 44.6 / 52.8 us, where the tiles with k split three ways take 41.9 / 43.7; 20480 x 4096, m = 64: 39.0
            // against the tiles' 34.8)
            const double idle = wgs < cus && wgs * 20.0 >= cus * 13.0 ? pow(wgs / cus, 0.45) : 1.0;
            return 0.80 * (0.65 + 0.35 * m / block_rows) * (5.0 + e.core * idle + e.partial);
        }
        // (32-row blocks in more than a round and a half of workgroups take 0.82 - 0.86 of it: 48 / 64 x 128256 x 4096 161 / 163 us,
        // 48 / 64 x 50304 x 4096 79 / 81, where the tiles take 138 / 146 and 66 / 67)
        const double wgs = (double)((m + 16u * pl.mb - 1u) / (16u * pl.mb)) * (double)((n + pl.cols - 1u) / pl.cols) * pl.splits;
        if (pl.mb == 2u && wgs * 2.0 > 3.0 * (double)machine_cus()) return 0.84 * ranked;
        // (beyond 256 rows, unsplit: ten row blocks and more over few column blocks take all the estimate says and up to 1.4
        // times it — 320 x 2816 x 6144: 39.9 us, the tiles 29.0; 512 x 1280 x 5120: 35.9 / 26.7; 320 x 12032 x 6144: 101.7 / 93.6)
        // (... and their 8-wave workgroups count as a busy machine in the estimate from 128 of them on: CUs left without one
        // are charged here)
        if (m > 256u && pl.splits == 1u) {
            const double cus = (double)machine_cus();
            return 5.0 + e.core * (wgs < cus ? cus / wgs : 1.0);
        }
        return 0.76 * ranked;
    }
    // (64-row blocks: the hand-over at 0.9 of its term — at 0.65 the family ran up to 13 % over the tiles' time at 48 - 64 rows
    // against 8192 x 11008 and 8192 x 8192; 5 of 105 shapes scanned are then more than 2.5 % off, the worst 96 x 4096 x 11008
    // at 13 %.  Scaling a single block by its fill, which suits 4-bit codes, sends those same shapes back to the family.)
    if (pl.splits > 1u) return 0.87 * (5.0 + e.core + (pl.mb == 4u ? 0.9 : 0.2) * e.partial);
    return (pl.mb == 4u ? 1.05 : 0.93) * (5.0 + e.core);
}

// Tall tiles: at most 256 rows x 128 columns; the rows spread evenly over as many tiles as 256 rows each would take, in blocks of 16.
static uint32_t tall_tile_blocks(uint32_t m)
{
    const uint32_t rows_of_tiles = (m + 255u) / 256u, needed = (m + 16u * rows_of_tiles - 1u) / (16u * rows_of_tiles);
    return needed <= 10u ? 10u : needed <= 12u ? 12u : 16u;
}
// Up to a k of 1024 (2048 for tiles of 10 blocks) the form that adds an output's products in one chain of ascending k, as the large tiles do:
// a product of a short k has the bits of the large tiles, whichever of the two its size picks (bfaintb_prefill256x128_wreg_kernel).  That is
// the whole reason: beyond it the small tiles' kernel with 10 to 16 blocks of 16 rows, which adds two chains, runs, and below it it would
// mostly be the faster one as well.  us, one chain / the other, k = 512 / 1024 / 2048 / 4096: 16 blocks, 2048 x 4096 8-bit 17.3 / 17.0, 24.8 /
// 24.1, 40.2 / 35.5, 70.9 / 63.3; 512 x 11008 4-bit 17.2 / 15.1, 24.9 / 20.5, 40.7 / 31.5, 71.8 / 54.2; 10 blocks, 300 x 12288 8-bit 15.2 / 11.0, 22.0 /
// 15.8, 35.0 / 24.6, 61.9 / 41.4; the other way round where 8-bit rows lie a large power of two apart and k is 512 (384 x 16384 16.0 / 21.4).
static bool tall_tiles_in_one_chain(uint32_t m, uint32_t k) { return k <= (tall_tile_blocks(m) == 10u ? 2048u : 1024u); }

// The tiled variant runs small tiles, of 128 columns and at most 128 rows, while those fit one per CU: four times the workgroups of
// 256x256 tiles, each with a quarter of the work per K-step.  Measured against the tall and the large tiles (8-bit, k = 4096, us,
// small / tall / large): 256 x 4096: 33.7 / 48.2 / 58.5, 1024 x 4096: 41.1 / 50.6 / 60.0, 512 x 8192 (4-bit, k = 8192): 78.2 / 95.6 / 133; with more
// tiles the others win (1536 x 4096: 67.4 / 54.7 / 60.8, 512 x 11008: 67.2 / 54.5 / 60.7).
// (One gap: a few tall tiles more than CUs — 640 x 11008 makes 258, two rounds, 98.5 us — would go to 129 large tiles on half the machine,
// 85.7 us; the small tiles take it in two rounds, 430 of them, in 70.8 us.  So: also up to two rounds of small tiles where the tall
// ones do not fit one round and the large ones fill at most 60 % of the CUs.)
static bool prefill_small_tiles(uint32_t m, uint32_t n, uint32_t k, int bits)
{
    const uint64_t cus = machine_cus();
    const uint64_t small = (uint64_t)((m + 127u) / 128u) * ((n + 127u) / 128u);
    if (small <= cus) return true;
    // One row of tiles: 256-row tiles would spend half their matrix instructions or more on rows that do not exist, however
    // many rounds the small ones take (us, small / large, 8-bit and 4-bit codes: 64 x 128256 x 4096, 1002 small tiles, 126 / 187
    // and 119 / 203; 128 x 128256 x 4096 169 / 204 and 163 / 210; 96 x 50304 x 4096, 393 tiles, 66.5 / 86.5 and 65.1 / 102;
    // 128 x 36864 x 8192, 288 tiles, 135 / 158 and 133 / 193; from 129 rows on the large tiles win: 192 x 50304 x 4096 123 / 98)
    if (m <= 128u) return true;
    // 4-bit codes where the tall tiles would be those of one chain, whose kernel converts every weight in two waves: small ones while a
    // second round of them is about a third full.  Made when a long k ran so as well (k = 4096, us, small / one chain: 1152 x 4096, 288 tiles,
    // 67.2 / 71.0; 512 x 11008, 344, 69.7 / 72.0); at the k that is left of it the two are level to a tenth apart (k = 1024: 25.2 / 24.5 and 25.1 /
    // 24.9; k = 512: 18.4 / 16.7 and 18.5 / 17.1), and the rule goes with the tall tiles' (8-bit codes: 23.4 / 21.5 at 1152 x 4096 x 1024).
    if (bits == 4 && tall_tiles_in_one_chain(m, k) && small * 20u <= cus * 27u) return true;
    const uint64_t tall = (uint64_t)((m + 255u) / 256u) * ((n + 127u) / 128u);
    const uint64_t large = (uint64_t)((m + 255u) / 256u) * ((n + 255u) / 256u);
    // (0.6 of the CUs at most: 640 x 12032 x 3584, 141 large tiles, 76.5 us; 470 small ones 66.5)
    return small <= 2u * cus && tall > cus && large * 5u <= cus * 3u;
}

// Between the two: more small tiles than CUs, but at most one tile of 256 rows x 128 columns per CU.  The large tiles would
// occupy a quarter to a half of the CUs there; the tall ones run one per CU and share one conversion among 10 to 16 blocks of rows
// (us, tall / large, 8-bit, 64 steps: 1536 x 4096: 54.7 / 60.8; 512 x 11008: 54.5 / 60.7; 2048 x 4096: 63.4 / 72.3; 128 steps,
// 1024 x 8192: 117 / 133; 4-bit, 768 x 8192: 103 / 134).
static bool prefill_tall_tiles(uint32_t m, uint32_t n, uint32_t k, int bits)
{
    return !prefill_small_tiles(m, n, k, bits) && (uint64_t)((m + 255u) / 256u) * ((n + 127u) / 128u) <= machine_cus();
}

static bool is_prefill(int v)
{
    return v == BFAINTB_VARIANT_PREFILL || v == BFAINTB_VARIANT_PREFILL_256 || v == BFAINTB_VARIANT_PREFILL_128 ||
           v == BFAINTB_VARIANT_PREFILL_256_LDS || v == BFAINTB_VARIANT_PREFILL_128_LDS || v == BFAINTB_VARIANT_PREFILL_256X128;
}

// tile size of a tiled-variant launch: forced, or by shape
static bool use_small_tiles(int v, uint32_t m, uint32_t n, uint32_t k, int bits)
{
    return v == BFAINTB_VARIANT_PREFILL_128 || v == BFAINTB_VARIANT_PREFILL_128_LDS || (v == BFAINTB_VARIANT_PREFILL && prefill_small_tiles(m, n, k, bits));
}

// The small-tile kernel may split k: grid y walks the splits, each workgroup runs its share of
// the K-steps and the workgroup of the last split adds the others' sums (same workspace and protocol as the decode
// family).  Worth it while tiles x splits still fit one workgroup per CU.
struct TilePlan {
    uint32_t k_per_wg, splits;
    uint32_t blocks;  // of 16 rows of a tile
    uint32_t finish_launch;  // 1: every split's sums go to the workspace and a second launch adds them
    double us;
};
constexpr uint32_t kMaxTileSplits = 16;
constexpr uint32_t kFinishLaunchSplits = 6;  // from here on a second launch adds the sums (unless the split factor is the caller's)

static size_t split_workspace_bytes(uint32_t splits, uint32_t m, uint32_t n)
{
    if (splits <= 1) return 0;
    // the header, then one fp32 word per (split but the last, row, column), rounded up to 256 bytes
    return bfaintb::kWorkspaceHeaderBytes + ((((size_t)(splits - 1u) * m * n * sizeof(float)) + 255u) & ~(size_t)255u);
}

// (with a second launch the last split's sums lie there as well)
static size_t tile_workspace_bytes(const TilePlan& t, uint32_t m, uint32_t n) { return split_workspace_bytes(t.splits + t.finish_launch, m, n); }

// A K-step of a tile of 16 x blocks rows and 128 columns, in us, with `load` of the CUs holding a workgroup: what is issued beside the
// matrix instructions, the matrix instructions, and the clock that gives way to the board's power.  8-bit, us a step at 96 / 256
// workgroups, 4 / 6 / 8 / 10 / 12 / 16 blocks: 0.33 / 0.39 / 0.44 / 0.50 / 0.52 / 0.60 and 0.33 / 0.40 / 0.46 / 0.60 / 0.66 / 0.82; 4-bit and
// grouped scales within 7 %.  One row of tiles reads each code once, from memory, which costs some
// 0.05 on a full machine, at 6 TB/s at most (8-bit, 256 workgroups, 4 / 6 / 8 blocks: 0.34 / 0.45 / 0.55).
static double tile_step_us(uint32_t blocks, uint32_t m, int bits, double load)
{
    const double issue = 0.23 + 0.0255 * blocks + 0.00105 * blocks * blocks * load * load * load;
    if (m > 16u * blocks) return issue;
    const double stream = load * machine_cus() * 1024.0 * bits / 6.0e6;
    return issue + 0.05 * load > stream ? issue + 0.05 * load : stream;
}
// The beginning and the end of a launch of such tiles (8 / 16 blocks: 6 / 9 us in a run of launches).
static double tile_ends_us(uint32_t blocks) { return 3.3 + 0.34 * blocks; }

// second_launch: whether the plan may be one whose sums a second launch adds.  Here and below, false is for the caller who
// brings less scratch than such a plan needs (all splits' sums) and gets what the library does without it.
static TilePlan tile128_plan(uint32_t m, uint32_t n, uint32_t k, int bits, uint32_t forced_splits, bool second_launch = true)
{
    const uint32_t ksteps = (k + 63u) / 64u;
    // blocks of 16 rows of a tile: the rows, spread evenly over as many tiles as 128 rows each would take
    const uint32_t rows_of_tiles = (m + 127u) / 128u, needed = (m + 16u * rows_of_tiles - 1u) / (16u * rows_of_tiles);
    const uint32_t blocks = needed <= 2u ? 2u : needed <= 4u ? 4u : needed <= 6u ? 6u : 8u;
    const double tiles = (double)rows_of_tiles * (double)((n + 127u) / 128u);
    const double cus = (double)machine_cus();
    const double fill = (double)m / (double)((m + 127u) / 128u * 128u);  // the share of the tiles' rows that exist
    auto shape = [&](uint32_t want) {
        TilePlan t;
        t.finish_launch = 0u;
        t.blocks = blocks;
        if (want > kMaxTileSplits) want = kMaxTileSplits;
        if (want < 1u) want = 1u;
        const uint32_t per = (ksteps + want - 1u) / want;
        t.k_per_wg = per * 64u;
        t.splits = (ksteps + per - 1u) / per;
        // the hand-over: the producers' device-scope stores have to arrive, then the reducing workgroup fetches the rows of a tile that
        // exist, per split, through its one CU, slower the more CUs do so at once (fitted, with the steps' factor, on 60 shapes of 33 ...
        // 577 rows, both code widths and weight orders, 2 to 4 splits: 7 % rms)
        const double hand_over = t.splits > 1u ? 1.8 + (t.splits - 1.0) * (2.5 * fill + 0.024 * tiles) : 0.0;
        const double wgs = tiles * t.splits;
        const double whole = (double)(uint64_t)(wgs / cus), rest = wgs - whole * cus;
        if (!second_launch) {
            // (A caller who brings the scratch that a call needed before there were second launches, or none, is served with that much.  So these
            // plans, and the choice between them and the family, go by the steps' times of then, not by what the kernels take now: the
            // estimate decides how much scratch such a caller has to bring, and by today's steps 206 of 8000 random calls without any, 33 ...
            // 1500 rows, would be refused that are served.  What it costs is a slower plan for a caller with too little scratch.)
            auto step_us = [&](double load) { return ((bits == 4 ? 0.41 : 0.40) + 0.15 * load * load * load) * (0.8 + 0.2 * fill); };
            t.us = 4.0 + (wgs > 2.0 * cus ? 1.12 : 1.0) * per * (whole * step_us(1.0) + (rest > 0.0 ? step_us(rest / cus) : 0.0)) +
                   (t.splits > 1u ? 3.0 + (t.splits - 1.0) * (0.6 + 1.6 * fill + 0.008 * tiles) : 0.0);
            if (t.splits > 2u) t.us *= 1.07;
            return t;
        }
        const double steps_us = whole * tile_step_us(blocks, m, bits, 1.0) + (rest > 0.0 ? tile_step_us(blocks, m, bits, rest / cus) : 0.0);
        // (further rounds of tiles begin behind the ones before them, each at four fifths of a launch's beginning and end)
        t.us = tile_ends_us(blocks) * (0.2 + 0.8 * (whole + (rest > 0.0 ? 1.0 : 0.0))) + 0.94 * per * steps_us + hand_over;
        // (three splits and more: the hand-over scatters more than this says, and where the row-blocked family is about as
        // fast it is the safer pick — 192 x 4096 x 4096: 25.5 against 22.9 us, 128 x 4096 x 11008: 39.0 against 34.3)
        if (t.splits > 2u) t.us *= 1.07;
        return t;
    };
    if (forced_splits) return shape(forced_splits);
    // with the second launch: the two launches' beginnings and ends (a little more where a thread fetches twice, beyond eight splits), the
    // steps, and the words' way through memory (fitted on the same shapes, 6 to 16 splits, 102 times: 5 % rms)
    auto finish_us = [&](const TilePlan& t) {
        return 7.8 - 0.2 * blocks + (t.splits > 8u ? 0.7 : 0.0) + 1.1 * (t.k_per_wg / 64u) * tile_step_us(blocks, m, bits, tiles * t.splits / cus) +
               0.54e-6 * t.splits * (double)m * n * 4.0;
    };
    TilePlan best = shape(1);
    static const uint32_t kCandidates[] = {2, 3, 4, 6, 7, 8, 10, 12, 14, 16};
    for (uint32_t s : kCandidates) {
        if (tiles * s > cus) break;
        // (one launch deals a split's tiles out in eights: 85 tiles x 3 are 33 workgroups on seven of the XCDs of 32 CUs, 54 us at 515 x 2080 x
        // 8192, two splits 40)
        if ((!second_launch || s < kFinishLaunchSplits) && (double)(((uint32_t)tiles + 7u) / 8u * 8u) * s > cus) continue;
        TilePlan t = shape(s);
        if (t.splits != s) continue;  // k does not divide that way
        // from six splits on their sums are added by a second launch, if all of them fit the scratch of the entry point that
        // brings its own
        // (not for 4-bit codes beyond 256 rows: there the family's rule above keeps the shapes that would split so far)
        if (!second_launch && (s == 7u || s > 8u)) continue;  // (measured with the second launch only)
        if (second_launch && s >= kFinishLaunchSplits) {
            if (bits == 4 && m > 256u) break;
            t.finish_launch = 1u;
            if (tile_workspace_bytes(t, m, n) > BFAINTB_STATIC_SCRATCH_BYTES) break;
            t.us = finish_us(t);
        }
        // (at most 256 tiles' worth of sums in all, 14 MiB: within the 32-bit offsets of the kernel and within the scratch of
        // the entry point that brings its own)
        if (t.us < best.us) best = t;
    }
    // One row of tiles that leaves a third or more of the CUs idle (half to five eighths of a round) and a long k: three
    // splits, as the decode family does on such widths — the estimate has the two forms level, the machine does not (us,
    // unsplit / three splits, 8-bit and 4-bit codes: 48 x 18432 x 8192, 144 tiles, 51.9 / 47.3 and 51.8 / 45.2; 96 x 18432 x
    // 8192 63.8 / 59.0 and 58.6 / 53.9; 48 x 20480 x 8192, 160 tiles, 56.2 / 51.8 and 52.1 / 45.7).  The launch rounds a split's
    // workgroups up to a multiple of 8, and three splits must stay clear of two rounds: 170 tiles make 528 and lose (44.7 /
    // 65.5).  A shorter k gains little or loses (k = 6144: 40.5 / 40.3 and 40.3 / 37.6 at 48 rows, 49.5 / 49.4 at 96; k = 4096: 29.2 / 31.6).
    // (While the partial sums stay within the 14 MiB of the note above.)
    const double per_split = (double)(uint64_t)((tiles + 7.0) / 8.0) * 8.0;
    if (best.splits == 1u && m <= 128u && tiles * 2.0 > cus && per_split * 3.0 * 16.0 <= cus * 31.0 && k >= 8192u &&
        2ull * m * n * sizeof(float) <= (14ull << 20)) {
        TilePlan t = shape(3);
        t.us *= 0.88;  // (measured against what shape() says of them: 0.85 - 0.92)
        if (t.splits == 3u) best = t;
    }
    return best;
}

// Tiles of 256 columns and 16 x blocks rows, all in one launch: the rows spread evenly over the tiles, and as many rows of tiles as make the
// rounds of one tile per CU come out best (blocks 0: not such tiles).
struct WideTiles {
    uint32_t blocks, rows_of_tiles;
    double us;
};
// What they take, in us: fitted to 24000 timings of 7269 random shapes (33 ... 4096 rows, both code widths and weight orders, weights cold), 4.3 %
// rms, of the kernel's first form.  A K-step is 128 cycles of matrix instructions a block and some 770 (8-bit) or 840 (4-bit codes, mostly with group
// scales) beside them, at 2.39 GHz while few CUs hold few rows, and at what the board's power leaves otherwise: 0.83 of it with 14 blocks on every CU.
// Not fitted again: the kernel takes 330 (16 blocks) to 570 (8) and 540 to 720 beside them today, packed codes alike, and the fit's other terms hold part of
// the difference.  us, what this says / what a call takes: 384 x 22016 x 4096 8-bit 74.2 / 69.6, 577 x 13824 x 5120 packed 4-bit g128 86.1 / 83.5, packed
// 8-bit 83.6 / 78.6, 148 x 43680 x 4096 8-bit g128 64.8 / 70.1, 4096 x 4096 x 4096 8-bit 100.2 / 101.7.
static double wide_tiles_us(uint32_t blocks, double tiles, uint32_t k, int bits)
{
    const double cus = (double)machine_cus();
    auto step_us = [&](double load) {
        const double heat = blocks * load, slower = heat <= 7.0 ? 1.0 : heat <= 10.0 ? 1.0 + 0.040 * (heat - 7.0) : 1.12 + 0.012 * (heat - 10.0);
        return (128.0 * blocks + (bits == 8 ? 770.0 : 840.0) + (blocks < 14u ? 22.0 * (14u - blocks) * load * load : 0.0)) / 2390.0 * slower;
    };
    const double whole = (double)(uint64_t)(tiles / cus), rest = tiles - whole * cus;
    return 6.5 + 0.234 * blocks + 7.3 * (whole + (rest > 0.0 ? 1.0 : 0.0) - 1.0) + (double)((k + 63u) / 64u) * (whole * step_us(1.0) + (rest > 0.0 ? step_us(rest / cus) : 0.0));
}
static WideTiles wide_tiles_best(uint32_t m, uint32_t n, uint32_t k, int bits)
{
    WideTiles best{0u, 0u, 0.0};
    const double cols = (double)((n + 255u) / 256u);
    for (uint32_t blocks = 8; blocks <= 16u; blocks += 2u) {
        const uint32_t rows = (m + 16u * blocks - 1u) / (16u * blocks);
        const double us = wide_tiles_us(blocks, rows * cols, k, bits);
        if (best.blocks == 0u || us < best.us) best = WideTiles{blocks, rows, us};
    }
    return best;
}
// The 256x256 tiles whose last round, if it is thin, runs as half tiles in a launch of its own.  Fitted to the same timings, 4 % rms, while the halves were
// 256 x 128, and not again: over 130 random shapes with a thin last round (257 ... 4096 rows, both code widths and weight orders) it stands 3 % higher beside
// the estimate of the lower tiles than the times do, and the choice between them takes 0.2 % longer than the faster form on average, 4.8 % at worst; with the
// halves at wide_tiles_us(8, 2 thin) + 2 us it would be 0.15 and 4.8.
static double square_tiles_us(uint32_t m, uint32_t n, uint32_t k, int bits)
{
    const uint32_t tiles = ((m + 255u) / 256u) * ((n + 255u) / 256u), thin = bfaintb::thin_round_tiles(tiles, m, machine_cus());
    const double load = 2.0 * thin / (double)machine_cus();
    return (tiles != thin ? wide_tiles_us(16u, tiles - thin, k, bits) : 0.0) + (thin != 0u ? 12.4 + (double)((k + 63u) / 64u) * (0.81 + 0.135 * load * load * load) : 0.0);
}
// Whether a tiled launch of the library's own choice goes to them: where neither small nor tall tiles fit one round, unless the 256x256 tiles
// and their thin last round are estimated faster; and for 97 to 128 rows that make more small tiles than CUs.  Of 7269 random shapes the tall tiles, and
// the small ones within a round, lead on all but a few; where the 256x256 tiles ran, these are 1.15 times as fast (geometric mean of 1854; 1741 of
// them faster), where a product ran as two launches by rows 1.07 times.  By this rule, over 4484 other random shapes of 33 ... 4096 rows: 1.046 times
// as fast on the whole, 871 more than 10 % faster, 9 more than 5 % slower, worst 0.90.  (All of that with the kernel's first form.)  us, before there were
// such tiles / with the kernel of today: 148 x 43680 x 4096 8-bit g128 97.8 / 70.1; 418 x 17728 x 9728 packed 8-bit g128 193 / 155; 577 x 13824 x 5120
// packed 4-bit g128 95.6 / 83.5; 913 x 9296 x 3328 packed 8-bit 73.6 / 54.8; 1010 x 17776 x 1024 8-bit 57.2 / 48.8.
// (At least 96 of them: the estimates are for a machine's worth of tiles.)
static WideTiles wide_tiles_rule(uint32_t m, uint32_t n, uint32_t k, int bits)
{
    const WideTiles none{0u, 0u, 0.0};
    const uint64_t cus = machine_cus();
    if (prefill_small_tiles(m, n, k, bits)) {
        if ((uint64_t)((n + 127u) / 128u) <= cus || m > 128u || k < 1024u) return none;
        const WideTiles w = wide_tiles_best(m, n, k, bits);
        return w.us < 0.95 * tile128_plan(m, n, k, bits, 0).us ? w : none;
    }
    if (prefill_tall_tiles(m, n, k, bits)) return none;
    const WideTiles w = wide_tiles_best(m, n, k, bits);
    return w.rows_of_tiles * ((n + 255u) / 256u) >= 96u && w.us < square_tiles_us(m, n, k, bits) ? w : none;
}
// (a call asks up to five times, for its scratch, its choices and its launch: each thread keeps the last answers, one per slot of a hash of the question;
// host time of a known call, ns, without / with: 128 x 43680 x 4096 768 / 70, 913 x 9296 x 3328 packed 731 / 68, 2048 x 28672 x 8192 4-bit 557 / 206)
static WideTiles wide_tiles(uint32_t m, uint32_t n, uint32_t k, int bits)
{
    if (m <= 96u) return WideTiles{0u, 0u, 0.0};
    struct Answer {
        uint32_t m, n, k, bits, cus;
        WideTiles tiles;
    };
    static thread_local Answer answers[256] = {};
    const uint32_t cus = machine_cus();
    Answer& a = answers[((m * 2654435761u) ^ (n * 2246822519u) ^ (k * 3266489917u) ^ (uint32_t)bits) >> 24];
    if (a.m != m || a.n != n || a.k != k || a.bits != (uint32_t)bits || a.cus != cus) a = Answer{m, n, k, (uint32_t)bits, cus, wide_tiles_rule(m, n, k, bits)};
    return a.tiles;
}

// The same for a call that may name a split of k: one that does keeps the small tiles, which have it, wherever they would run without these.
static WideTiles wide_tiles(uint32_t m, uint32_t n, uint32_t k, int bits, uint32_t split_k)
{
    return split_k != 0u && prefill_small_tiles(m, n, k, bits) ? WideTiles{0u, 0u, 0.0} : wide_tiles(m, n, k, bits);
}

// Whether they run by the library's own choice, and nobody asks the row-blocked family.  From a k of 512 on its estimate is the higher one on every one
// of 60000 random shapes; below, the estimate leaves out what a workgroup's start costs, some 6 us a round of them, and the family takes 1.8 to 3.9
// times as long (us, family / tiles: 1952 x 28640 x 128 8-bit g32 168.6 / 49.4; 3630 x 13840 x 128 packed 4-bit 154.4 / 48.6; 350 x 33264 x 128 packed
// 8-bit 39.9 / 16.8; 529 x 25456 x 256 packed 8-bit 50.7 / 20.7).  Nor do the tiles need the device's set-up, so such a call may be a first one under capture.
static bool wide_tiles_run(uint32_t m, uint32_t n, uint32_t k, int bits, bool second_launch) { return second_launch && wide_tiles(m, n, k, bits).blocks != 0u; }

// What the other tiles take.
static double prefill_estimate_us(uint32_t m, uint32_t n, uint32_t k, int bits, bool second_launch = true)
{
    if (prefill_small_tiles(m, n, k, bits)) return tile128_plan(m, n, k, bits, 0, second_launch).us;
    const double cus = (double)machine_cus();
    if (prefill_tall_tiles(m, n, k, bits)) {
        const double load = (double)((m + 255u) / 256u) * (double)((n + 127u) / 128u) / cus;
        const uint32_t blocks = tall_tile_blocks(m);
        if (!tall_tiles_in_one_chain(m, k)) return tile_ends_us(blocks) + (k / 64.0) * tile_step_us(blocks, m, bits, load);
        // the form of one chain (8-bit, us per K-step: 512 x 11008 x 4096, 172 tiles: 0.87; 768 x 8192 x 8192 and 1536 x 4096 x 4096,
        // 192: 0.84 and 0.88; 2048 x 4096 x 4096 and x 11008, 256: 1.02 and 0.98)
        return 4.0 + (k / 64.0) * (0.83 + 0.17 * load * load * load);
    }
    // whole rounds of 256x256 tiles at what the board's power allows (4096^3: 1.55 us per K-step and round)
    const double tiles = (double)((m + 255u) / 256u) * (double)((n + 255u) / 256u);
    const double rounds = (double)(uint64_t)((tiles + cus - 1.0) / cus);
    return 4.0 + rounds * (k / 64.0) * 1.5;
}

// The family's estimate, corrected to what it takes where it meets the tiles (fitted on 665 random shapes with cold weights, 33 ... 1500
// rows; it then scatters by 13 - 21 %, most of all for codes in rows of which a workgroup's 128 are not whole; the tiles' estimate by 6 -
// 8 %).  The lower of the two picks 2 % over the faster form on average (always the tiles 4.5 %, always the family 26 %).
static double family_beside_tiles_us(double us, uint32_t m, uint32_t n, int bits, bool packed)
{
    const double ragged = n % 128u == 0 ? 0.0 : 1.0;
    if (packed) return bits == 8 ? 1.19 * us - 0.7 + 0.0037 * m : 0.97 * us + 1.8 + 0.0044 * m;
    return bits == 8 ? (1.035 + 0.165 * ragged) * us + 0.7 * (ragged - 1.0) + 0.0016 * m : (0.80 + 0.2 * ragged) * us + 2.3;
}

// Whether the row-blocked family, at its estimated time, is the one to run; where tiles of 256 columns run it is not asked.
static bool family_leads_tiles(double family_us, uint32_t m, uint32_t n, uint32_t k, int bits, bool packed, bool second_launch)
{
    if (!prefill_small_tiles(m, n, k, bits)) return family_us < prefill_estimate_us(m, n, k, bits, second_launch);
    const TilePlan t = tile128_plan(m, n, k, bits, 0, second_launch);
    if (!second_launch) return family_us < t.us;  // (the estimates of the time before: see tile128_plan)
    // (packed 4-bit codes in one 64-row block of the family, which reads each code once as a tile does, against split tiles that leave
    // a third of the CUs idle: level, 48 x 11008 x 8192 33.9 against 32.7)
    const uint64_t wgs = (uint64_t)((n + 127u) / 128u) * t.splits, cus = machine_cus();
    const double level = packed && bits == 4 && m <= 64u && t.splits > 1u && !t.finish_launch && wgs * 10u <= cus * 7u ? 1.12 : 1.0;
    return family_beside_tiles_us(family_us, m, n, bits, packed) < level * t.us;
}

// The decode family in row blocks: grid z walks blocks of 16*mb rows.  128 columns x 64 rows (mb = 4, 4 waves: one
// wave per SIMD, 128 accumulator registers) amortises the dequantisation best; smaller row blocks give more
// workgroups when columns x row blocks alone do not fill the machine.  Picked by estimate.  (Columns per workgroup
// are fixed by the code width here: what the kernels over packed weights need.)  max_mb: the largest row block to
// consider, in units of 16 rows; wide8: blocks of 16 rows of 4-bit codes run 8 waves instead of 4.
DecodePlan decode_plan_row_blocks(uint32_t m, uint32_t n, uint32_t k, int bits, uint32_t forced_splits, bool packed = false,
                                  uint32_t max_mb = 4u, bool wide8 = false, bool nibbles = false)
{
    DecodePlan best{};
    double best_t = 0.0;
    const uint32_t only_mb = g_force_row_block.load(std::memory_order_relaxed);
    for (uint32_t mb = bits == 8 ? max_mb : (max_mb < 2u ? max_mb : 2u); mb >= 1u; mb >>= 1) {
        if (only_mb != 0u && mb != only_mb && only_mb <= (bits == 8 ? max_mb : 2u)) continue;
        DecodePlan c;
        c.unit_bits = nibbles ? 4u : 0u;
        c.cols = bits == 8 ? 128u : 256u;
        c.waves = ((bits == 8 && mb <= 2u) || (wide8 && mb == 1u)) ? 8u : 4u;  // wide8: 4-bit codes, 256 columns x 8 waves
        c.mb = mb;
        const uint32_t tiles = ((n + c.cols - 1u) / c.cols) * ((m + 16u * mb - 1u) / (16u * mb));
        // 8-bit codes: split along k until the workgroups fill one round of the 256 CUs, not beyond: measured at m = 40 and 64 over
        // n x k = 4096 x 4096, 8192 x 8192, 11008 x 4096 and 4096 x 11008, every row-block size ran fastest with the most
        // workgroups that still fit one round (4096 x 4096, m = 40, 32-row blocks: 19.3 / 14.4 / 11.2 / 15.7 us with
        // 64 / 128 / 256 / 512 workgroups; 11008 x 4096: 21.2 us with 172, 25.4 us with 344).
        if (bits == 8 && forced_splits == 0) {
            // (at most 16 splits, 8 while k is short: 512 x 4096, m = 48: 11.0 us with 16 splits, 7.0 with 8; 1024 x 8192, m = 32:
            // 9.1 with 16, 10.1 with 8)
            uint32_t s = machine_cus() / (tiles ? tiles : 1u);
            const uint32_t most = k >= 8192u ? 16u : k / 512u > 8u ? k / 512u : 8u;
            if (s > most) s = most;
            for (; s > 1u; --s) {
                set_splits(c, k, bits, s, packed);
                if (c.splits == s) break;  // k divides that way
            }
            set_splits(c, k, bits, s < 1u ? 1u : s, packed);
            const double t = decode_family_estimate_us(m, n, k, bits, c);
            if (best_t == 0.0 || t < best_t) { best_t = t; best = c; }
            continue;
        }
        // 4-bit codes (256 columns per workgroup, so fewer workgroups to begin with): the split factor the estimate likes
        // best; filling the round as above over-splits long k here (4096 x 11008, m = 32: 32.5 against 21.6 us)
        for (uint32_t s = 1; s <= 16u; s += (s < 4u ? 1u : s < 8u ? 2u : 4u)) {
            if (forced_splits && s != 1u) break;
            set_splits(c, k, bits, forced_splits ? forced_splits : s, packed);
            if (!forced_splits && c.splits != s && s != 1u) continue;  // k does not divide that way
            if (!forced_splits && s > 1u && tiles * s > 3u * machine_cus()) break;
            double t = decode_family_estimate_us(m, n, k, bits, c);
            // (packed codes: the kernels of 16-row blocks are the weaker ones there, and the estimate's price of a split sends
            // 17 to 32 rows against many columns to them — 32000 x 4096, m = 32: 47.8 us in two blocks of 16 rows, 32.0 in one of
            // 32 with k split in two; 28672 x 4096: 36.9 / 30.5; 13824 x 5120: 29.8 / 25.4.  With two thirds of that price the
            // pick is within 3 % of the better form on all 45 shapes scanned; for row-major codes the full price picks better.)
            if (packed) t -= 4.0 * (c.splits - 1.0) * m * n / 1.5e6;
            // (row-major codes: only the one block of 32 rows with k split in two is priced too high — 17 to 32 rows against
            // 224 to 250 blocks of columns went to two blocks of 16 rows without a split, a round of workgroups filled exactly:
            // 32000 x 4096, m = 32: 32.1 us against 28.1; 28672 x 4096: 31.2 / 29.1)
            else if (c.splits == 2u && mb == 2u) t -= 3.0 * m * n / 1.5e6;
            if (best_t == 0.0 || t < best_t) { best_t = t; best = c; }
        }
    }
    // 4-bit codes in rows, one block of 32 rows, one workgroup per column block and a third or more of the CUs idle: three splits,
    // as for 16 rows (decode_plan) — the estimate's price of a split keeps it from them while k is short (m = 24 / 32,
    // 36864 x 4096: 40.7 / 41.0 us unsplit, 36.6 / 37.6 split three ways; with k = 8192 the estimate picks the three itself)
    if (bits == 4 && !packed && forced_splits == 0 && m <= 32u && best.mb == 2u && best.splits == 1u && best.cols == 256u) {
        const uint32_t cus = machine_cus(), col_blocks = (n + 255u) / 256u;
        if (col_blocks * 2u > cus && col_blocks * 3u <= cus * 2u) {
            DecodePlan probe = best;
            set_splits(probe, k, bits, 3u, packed);
            if (probe.splits == 3u) best = probe;
        }
    }
    return best;
}

// nibbles: the plan is for 4-bit codes in the 128-column form, which takes the launch shapes of 8-bit codes (bits == 8 here)
DecodePlan decode_plan(uint32_t m, uint32_t n, uint32_t k, int bits, uint32_t forced_splits, bool packed = false, bool nibbles = false)
{
    // 4-bit codes in rows also have a 128-column form (a lane loads 4 bytes of a row, 16 lanes half a cache line — the
    // kernel gives the two halves of a line to workgroups that share an L2): twice the column blocks, so half the splits
    // for the same number of workgroups, and 8 waves from one row on.  It takes the launch shape 8-bit codes of the same
    // n x k would get.  Measured against the 256-column plan over 15 weight shapes x m = 1 .. 64 (us, 128 / 256 columns): up
    // to 24 MiB of codes every m gains (2048 x 8192: 7.8 / 9.6 at m = 1, 9.8 / 14.1 at 16, 12.4 / 17.7 at 64; 4096 x 4096:
    // 6.8 / 7.9, 8.0 / 10.7, 11.4 / 15.4; 6144 x 4096: 8.4 / 9.1, 10.0 / 11.3, 16.1 / 21.2; 4096 x 11008: 11.0 / 11.3, 13.4 /
    // 16.3, 21.4 / 26.3; 11008 x 4096: 11.3 / 11.2, 12.3 / 13.2, 14.6 / 18.9 at 24); up to 40 MiB from 16 rows on (8192 x
    // 8192, m = 16 / 24 / 32: 15.4 / 15.8, 17.4 / 21.3, 18.7 / 21.4; 5120 x 13824: 17.4 / 19.4, 19.6 / 24.3, 20.9 / 24.5; with
    // fewer rows the two are level); up to 64 MiB from 17 rows on, where the 256-column form needs row blocks of its own
    // (8192 x 11008, m = 20 / 24 / 32: 21.3 / 24.7, 22.1 / 25.9, 23.5 / 26.3; 11008 x 8192: 23.3 / 27.1, 24.2 / 27.6, 26.2 / 28.7;
    // 32000 x 4096: 22.8 / 26.0, 23.6 / 25.8, 25.3 / 26.7; 14336 x 8192 and 16384 x 8192: level; 12288 x 12288, 72 MiB: 38.0 /
    // 34.9, 42.8 / 37.3).  More weights stream better in whole lines per workgroup (14336 x 8192, m = 8 /
    // 16: 22.8 / 19.9, 25.1 / 21.2; 16384 x 8192, m = 1 .. 16: 12 - 15 % slower; 12288 x 12288, m = 8 .. 32: 10 - 44 %; 8192 x
    // 28672, m = 1 .. 32: 9 - 31 %; 28672 x 8192: 2 - 5 %).
    // A short k and more than half a round of 128-column blocks: those, unsplit — a split's hand-over costs more than the k it
    // saves (us, this / the plan below, m = 1 / 8 / 16 / 32: 24576 x 1536 8-bit 10.0 / 10.8 / 11.9 / 14.4 against 11.5 / 12.1 /
    // 13.6 / 19.5, 4-bit 9.3 / 9.7 / 10.5 / 12.6 against 10.1 / 11.4 / 12.3 / 19.0; 24576 x 2048 4-bit, m = 8 / 16 / 32: 12.1 / 12.9 /
    // 15.4 against 12.9 / 13.8 / 18.9; 16640 x 2048 8-bit, m = 32: 15.0 / 17.5).  At k = 2048 few rows are level or lose: 20480 x
    // 2048 8-bit, m = 1 / 16: 13.0 / 14.8 against 11.7 / 14.2.  From three quarters of a round on 4 waves lead 8 by 1 - 5 %
    // up to 16 rows (32768 x 1536 8-bit, m = 1: 10.8 / 11.6).
    if (!packed && forced_splits == 0 && m <= 32u && (k <= 1536u || (k <= 2048u && (m > 16u || (bits == 4 && m >= 8u))))) {
        const uint32_t blocks = (n + 127u) / 128u, cus = machine_cus();
        if (blocks * 2u > cus && blocks <= cus) {
            DecodePlan pl;
            pl.cols = 128u;
            pl.waves = m <= 16u && blocks * 4u >= cus * 3u ? 4u : 8u;
            pl.mb = m <= 16u ? 1u : 2u;
            set_splits(pl, k, bits, 1u);
            return pl;
        }
    }
    if (bits == 4 && !packed) {
        const uint64_t code_bytes = (uint64_t)n * k / 2u;
        if (code_bytes <= (24ull << 20) || (m >= 16u && code_bytes <= (40ull << 20)) || (m > 16u && code_bytes <= (64ull << 20)))
            return decode_plan(m, n, k, 8, forced_splits, false, true);
    }
    const uint64_t weight_bytes = (uint64_t)n * k * (uint32_t)bits / 8u;
    // 4-bit codes, 17 to 32 rows, a small or narrow matrix (row-major only: the kernels over packed 4-bit codes are built
    // for 4 waves): the two 16-row blocks run 8 waves each (m = 32, 1024 x 4096: 10.5 against 13.7 us, 17 rows: 10.6 / 17.2; 2048 x 8192:
    // 15.3 / 18.4; 4096 x 4096: 14.3 / 16.6; larger matrices lose: 4096 x 11008: 26.5 / 21.8)
    if (bits == 4 && m > 16 && m <= 32 && forced_splits == 0 && !packed && (weight_bytes <= (8ull << 20) || n <= 2048u))
        return decode_plan_row_blocks(m, n, k, bits, 0, false, 1u, true, nibbles);
    // 8-bit codes, more than 32 rows, but so few columns that even 16-row blocks make at most 40 workgroups per split: only
    // those (the 32- and 64-row kernels spend longer in their reductions than such a launch has; 768 x 5120, m = 48: 7.5
    // against 10.8 us; 1536 x 8960: 10.8 / 14.3; 256 x 7168, m = 128: 7.8 / 11.7; with more blocks the larger ones win:
    // 2048 x 8192, m = 128: 20.2 / 16.3)
    if (bits == 8 && m > 32 && forced_splits == 0 && (uint64_t)((n + 127u) / 128u) * ((m + 15u) / 16u) <= machine_cus() * 5u / 32u)
        return decode_plan_row_blocks(m, n, k, bits, 0, packed, 1u, false, nibbles);
    // More than 32 rows of A; 4-bit codes from 17 rows on: three blocks of 16 rows with their own workgroups beat one
    // 32-row block (n = k = 4096, m = 32: 15.8 against 21.4 us; 28672 x 8192, group 128: 46.5 against 53.0 us).
    if (m > 32 || (bits == 4 && m > 16)) return decode_plan_row_blocks(m, n, k, bits, forced_splits, packed, 4u, false, nibbles);
    DecodePlan pl;
    pl.unit_bits = nibbles ? 4u : 0u;
    // 8-bit codes, 17 to 32 rows, a small or narrow matrix: one 32-row block per workgroup cannot fill the machine without
    // splitting k further than it likes; two blocks of 16 rows with their own workgroups (the second stream hits in cache)
    // and the split that fills one round do (m = 32, n x k = 1024 x 4096: 7.0 against 8.9 us; 2048 x 8192: 10.9 against
    // 14.0; 1024 x 16384: 11.7 against 16.3; 4096 x 2048: 7.9 against 9.3; 4096 x 4096: 10.7 against 10.8; beyond 16 MiB
    // at more than 2048 columns the one block wins: 3072 x 8192: 15.4 against 14.4)
    if (bits == 8 && m > 16 && forced_splits == 0 && (weight_bytes <= (16ull << 20) || n <= 2048u))
        return decode_plan_row_blocks(m, n, k, bits, 0, packed, 1u, false, nibbles);
    {
        // 8-bit codes, 128 columns x 8 waves ("narrow": a lane loads 8 bytes of a row, 16 lanes one 128-byte line)
        // needs half the splits of 256 columns x 4 waves ("wide") for the same number of waves, so half the
        // partial-sum traffic.  Narrow workgroups run one per CU, so they pay for a ragged last round of 256.
        // Measured (n = 4096, 8192, 11008, 28672): narrow wins while the weights are few (latency-bound
        // launch), for m >= 8 (partial sums weigh most), and elsewhere when its best split factor fills whole
        // rounds; otherwise large matrices stream better in 256-byte row segments.  4-bit codes: wide.
        const bool few = weight_bytes <= (32ull << 20);
        // Up to 8 rows and 24 to 72 MiB of weights, the narrow form runs 4 waves instead of 8: each has twice the steps behind its
        // first loads, the workgroup half the sums to add through LDS, and k divides into more split factors (one launch after
        // the other over cold weights, 24 shapes: 1.03 times as fast on average, 0.97 - 1.11; us, 8 / 4 waves, m = 1 / 8: 4096 x 11008
        // 12.7 / 12.1 and 13.8 / 13.0; 8192 x 4096 10.3 / 9.4 and 11.0 / 10.1; 3072 x 8192 9.8 / 9.2 and 10.8 / 9.9; 8192 x 8192 15.6 / 14.8 and
        // 16.6 / 16.0; 3584 x 18944 15.9 / 15.3 and 17.1 / 16.2; level at 4096 x 14336, 16384 x 4096 and 11008 x 4096).  In the four
        // products of a decoder block, replayed as one graph, what is left of it is 0 - 3 % of the step (8 rows; hidden and MLP width 3072 and
        // 8192: 42.5 -> 41.2; 4096 and 11008: 59.7 -> 59.1; 4096 and 14336: 65.0 -> 65.4).  Fewer bytes are over before the longer chain pays (4096 x 4096, m = 1: 7.4 / 8.3), more rows want the
        // waves to hide their activations behind (m = 16: 3072 x 8192 11.7 / 12.0, 2560 x 10240 11.4 / 13.0).
        // (rows of B that are not whole cache lines: 1 % on average and up to 8 % slower over 24 shapes, so whole lines only)
        const bool four_waves = bits == 8 && !packed && !nibbles && m <= 8u && n % 128u == 0 && weight_bytes >= (24ull << 20) && weight_bytes <= (72ull << 20);
        // the split-K partial sums (written, read back and cleared as fp32) stay below a quarter of the weight bytes
        uint32_t cap = (uint32_t)(((uint64_t)k * (uint32_t)bits) / (256u * (m ? m : 1u)));
        if (cap < 1) cap = 1;
        // ... unless the weights are few: such launches are bound by latency, not by traffic, and want workgroups
        // (n = k = 4096, m = 32: 10.7 us with 8 splits against 12.6 us with 4; 16 splits are slower again)
        if (few && cap < 8u) cap = 8u;
        // narrow, large matrix: every further split costs traffic and a longer reduction; whole rounds count
        const uint32_t narrow_blocks = (n + 127u) / 128u;
        uint32_t narrow_splits = 1;
        double best = 0.0;
        const uint32_t cus = machine_cus();
        for (uint32_t s = 1; s <= cap && s <= 16u; ++s) {
            // (only the factors k divides into: another one would be rounded to its neighbour, whose workgroups may fill
            // the rounds far worse — 4-bit codes, 11008 x 8192: 5 splits, 430 workgroups, would have become 4 and 344:
            // 24.3 us at m = 16 against 22.0 with 2 splits)
            DecodePlan probe{};
            probe.unit_bits = nibbles ? 4u : 0u;
            probe.cols = 128u;
            probe.waves = four_waves ? 4u : 8u;
            probe.mb = m <= 16 ? 1u : 2u;
            set_splits(probe, k, bits, s, packed);
            if (probe.splits != s) continue;
            // Packed weights, and 4-bit codes in this form: one round of workgroups at most.  Measured over packed weights,
            // best factor within a round against the best beyond, us.  4-bit codes at m = 4 / 16 / 32: 12288 x 12288 2 splits
            // 26.3 / 28.3 / 33.8, 5 splits 28.8 / 30.6 / 36.2; 22016 x 4096 1 split 20.2 / 21.6 / 24.4, 4 splits 21.1 / 22.5 / 28.0;
            // 14336 x 8192 2 splits 21.1 / 23.7 / 27.1, 4 splits 23.6 / 25.9 / 30.9; only 16384 x 8192 likes two rounds (4 splits
            // 26.1 / 27.4 / 32.3 against 2 splits 29.2 / 29.9 / 32.4).  8-bit codes at m = 8 / 16 / 32: 11008 x 8192 2 splits
            // 20.0 / 21.0 / 24.3, 8 splits 24.5 / 25.3 / 29.9; 22016 x 4096 1 split 18.7 / 19.5 / 22.0, 4 splits 23.3 / 23.9 / 27.9;
            // 12288 x 12288 2 splits 30.5 / 32.7 / 36.3, 5 splits 30.6 / 31.6 / 36.1.  (8-bit codes in rows are within 7 % of
            // their best factor as the formula below picks it: 11008 x 8192, m = 8: 5 splits 22.5, 2 splits 21.0.)
            if ((nibbles || packed) && s > 1u && narrow_blocks * s > cus) break;
            const double rounds = (double)((narrow_blocks * s + cus - 1u) / cus);
            const double g = rounds / s + 0.04 * s * 4096.0 / k;  // time of the rounds + what a split costs, both relative to one pass over k
            if (best == 0.0 || g < best) { best = g; narrow_splits = s; }
        }
        const uint32_t narrow_wgs = narrow_blocks * narrow_splits;
        // (one round, at least 95 % full.  Several rounds of narrow workgroups lose to the wide form however well they fill them,
        // m = 1 / 8 / 16: 36864 x 4096, 6 splits x 288 blocks = 6.75 rounds, 39.8 / 43.3 / 47.9 us, its best factor, 2, 37.1 /
        // 39.4 / 42.7, wide 31.5 / 33.2 / 35.4; 24576 x 4096, 4 x 192 = 3 rounds, 23.6 / 25.7 / 28.2 against 20.5 / 21.8 / 23.5)
        const bool fills_rounds = narrow_wgs <= cus && narrow_wgs * 20u >= cus * 19u;
        // 4-bit codes, 17 to 32 rows, two thirds to three quarters of a round of 128-column blocks (too many 256-column ones for three
        // splits in a round, so that form makes one thin round of 4-wave workgroups, k split in two).  A launch of 4-wave
        // workgroups takes its rounds of one per CU over its splits: with s splits whose workgroups stay within s - 1 rounds, (s - 1) /
        // s of one unsplit pass over k, and here that is s = 4 (us by splits 2 / 3 / 4 / 5 / 6, 22016 x 4096, m = 32: 27.0 / 28.7 / 23.7 /
        // 27.0 / 30.3; 24064 x 3072, m = 18: 19.5 / 20.7 / 18.3 / 19.9 / 22.4).  Against the 256-column form over the whole range, k = 2176
        // ... 5120: 1.02 - 1.23 times as fast at 17 to 20 rows, 0.95 - 1.10 at 28 to 32 (22016 x 4096, m = 18 / 32: 25.4 / 26.6 -> 20.6 /
        // 23.7; 24064 x 5120 28.7 / 29.7 -> 25.1 / 29.1; 23552 x 4352, m = 32: 0.95).  A little past three quarters a fifth split is needed
        // and the gain is gone (24832 x 4608, m = 18 / 32: 26.5 / 28.0, five splits 25.4 / 29.8).  Rows that start in the same few memory
        // channels (multiples of 2048 columns) slow the 128-column form: up to 20 rows it is level there or ahead, beyond it loses up
        // to 10 % (24576 x 5120, m = 18 / 32: 28.9 / 30.5 against 28.7 / 33.5).  Rows that are not whole lines lose 2 - 5 % at 32 (24000 x 4608:
        // 29.5 / 30.5).
        if (nibbles && !packed && forced_splits == 0 && m > 16u && (n + 255u) / 256u * 3u > cus && narrow_blocks * 4u <= cus * 3u && n % 256u == 0 &&
            (n % 2048u != 0 || m <= 20u) && k <= 5120u) {
            DecodePlan probe = pl;
            probe.cols = 128u;
            probe.waves = 4u;
            probe.mb = 2u;
            set_splits(probe, k, bits, 4u, packed);
            if (probe.splits == 4u) return probe;
        }
        // m >= 8 on a wide matrix: once 256-column blocks fill their one round with at most 3 splits (more than 64 of
        // them) their partial sums no longer outweigh the better stream (m = 8 / 16 / 32, wide against narrow:
        // 22016 x 4096 20.9 / 22.7 / 28.2 against 21.9 / 23.4 / 31.6 us; 28672 x 8192 46.2 / 48.3 / 54.2 against 49.8 / 53.1 /
        // 61.5; 18944 x 3584 16.9 / 18.3 / 24.0 against 18.0 / 19.9 / 25.1; with fewer blocks narrow stays ahead:
        // 11008 x 4096 13.9 / 14.9 / 17.9 against 13.8 / 16.5 / 22.1; 14336 x 4096 17.2 / 18.5 / 21.4 against 17.6 / 19.0 / 25.1)
        const bool many_wide_blocks = (n + 255u) / 256u > cus / 4u;
        // (n not a multiple of 16: only the 8-codes-per-lane shape can read the last columns)
        // (packed weights: the kernels are built for 128 columns; packed 4-bit codes: the 256-column form, 4 waves, is at
        // best 6 % ahead — 16384 x 8192 and 32000 x 4096 up to 16 rows — and up to 30 % behind)
        // (... and up to 96 MiB of weights: beyond, 256-column blocks win again unless the narrow ones fill their rounds — m = 8 /
        // 16, wide against narrow: 12288 x 12288 29.3 / 31.9 against 34.3 / 37.4 us; 14336 x 8192 24.8 / 26.9 against 26.2 / 28.3;
        // 32000 x 4096, 250 narrow blocks, stays narrow: 25.0 / 25.2 against 23.7 / 24.5)
        // (whole rounds decide up to 160 MiB: 8192 x 28672, 224 MiB, 4 splits x 64 blocks: narrow 41.5 - 47.9 us at m = 1 .. 16, wide
        // 39.7 - 45.5)
        const bool narrow = bits == 8 && (few || (fills_rounds && weight_bytes <= (160ull << 20)) || n % 16u != 0 ||
                                          (m >= 8 && (packed || (!many_wide_blocks && weight_bytes <= (96ull << 20)))) || (nibbles && packed));
        pl.cols = narrow ? 128u : 256u;
        // 4-bit codes, 8 to 16 rows: the same 256 columns with 8 waves (twice the waves to hide the activation loads and
        // the matrix instructions behind; n = k = 4096, m = 16: 11.6 against 14.7 us, 1024 x 8192: 14.1 / 17.4,
        // 8192 x 8192: 17.2 / 19.2, 28672 x 8192: 36.2 / 37.5; m = 8: 10.1 / 11.2, 10.2 / 12.7, 15.7 / 17.8, 35.1 / 35.3;
        // no difference at m = 1).  The kernels over packed 4-bit codes are built for 4 waves.
        const bool wide8 = bits == 4 && m >= 8u && !packed;
        pl.waves = ((narrow && !four_waves) || wide8) ? 8u : 4u;
        pl.mb = m <= 16 ? 1u : 2u;
        uint32_t splits = forced_splits;
        if (splits == 0) {
            if (narrow && !few) {
                splits = narrow_splits;
            } else {
                // about 256 workgroups of 8 waves or 480 of 4: enough waves on every CU to keep the memory system busy
                const uint32_t col_blocks = (n + pl.cols - 1) / pl.cols;
                // (8 waves: one workgroup per CU, so never a few workgroups past a whole round - 4-bit codes, m = 8,
                // 11008 x 4096: 13.4 us with 5 splits = 215 workgroups, 16.7 with 6 = 258; 22016 x 4096: 20.5 / 28.9)
                // 4-bit codes with 4 waves like one round as well while the column blocks are few (m = 1: 8192 x 8192
                // 14.1 us with 256 workgroups, 15.7 with 416; 5120 x 5120 9.7 / 11.7; 8192 x 4096 10.6 / 11.8; from 100
                // column blocks on the 480 are as good or a little better: 28672 x 8192 35.0 against 36.0)
                // 8-bit codes with 4 waves: one round on every shape measured (m = 1: 11008 x 4096 12.7 us with 215 workgroups,
                // 13.2 with 473; 9216 x 4096 11.7 / 13.1; 5120 x 8192 12.8 / 15.7; 18944 x 3584 15.8 / 17.4; 22016 x 4096
                // 19.6 / 21.8; 28672 x 8192 43.8 / 44.8; a few workgroups past the round are the worst case: 258 -> 15.3 us)
                const bool one_round = pl.waves == 8u || bits == 8 || (bits == 4 && col_blocks <= cus / 4u);
                splits = one_round ? decode_target_wgs_narrow() / col_blocks : (decode_target_wgs() + col_blocks / 2) / col_blocks;
                if (splits > cap) splits = cap;
                // One workgroup per column block that leaves a third or more of the CUs idle: three splits, one and a half to two rounds,
                // once k is long enough to pay for them (m = 8 / 16, 1 split against 3: 4-bit 38400 x 8192 50.4 / 50.8 against
                // 42.1 / 43.4 us, 34816 x 8192 51.2 / 53.9 against 43.4 / 46.3; 8-bit, m = 1 / 8 / 16, 36864 x 8192 59.2 / 62.5 / 66.4
                // against 52.8 / 56.6 / 59.9; no difference at k = 4096: 4-bit 38400 x 4096 27.7 / 28.1 against 27.3 / 28.8)
                // (up to two thirds of a round, so that the three splits stay within two rounds: 40960 x 8192, 160 blocks, m = 1 / 8 / 16:
                // 8-bit 61.4 / 64.9 / 68.6 against 55.3 / 59.1 / 62.7, 4-bit at m = 8 / 16 54.0 / 57.1 against 45.4 / 48.9; 170 blocks alike)
                if (one_round && splits == 1u && col_blocks * 3u <= cus * 2u && col_blocks * 2u > cus && k > 4096u && cap >= 3u) {
                    DecodePlan probe = pl;
                    set_splits(probe, k, bits, 3u, packed);
                    if (probe.splits == 3u) splits = 3u;
                }
                // More column blocks of 4-bit codes, 4 waves: rounds of one workgroup per CU count here as well, and a few
                // workgroups past a round cost 10 - 20 %.  The same cost as for the narrow form (rounds over the splits + what
                // a split costs) ranks the factors as measured (m = 1, k = 4096, us by splits: 22016 columns 5: 16.4, 6: 17.1,
                // 7: 17.7, 8: 15.6; 26624 4: 18.0, 5: 21.5, 6: 20.2, 7: 18.9; 33280 3: 21.7, 4: 24.0, 5: 22.7, 6: 23.4;
                // 45056 2: 29.0, 3: 30.7, 4: 25.4, 5: 28.6; 34816 x 8192 3: 37.9, 4: 41.5, 5: 37.1, 6: 40.3; m = 4 alike).
                if (!one_round) {
                    double least = 0.0;
                    for (uint32_t s = 1; s <= cap && s <= 16u; ++s) {
                        DecodePlan probe = pl;
                        set_splits(probe, k, bits, s, packed);
                        if (probe.splits != s) continue;
                        // (between one and a half and three rounds: two workgroups of 4 waves per CU are what keeps the
                        // memory system busy - 22016 x 4096 with 2 splits, 172 workgroups, one round: 18.3 us)
                        if (col_blocks * s * 2u < cus * 3u || col_blocks * s > cus * 3u) continue;
                        const double rounds = (double)((col_blocks * s + cus - 1u) / cus);
                        const double g = rounds / s + 0.04 * s * 4096.0 / k;
                        if (least == 0.0 || g < least) { least = g; splits = s; }
                    }
                }
                // More column blocks than two rounds, fewer than 8 rows: the same cost picks among 1 to 4 splits (m = 1, 151936 x
                // 4096, 594 blocks, us with 1 / 2 / 3 / 4 splits: 8-bit 102.7 / 96.1 / 95.7 / 98.2, 4-bit 85.6 / 80.0 / 80.7 / 83.0;
                // 128256 x 4096, 501 blocks, 1.96 rounds, stays whole: 78.4 / 80.5 and 56.9 / 58.7; from 8 rows on the partial
                // sums take the gain back: m = 8, 594 blocks: 103.2 / 101.4 / 104.4)
                if (col_blocks > 2u * cus && m < 8u) {
                    double least = 0.0;
                    for (uint32_t s = 1; s <= cap && s <= 4u; ++s) {
                        DecodePlan probe = pl;
                        set_splits(probe, k, bits, s, packed);
                        if (probe.splits != s) continue;
                        const double rounds = (double)((col_blocks * s + cus - 1u) / cus);
                        const double g = rounds / s + 0.04 * s * 4096.0 / k;
                        if (least == 0.0 || g < least) { least = g; splits = s; }
                    }
                }
                // a narrow matrix reaches that target only with very many splits, whose waves then run a single step each
                // and whose partial sums the reducing workgroup must collect: beyond 16 splits (32 once k is long enough
                // for four steps per wave) the launch gets slower again.  Measured at m = 1, 16 splits against what the
                // target asks for: 4-bit 1024 x 8192 9.6 / 14.5 us, 1024 x 4096 7.7 / 9.0, 4096 x 8192 10.9 / 12.8,
                // 4096 x 11008 12.7 / 13.9; 8-bit 1024 x 8192 7.9 / 9.3, 256 x 16384 8.6 / 13.6; 32 splits: 4-bit
                // 1024 x 16384 12.2 (16: 14.0, 64: 15.5), 1024 x 28672 15.5 (16: 19.5, 56: 16.8).
                const uint32_t most = k >= (bits == 4 ? 16384u : 24576u) ? 32u : 16u;
                if (splits > most) splits = most;
            }
        }
        set_splits(pl, k, bits, splits, packed);
    }
    return pl;
}

// The decode family up to 32 rows of A; beyond that whichever of the two the estimates favour (the prefill
// kernel's 256x256 tiles leave most of the machine idle until m*n reaches a few hundred tiles).
int resolve_variant(uint32_t m, uint32_t n, uint32_t k, int bits, int variant, bool second_launch = true)
{
    if (variant == BFAINTB_VARIANT_AUTO) {
        if (m <= kDecodeAutoMaxM) return BFAINTB_VARIANT_DECODE;
        if (m > kDecodeFamilyAutoMaxM || wide_tiles_run(m, n, k, bits, second_launch)) return BFAINTB_VARIANT_PREFILL;
        const DecodePlan pl = decode_plan(m, n, k, bits, 0);
        return family_leads_tiles(decode_family_time_us(m, n, k, bits, pl), m, n, k, bits, false, second_launch) ? BFAINTB_VARIANT_DECODE : BFAINTB_VARIANT_PREFILL;
    }
    if (variant == BFAINTB_VARIANT_DECODE) return m <= kDecodeMaxM ? variant : BFAINTB_ERR_BAD_VARIANT;
    if (is_prefill(variant)) return variant;
    return BFAINTB_ERR_BAD_VARIANT;
}

// 17 to 32 rows whose launch by the library's own choice goes to tiles of 32 rows x 128 columns, unsplit, instead of the family (which
// keeps its place for calls that name it, and its scratch is asked for all the same).  pitch: codes from one row of B to the next.
// us, family / tiles (32 rows of A unless said; B cold):
// Over 174 random shapes that it takes, 17 ... 32 rows, 1.12 times as fast as the family.
//   - nine sixteenths of a round of tiles at least; with fewer the family's split fills the machine (128 tiles, k = 4096: 8-bit 19.9 /
//     24.6, 4-bit 18.0 / 24.3).
//   - packed 4-bit codes, however many rounds: 22016 x 4096 23.5 / 21.1, 32768 x 4096 27.4 / 22.7, 27008 x 1280 12.7 / 10.8, 50304 x
//     4096 44.9 / 40.6; level at k = 6144 (29.5 / 29.3), behind at 8192 (36.2 / 38.6), where the family's longer walk amortises its
//     start.  The family walks in whole steps of 1024 rows and is at its best where k is just those and they are few: over 24 calls each, 18432 to
//     50304 columns, family / tiles on average 1.09 at k = 1536, 1.00 at 1920, 0.985 at 2048 (0.945 - 1.03), 1.15 at 2176 (a third step), 1.14
//     at 2560, 1.06 at 3072, 1.11 at 4096, 1.03 at 5120: so not at 2048, its two whole steps.
//   - packed 8-bit codes: 20480 x 4096 22.9 / 20.7, 22016 x 5120 28.6 / 26.5, 50304 x 4096 47.5 / 44.0; a short k has too few steps to
//     fill the pipeline (22016 x 2048 15.6 / 17.3), a long one is level or behind (28672 x 6144, 20 rows 31.4 / 33.3), and so are several rounds with one scale per column
//     (50944 x 3456, 20 rows 38.4 / 40.5, 34560 x 3584, 29 rows 38.5 / 40.3; groups of 128, 47344 x 4096, 30 rows 49.2 / 44.1).
//   - codes in rows: one round of tiles at most (36864 x 4096, 288 tiles: 8-bit 41.9 / 45.3, 4-bit 37.8 / 43.8), and not where the rows lie
//     a multiple of 1024 codes apart, which crowds the memory channels and which whole rows of 128 columns feel more than the family's
//     blocks do (8-bit 20480 x 4096 27.3 / 28.7, 18432 x 4096 26.1 / 26.9, 23552 x 5880, 29 rows 37.8 / 43.3).  Otherwise 8-bit 22016 x 4096 26.5 / 24.3, 18560 x
//     2432 20.7 / 15.5, 31328 x 1152, 24 rows, 14.3 / 12.0, 27808 x 4992, 17 rows, 36.3 / 30.6; 4-bit 22016 x 4096 23.7 / 21.5, 27728 x
//     5504, 20 rows, 32.8 / 27.6.  Up to two thirds of a round only where the family does not split a long k three ways (20272 x 1536 8-bit
//     16.6 / 13.8, 19216 x 2560 4-bit 20.7 / 15.8; 18944 x 4192 8-bit 23.4 / 25.3, 18560 x 6272 4-bit 26.7 / 29.3).  Up to 20 rows of 4-bit codes only where rows are not whole lines (22016 x 5120, 20 rows: 24.4 / 25.0).
static bool few_rows_on_tiles(uint32_t m, uint32_t n, uint32_t k, int bits, bool grouped, bool packed, uint32_t pitch)
{
    const uint32_t cus = machine_cus(), tiles = n / 128u + (n % 128u != 0u);
    if (m < 17u || m > 32u || tiles * 16ull < cus * 9ull) return false;
    if (packed && bits == 4) return k > 1024u && k <= 5120u && k != 2048u;
    if (packed) return k >= 3072u && k <= 5632u && (tiles <= cus || grouped);
    if (tiles * 3ull <= cus * 2ull && k > 4096u) return false;
    if (tiles > cus || pitch % 1024u == 0u || k <= 1024u || k >= 8192u) return false;
    return bits == 8 || m > 20u || pitch % 256u != 0u;
}

static hipError_t launch_few_rows_on_tiles(GemmParams p, int bits, bool packed, hipStream_t stream)
{
    p.k_per_wg = (p.k + 63u) / 64u * 64u;  // (whole K-steps)
    p.splits = 1u;
    p.tile_blocks = 2u;
    p.finish_launch = 0u;
    return bfaintb::launch_prefill128_wreg(p, bits, packed, stream);
}

// whether a tiled-variant launch over row-major weights goes to the small-tile kernel that can split k
static bool tiled_may_split(int v, uint32_t m, uint32_t n, uint32_t k, int bits, uint32_t split_k = 0)
{
    return use_small_tiles(v, m, n, k, bits) && v != BFAINTB_VARIANT_PREFILL_128_LDS && !(v == BFAINTB_VARIANT_PREFILL && wide_tiles(m, n, k, bits, split_k).blocks != 0u);
}

size_t workspace_need(uint32_t m, uint32_t n, uint32_t k, int bits, int variant, uint32_t forced_split)
{
    if (m == 0 || n == 0) return 0;
    if (variant == BFAINTB_VARIANT_DECODE) return split_workspace_bytes(decode_plan(m, n, k, bits, forced_split).splits, m, n);
    if (is_prefill(variant) && tiled_may_split(variant, m, n, k, bits, forced_split)) return tile_workspace_bytes(tile128_plan(m, n, k, bits, forced_split), m, n);
    return 0;
}

inline bool misaligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) != 0; }

// ---- per-device set-up: kernel attributes, and the address and first filling of the static scratch ----
constexpr int kMaxDevices = 64;
struct DeviceState {
    std::atomic<int> ready{0};      // kernel attributes set on this device
    std::atomic<int> scratch_ready{0};  // static scratch resolved and filled with the empty pattern
    void* scratch_ptr = nullptr;
};
DeviceState g_devices[kMaxDevices];
std::mutex g_setup_mutex;
std::atomic<uint32_t> g_split_wait_limit{bfaintb::kDefaultSplitWaitLimit};
std::atomic<uint32_t> g_debug_flags{0};

bool stream_is_capturing(hipStream_t stream)
{
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &status) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return status != hipStreamCaptureStatusNone;
}

// The current device's state, its kernels prepared.  The set-up makes runtime calls that are not stream operations, so
// it must not run for the first time under stream capture: such a call is refused (BFAINTB_ERR_NOT_INITIALISED) and
// bfaintb_init is the way to run it beforehand.
int device_state(hipStream_t stream, DeviceState** out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= kMaxDevices) return BFAINTB_ERR_UNSUPPORTED;
    DeviceState& st = g_devices[dev];
    if (!st.ready.load(std::memory_order_acquire)) {
        if (stream_is_capturing(stream)) return BFAINTB_ERR_NOT_INITIALISED;
        std::lock_guard<std::mutex> lock(g_setup_mutex);
        if (!st.ready.load(std::memory_order_relaxed)) {
            e = bfaintb::decode_prepare_device();
            if (e != hipSuccess) return (int)e;
            st.ready.store(1, std::memory_order_release);
        }
    }
    *out = &st;
    return BFAINTB_OK;
}

// The launches of one call that meet in a workspace (the tiles of a product and the second launch that adds their sums; the two
// fills of an initialisation) leave and expect it at rest as one: on a stream nothing else that uses the workspace may come
// between them, also where two host threads share stream and workspace.  So every launch that uses a workspace is made under
// a lock that belongs to the workspace's address (one of 64: threads with workspaces of their own hardly ever meet), held
// over all of the call's launches and nothing else.
std::mutex& workspace_order(const void* workspace)
{
    static std::mutex locks[64];
    return locks[(reinterpret_cast<uintptr_t>(workspace) >> 8) * 0x9e3779b97f4a7c15ull >> 58];
}

int init_workspace_on(void* workspace, size_t workspace_bytes, hipStream_t stream)
{
    if (workspace_bytes % 4 != 0 || workspace_bytes / 4 >= (1ull << 32) || workspace_bytes < bfaintb::kWorkspaceHeaderBytes)
        return BFAINTB_ERR_WORKSPACE;
    // every word becomes "no partial sum here" (and "no failure" in the header), then the header gets its mark; fill
    // kernels rather than hipMemsetAsync, so that the call may be recorded into a HIP graph
    std::lock_guard<std::mutex> in_order(workspace_order(workspace));
    hipError_t e = bfaintb::launch_fill_u32(static_cast<uint32_t*>(workspace), (uint32_t)(workspace_bytes / 4), kEmptyWord, stream);
    if (e == hipSuccess) e = bfaintb::launch_fill_u32(static_cast<uint32_t*>(workspace) + 1, 1u, bfaintb::kWorkspaceMagic, stream);
    return (int)e;
}

// The device's static scratch, resolved and (the first time, outside any capture) filled with the empty pattern.
int static_scratch(DeviceState& st, hipStream_t stream, void** out)
{
    if (!st.scratch_ready.load(std::memory_order_acquire)) {
        if (stream_is_capturing(stream)) return BFAINTB_ERR_NOT_INITIALISED;
        std::lock_guard<std::mutex> lock(g_setup_mutex);
        if (!st.scratch_ready.load(std::memory_order_relaxed)) {
            void* ptr = nullptr;
            hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
            if (e != hipSuccess) return (int)e;
            if (ptr == nullptr) return BFAINTB_ERR_WORKSPACE;
            const int rc = init_workspace_on(ptr, BFAINTB_STATIC_SCRATCH_BYTES, stream);
            if (rc) return rc;
            e = hipStreamSynchronize(stream);  // once per device: every stream may use the scratch from here on
            if (e != hipSuccess) return (int)e;
            st.scratch_ptr = ptr;
            st.scratch_ready.store(1, std::memory_order_release);
        }
    }
    *out = st.scratch_ptr;
    return BFAINTB_OK;
}

}  // namespace

extern "C" {

static uint32_t row_split_head(uint32_t m, uint32_t n, uint32_t k, int bits, bool packed, bool grouped);
static size_t row_split_workspace(uint32_t head, uint32_t rest, uint32_t n, uint32_t k, int bits, bool packed);

int bfaintb_version(void) { return BFAINTB_VERSION; }

const char* bfaintb_error_string(int code)
{
    switch (code) {
        case BFAINTB_OK: return "success";
        case BFAINTB_ERR_NULL_POINTER: return "null device pointer";
        case BFAINTB_ERR_BAD_SHAPE: return "unsupported shape: need n % 8 == 0 (4-bit codes: n % 16 == 0), k % 8 == 0, k > 0, sizes below 2^31; pre-packed weights: n % 16 == 0, k % 64 == 0 (4-bit: k % 128 == 0)";
        case BFAINTB_ERR_BAD_LD: return "bad leading dimension: need lda >= k, n <= ldb < 2^27, ldc >= n, lda % 8 == 0, ldb % 16 == 0, ldc % 8 == 0";
        case BFAINTB_ERR_ALIGNMENT: return "pointer not 16-byte aligned";
        case BFAINTB_ERR_UNSUPPORTED: return "unsupported format: weight_bits must be 8 or 4; group_size 0 or a multiple of 32 that divides k";
        case BFAINTB_ERR_WORKSPACE: return "workspace missing or smaller than bfaintb_gemm_workspace_bytes reports";
        case BFAINTB_ERR_BAD_VARIANT: return "unknown kernel variant, or variant cannot run this shape";
        case BFAINTB_ERR_NOT_INITIALISED: return "first call on this device made under stream capture: call bfaintb_init() beforehand";
        case BFAINTB_ERR_WORKSPACE_POISONED: return "a split-K wait gave up on this workspace (results of that call hold NaNs): initialise it again";
        case BFAINTB_ERR_STATIC_SCRATCH: return "shape needs more split-K scratch than bfaintb_gemm_static holds (16 MiB): use bfaintb_gemm with a workspace";
        default: break;
    }
    if (code > 0) return hipGetErrorString(static_cast<hipError_t>(code));
    return "unknown bfaintb error code";
}

int bfaintb_gemm_variant(uint32_t m, uint32_t n, uint32_t k, int weight_bits, uint32_t group_size)
{
    int e = check_format(k, weight_bits, group_size);
    if (e) return e;
    e = check_shape(m, n, k, weight_bits);
    if (e) return e;
    return resolve_variant(m, n, k, weight_bits, BFAINTB_VARIANT_AUTO);
}

uint32_t bfaintb_gemm_split_k(uint32_t m, uint32_t n, uint32_t k, int weight_bits, uint32_t group_size)
{
    int v = bfaintb_gemm_variant(m, n, k, weight_bits, group_size);
    if (v >= 0) {
        const uint32_t head = row_split_head(m, n, k, weight_bits, false, group_size != 0);
        if (head != 0u) {
            m = head;
            v = resolve_variant(m, n, k, weight_bits, BFAINTB_VARIANT_AUTO);
        }
    }
    if (v == BFAINTB_VARIANT_DECODE) return decode_plan(m, n, k, weight_bits, 0).splits;
    if (v == BFAINTB_VARIANT_PREFILL && tiled_may_split(v, m, n, k, weight_bits)) return tile128_plan(m, n, k, weight_bits, 0).splits;
    return 1;
}

size_t bfaintb_gemm_workspace_bytes_ex(uint32_t m, uint32_t n, uint32_t k, int weight_bits, uint32_t group_size, int variant,
                                       uint32_t split_k)
{
    if (check_format(k, weight_bits, group_size) || check_shape(m, n, k, weight_bits)) return 0;
    const int v = resolve_variant(m, n, k, weight_bits, variant);
    if (v < 0) return 0;
    if (variant == BFAINTB_VARIANT_AUTO && split_k == 0) {
        const uint32_t head = row_split_head(m, n, k, weight_bits, false, group_size != 0);
        if (head != 0u) return row_split_workspace(head, m - head, n, k, weight_bits, false);
    }
    return workspace_need(m, n, k, weight_bits, v, split_k);
}

size_t bfaintb_gemm_workspace_bytes(uint32_t m, uint32_t n, uint32_t k, int weight_bits, uint32_t group_size)
{
    return bfaintb_gemm_workspace_bytes_ex(m, n, k, weight_bits, group_size, BFAINTB_VARIANT_AUTO, 0);
}

int bfaintb_workspace_init(void* workspace, size_t workspace_bytes, void* stream)
{
    if (workspace == nullptr || workspace_bytes == 0) return BFAINTB_OK;
    if (misaligned16(workspace)) return BFAINTB_ERR_ALIGNMENT;
    return init_workspace_on(workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}

int bfaintb_workspace_status(const void* workspace, void* stream)
{
    if (workspace == nullptr) return BFAINTB_ERR_NULL_POINTER;
    uint32_t header[2] = {0, 0};
    hipStream_t st = static_cast<hipStream_t>(stream);
    hipError_t e = hipMemcpyAsync(header, workspace, sizeof(header), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) return (int)e;
    if (header[1] != bfaintb::kWorkspaceMagic) return BFAINTB_ERR_WORKSPACE;
    return header[0] == kEmptyWord ? BFAINTB_OK : BFAINTB_ERR_WORKSPACE_POISONED;
}

// The same two calls for the scratch of bfaintb_gemm_static, whose address the library keeps to itself.
int bfaintb_static_scratch_status(void* stream)
{
    hipStream_t st = static_cast<hipStream_t>(stream);
    DeviceState* dev = nullptr;
    int rc = device_state(st, &dev);
    if (rc) return rc;
    void* ptr = nullptr;
    rc = static_scratch(*dev, st, &ptr);
    if (rc) return rc;
    return bfaintb_workspace_status(ptr, stream);
}

int bfaintb_static_scratch_reset(void* stream)
{
    hipStream_t st = static_cast<hipStream_t>(stream);
    DeviceState* dev = nullptr;
    int rc = device_state(st, &dev);
    if (rc) return rc;
    void* ptr = nullptr;
    rc = static_scratch(*dev, st, &ptr);  // (the first call on a device fills it anyway)
    if (rc) return rc;
    return init_workspace_on(ptr, BFAINTB_STATIC_SCRATCH_BYTES, st);
}

int bfaintb_init(void* stream)
{
    hipStream_t st = static_cast<hipStream_t>(stream);
    DeviceState* dev = nullptr;
    int rc = device_state(st, &dev);
    if (rc) return rc;
    (void)machine_cus();  // the device's compute units, asked for here rather than by a first plan made under capture
    void* ptr = nullptr;
    return static_scratch(*dev, st, &ptr);
}

// The two hooks that change what split-K launches do are for the library's own tests: they work only in a process that
// has BFAINTB_TEST_HOOKS=1 in its environment (read when the first of them is asked for), so that a stray call in a host
// application cannot turn every split-K result of the process into NaNs.
static bool test_hooks_armed()
{
    static const bool armed = [] {
        const char* v = getenv("BFAINTB_TEST_HOOKS");
        return v != nullptr && strcmp(v, "1") == 0;
    }();
    return armed;
}

int bfaintb_debug_control(uint32_t what, uint32_t value)
{
    if ((what == BFAINTB_DEBUG_SPLIT_WAIT_LIMIT || what == BFAINTB_DEBUG_WITHHOLD_PARTIALS) && !test_hooks_armed()) return BFAINTB_ERR_UNSUPPORTED;
    switch (what) {
        case BFAINTB_DEBUG_SPLIT_WAIT_LIMIT:
            g_split_wait_limit.store(value ? value : bfaintb::kDefaultSplitWaitLimit);
            return BFAINTB_OK;
        case BFAINTB_DEBUG_WITHHOLD_PARTIALS:
            if (value) g_debug_flags.fetch_or(bfaintb::kDebugWithholdPartials);
            else g_debug_flags.fetch_and(~bfaintb::kDebugWithholdPartials);
            return BFAINTB_OK;
        case BFAINTB_DEBUG_FORCE_ROW_BLOCK:
            if (value != 0u && value != 1u && value != 2u && value != 4u) return BFAINTB_ERR_UNSUPPORTED;
            g_force_row_block.store(value);
            return BFAINTB_OK;
        case BFAINTB_DEBUG_PLAN_COMPUTE_UNITS:
            if (value > 4096u) return BFAINTB_ERR_UNSUPPORTED;
            g_plan_cus_override.store(value);
            return BFAINTB_OK;
        default: return BFAINTB_ERR_UNSUPPORTED;
    }
}

// what the epilogue descriptor asks for, checked: bias and residual pointers (either may be null) and the residual's row stride
struct Epilogue {
    const void* bias = nullptr;
    const void* residual = nullptr;
    uint32_t ldr = 0;
    uint32_t activation = BFAINTB_ACT_NONE;
    // not an epilogue but set the same way: the reference kernel's arithmetic (fp32 scales, W and C narrowed by truncation)
    bool reference_arith = false;
    // columns of C (and of the residual) for n columns of B
    uint32_t out_cols(uint32_t n) const { return activation == BFAINTB_ACT_SILU_GATE ? n / 2u : n; }
    // the same for the rows of C from `row` on
    Epilogue from_row(uint32_t row) const
    {
        Epilogue e = *this;
        if (residual != nullptr) e.residual = static_cast<const uint16_t*>(residual) + (size_t)row * ldr;
        return e;
    }
};

static int read_epilogue(Epilogue& out, const bfaintb_epilogue* ep, uint32_t n)
{
    if (ep == nullptr) return BFAINTB_OK;
    if (ep->activation != BFAINTB_ACT_NONE && ep->activation != BFAINTB_ACT_SILU_GATE) return BFAINTB_ERR_UNSUPPORTED;
    out.bias = ep->bias;
    out.residual = ep->residual;
    out.ldr = ep->ldr;
    out.activation = ep->activation;
    if (ep->residual != nullptr && (ep->ldr < out.out_cols(n) || ep->ldr % 8u != 0)) return BFAINTB_ERR_BAD_LD;
    if (ep->activation == BFAINTB_ACT_SILU_GATE && n % 16u != 0) return BFAINTB_ERR_BAD_SHAPE;  // n / 2 output columns, stored 8 at a time
    return BFAINTB_OK;
}

// points the kernel at a split-K workspace: header first, partial sums behind it
static int attach_workspace(GemmParams& p, void* workspace, size_t workspace_bytes, size_t need)
{
    if (workspace == nullptr || workspace_bytes < need) return BFAINTB_ERR_WORKSPACE;
    if (misaligned16(workspace)) return BFAINTB_ERR_ALIGNMENT;
    if (need >= (1ull << 31)) return BFAINTB_ERR_BAD_VARIANT;  // the kernel addresses the workspace with 32-bit offsets
    p.ws_header = static_cast<uint32_t*>(workspace);
    p.partials = reinterpret_cast<unsigned long long*>(static_cast<uint8_t*>(workspace) + bfaintb::kWorkspaceHeaderBytes);
    p.partial_bytes = (uint32_t)(need - bfaintb::kWorkspaceHeaderBytes);
    p.split_wait_limit = g_split_wait_limit.load(std::memory_order_relaxed);
    p.debug_flags = g_debug_flags.load(std::memory_order_relaxed);
    return BFAINTB_OK;
}

// Whether two launches by rows can be made with what the caller brings: the scratch they need (a caller who brings less, or
// none, gets the one launch over all rows, which may need none), and a device whose set-up is done or can be done now (one
// launch of the tiled kernels needs none, so a capture before any other call keeps working).
static bool row_split_served(const void* workspace, size_t workspace_bytes, size_t need, bool use_static_scratch, hipStream_t stream)
{
    DeviceState* dev = nullptr;
    if (!use_static_scratch && need != 0 && (workspace == nullptr || workspace_bytes < need || misaligned16(workspace))) return false;
    if (device_state(stream, &dev) != 0) return false;
    void* scratch_ptr = nullptr;
    return !use_static_scratch || need == 0 || static_scratch(*dev, stream, &scratch_ptr) == 0;
}

static int gemm_impl(void* c, const void* a, const void* b, const void* scale, const Epilogue& ep, uint32_t m, uint32_t n, uint32_t k,
                     uint32_t lda, uint32_t ldb, uint32_t ldc, int weight_bits, uint32_t group_size, void* workspace,
                     size_t workspace_bytes, void* stream, int variant, uint32_t split_k, bool use_static_scratch = false, bool whole = false,
                     bool second_launch = true)
{
    const void* bias = ep.bias;
    int e = check_format(k, weight_bits, group_size);
    if (e) return e;
    if (ep.reference_arith && (weight_bits != 8 || group_size != 0)) return BFAINTB_ERR_UNSUPPORTED;
    e = check_shape(m, n, k, weight_bits);
    if (e) return e;
    if (lda < k || ldb < n || ldc < ep.out_cols(n) || lda % 8u != 0 || ldb % 16u != 0 || ldc % 8u != 0) return BFAINTB_ERR_BAD_LD;
    if (ldb >= (1u << 27)) return BFAINTB_ERR_BAD_LD;  // a lane's offset within 32 rows of B is kept in 32 bits
    // (the reference's arithmetic has no form that splits the tiles' k, let alone one with a second launch: where only that lets the
    // tiles lead, the family runs, at 96 x 4096 x 11008 34 us against 144; only a caller without its scratch gets the tiles)
    const int v = resolve_variant(m, n, k, weight_bits, variant, second_launch != ep.reference_arith);
    if (v < 0) return v;
    if (m == 0 || n == 0) return BFAINTB_OK;
    if (c == nullptr || a == nullptr || b == nullptr || scale == nullptr) return BFAINTB_ERR_NULL_POINTER;
    if (misaligned16(c) || misaligned16(a) || misaligned16(b) || misaligned16(scale) || misaligned16(bias) || misaligned16(ep.residual))
        return BFAINTB_ERR_ALIGNMENT;
    if (!whole && variant == BFAINTB_VARIANT_AUTO && split_k == 0 && !ep.reference_arith) {
        const uint32_t head = row_split_head(m, n, k, weight_bits, false, group_size != 0);
        if (head != 0u && row_split_served(workspace, workspace_bytes, row_split_workspace(head, m - head, n, k, weight_bits, false), use_static_scratch,
                                           static_cast<hipStream_t>(stream))) {
            e = gemm_impl(c, a, b, scale, ep, head, n, k, lda, ldb, ldc, weight_bits, group_size, workspace, workspace_bytes, stream, variant, 0,
                          use_static_scratch, true);
            if (e) return e;
            return gemm_impl(static_cast<uint16_t*>(c) + (size_t)head * ldc, static_cast<const uint16_t*>(a) + (size_t)head * lda, b, scale,
                             ep.from_row(head), m - head, n, k, lda, ldb, ldc, weight_bits, group_size, workspace, workspace_bytes, stream, variant, 0,
                             use_static_scratch, true);
        }
    }

    GemmParams p{};
    p.bias = static_cast<const uint16_t*>(bias);
    p.residual = static_cast<const uint16_t*>(ep.residual);
    p.ldr = ep.ldr;
    p.activation = ep.activation;
    p.reference_arith = ep.reference_arith ? 1u : 0u;
    p.c = static_cast<uint16_t*>(c);
    p.a = static_cast<const uint16_t*>(a);
    p.b = static_cast<const uint8_t*>(b);
    p.scale = static_cast<const uint16_t*>(scale);
    p.m = m; p.n = n; p.k = k;
    p.lda = lda;
    p.ldb_bytes = weight_bits == 8 ? ldb : ldb / 2u;
    p.ldc = ldc;
    p.lds = n;
    p.group_size = group_size;
    bfaintb::set_group_division(p);
    p.cus = machine_cus();
    p.k_per_wg = k;
    p.splits = 1;
    hipStream_t st = static_cast<hipStream_t>(stream);

    const bool tiled = is_prefill(v);
    bool small_wreg = false;  // the small-tile kernel that keeps row-major weights in registers (and may split k)
    if (tiled) {
        // the prefill kernel addresses B and a 256-row panel of A through 32-bit buffer extents
        if ((uint64_t)k * p.ldb_bytes >= (1ull << 31) || (uint64_t)256 * lda * 2u >= (1ull << 31)) return BFAINTB_ERR_BAD_SHAPE;
#ifdef BFAINTB_TRACE
        p.trace = static_cast<unsigned long long*>(workspace);  // per-quarter cycle totals, 8 words per wave
        return (int)bfaintb::launch_prefill(p, weight_bits, st, v != BFAINTB_VARIANT_PREFILL_256_LDS);
#endif
        // row-major weights on small tiles: that form, unless the other one is asked for by name
        small_wreg = tiled_may_split(v, m, n, k, weight_bits, split_k) && bfaintb::prefill128_wreg_serves(p);
        if (small_wreg) {
            const TilePlan tp = tile128_plan(m, n, k, weight_bits, split_k, second_launch);
            p.k_per_wg = tp.k_per_wg;
            p.splits = tp.splits;
            p.tile_blocks = tp.blocks;
            p.finish_launch = tp.finish_launch;
        }
    } else {
        const DecodePlan pl = decode_plan(m, n, k, weight_bits, split_k);
        p.k_per_wg = pl.k_per_wg;
        p.splits = pl.splits;
        p.decode_waves = pl.waves;
        p.decode_cols = pl.cols;
        p.decode_mb = pl.mb;
    }
    // with less scratch than this plan needs: what the library does without a second launch may need less, or none
    auto without_second_launch = [&] {
        return gemm_impl(c, a, b, scale, ep, m, n, k, lda, ldb, ldc, weight_bits, group_size, workspace, workspace_bytes, stream, variant, split_k,
                         use_static_scratch, true, false);
    };
    // (every argument check comes before the first runtime call)
    const size_t need = split_workspace_bytes(p.splits + p.finish_launch, m, n);
    if (p.splits > 1 && !use_static_scratch) {
        e = attach_workspace(p, workspace, workspace_bytes, need);
        if (e) return second_launch ? without_second_launch() : e;
    }
    if (use_static_scratch && need > BFAINTB_STATIC_SCRATCH_BYTES) return BFAINTB_ERR_STATIC_SCRATCH;
    DeviceState* dev = nullptr;
    if (!tiled || (p.splits > 1 && use_static_scratch)) {
        e = device_state(st, &dev);
        if (e) return p.finish_launch ? without_second_launch() : e;  // (a first call under capture)
    }
    if (p.splits > 1 && use_static_scratch) {
        void* static_ptr = nullptr;
        e = static_scratch(*dev, st, &static_ptr);
        if (e) return p.finish_launch ? without_second_launch() : e;
        workspace = static_ptr;
        e = attach_workspace(p, workspace, BFAINTB_STATIC_SCRATCH_BYTES, need);
        if (e) return e;
    }
    // (the tiled kernel addresses B and the rows of A through 32-bit buffer extents; the reference's arithmetic has no such form)
    if (variant == BFAINTB_VARIANT_AUTO && !tiled && split_k == 0 && !ep.reference_arith && few_rows_on_tiles(m, n, k, weight_bits, group_size != 0, false, ldb) &&
        (uint64_t)k * p.ldb_bytes < (1ull << 31) && (uint64_t)256 * lda * 2u < (1ull << 31))
        return (int)launch_few_rows_on_tiles(p, weight_bits, false, st);
    std::unique_lock<std::mutex> in_order;
    if (p.splits > 1) in_order = std::unique_lock<std::mutex>(workspace_order(p.ws_header));
    if (tiled) {
        if (small_wreg) return (int)bfaintb::launch_prefill128_wreg(p, weight_bits, false, st);
        if (v == BFAINTB_VARIANT_PREFILL && !p.reference_arith) {
            p.tile_blocks = wide_tiles(m, n, k, weight_bits).blocks;
            if (p.tile_blocks != 0u) return (int)bfaintb::launch_prefill(p, weight_bits, st, true);
        }
        if (v == BFAINTB_VARIANT_PREFILL && !tall_tiles_in_one_chain(m, k) && prefill_tall_tiles(m, n, k, weight_bits) && bfaintb::prefill128_wreg_serves(p)) {
            p.tile_blocks = tall_tile_blocks(m);
            p.k_per_wg = (k + 63u) / 64u * 64u;  // (whole K-steps)
            return (int)bfaintb::launch_prefill128_wreg(p, weight_bits, false, st);
        }
        if ((v == BFAINTB_VARIANT_PREFILL_256X128 || (v == BFAINTB_VARIANT_PREFILL && prefill_tall_tiles(m, n, k, weight_bits))) && !p.reference_arith)
            return (int)bfaintb::launch_prefill256x128_wreg(p, weight_bits, false, st);
        if (use_small_tiles(v, m, n, k, weight_bits)) return (int)bfaintb::launch_prefill128(p, weight_bits, false, st);
        return (int)bfaintb::launch_prefill(p, weight_bits, st, v != BFAINTB_VARIANT_PREFILL_256_LDS);
    }
#ifdef BFAINTB_TRACE
    // timestamp sink: behind the split-K area (instrumented callers pass a larger workspace)
    p.trace = reinterpret_cast<unsigned long long*>(static_cast<uint8_t*>(workspace) + ((workspace_need(m, n, k, weight_bits, BFAINTB_VARIANT_DECODE, split_k) + 255) & ~(size_t)255));
#endif
    return (int)bfaintb::launch_decode(p, weight_bits, st);
}

// the packed order has K-chunks of 64 rows for 8-bit and 128 rows for 4-bit codes
static int check_packed_shape(uint32_t n, uint32_t k, int weight_bits)
{
    const int e = check_shape(1, n, k);
    if (e) return e;
    return (n % 16u != 0 || k % (weight_bits == 4 ? 128u : 64u) != 0) ? BFAINTB_ERR_BAD_SHAPE : BFAINTB_OK;
}

size_t bfaintb_prepack_bytes(uint32_t n, uint32_t k, int weight_bits)
{
    if ((weight_bits != 8 && weight_bits != 4) || check_packed_shape(n, k, weight_bits)) return 0;
    return (size_t)n * k * (uint32_t)weight_bits / 8u;
}

int bfaintb_packed_header_init(bfaintb_packed_header* h, uint32_t n, uint32_t k, int weight_bits, uint32_t group_size, int has_bias)
{
    if (h == nullptr) return BFAINTB_ERR_NULL_POINTER;
    int e = check_format(k, weight_bits, group_size);
    if (e) return e;
    e = check_packed_shape(n, k, weight_bits);
    if (e) return e;
    memset(h, 0, sizeof(*h));
    memcpy(h->magic, "BFAINTB1", 8);
    h->header_bytes = (uint32_t)sizeof(*h);
    h->layout = BFAINTB_LAYOUT_MFMA16;
    h->weight_bits = (uint32_t)weight_bits;
    h->group_size = group_size;
    h->k = k;
    h->n = n;
    h->payload_bytes = (uint64_t)n * k * (uint32_t)weight_bits / 8u;
    h->scale_bytes = (uint64_t)(group_size ? k / group_size : 1u) * n * 2u;
    h->has_bias = has_bias ? 1u : 0u;
    return BFAINTB_OK;
}

int bfaintb_packed_header_check(const bfaintb_packed_header* h)
{
    if (h == nullptr) return BFAINTB_ERR_NULL_POINTER;
    if (memcmp(h->magic, "BFAINTB1", 8) != 0 || h->header_bytes != sizeof(*h) || h->layout != BFAINTB_LAYOUT_MFMA16)
        return BFAINTB_ERR_UNSUPPORTED;
    bfaintb_packed_header want;
    const int e = bfaintb_packed_header_init(&want, h->n, h->k, (int)h->weight_bits, h->group_size, (int)h->has_bias);
    if (e) return e;
    if (h->has_bias > 1u || h->reserved[0] || h->reserved[1] || h->reserved[2]) return BFAINTB_ERR_UNSUPPORTED;
    if (h->payload_bytes != want.payload_bytes || h->scale_bytes != want.scale_bytes) return BFAINTB_ERR_BAD_SHAPE;
    return BFAINTB_OK;
}

static int repack(void* dst, const void* src, uint32_t n, uint32_t k, uint32_t ldb, int weight_bits, void* stream, bool unpack)
{
    if (weight_bits != 8 && weight_bits != 4) return BFAINTB_ERR_UNSUPPORTED;
    const int e = check_packed_shape(n, k, weight_bits);
    if (e) return e;
    if (ldb < n || ldb % 16u != 0) return BFAINTB_ERR_BAD_LD;
    if (n == 0) return BFAINTB_OK;
    if (dst == nullptr || src == nullptr) return BFAINTB_ERR_NULL_POINTER;
    if (misaligned16(dst) || misaligned16(src)) return BFAINTB_ERR_ALIGNMENT;
    return (int)bfaintb::launch_pack(static_cast<uint8_t*>(dst), static_cast<const uint8_t*>(src), n, k,
                                     weight_bits == 8 ? ldb : ldb / 2u, weight_bits, unpack, static_cast<hipStream_t>(stream));
}

int bfaintb_quantize(void* b, void* scale, const void* w, int weight_type, uint32_t n, uint32_t k, uint32_t ldw, int weight_bits,
                     uint32_t group_size, void* stream)
{
    int e = check_format(k, weight_bits, group_size);
    if (e) return e;
    if (weight_type != BFAINTB_WEIGHT_BF16 && weight_type != BFAINTB_WEIGHT_F16 && weight_type != BFAINTB_WEIGHT_F32) return BFAINTB_ERR_UNSUPPORTED;
    e = check_shape(1, n, k, weight_bits);
    if (e) return e;
    if (k > (1u << 21)) return BFAINTB_ERR_BAD_SHAPE;  // (tiles and groups along k are the grid's y)
    if (ldw < k || ldw % 8u != 0) return BFAINTB_ERR_BAD_LD;
    if (n == 0) return BFAINTB_OK;
    if (b == nullptr || scale == nullptr || w == nullptr) return BFAINTB_ERR_NULL_POINTER;
    if (misaligned16(b) || misaligned16(scale) || misaligned16(w)) return BFAINTB_ERR_ALIGNMENT;
    return (int)bfaintb::launch_quantize(static_cast<uint8_t*>(b), static_cast<uint16_t*>(scale), w, weight_type, n, k, ldw, n * (uint32_t)weight_bits / 8u,
                                         weight_bits, group_size, static_cast<hipStream_t>(stream));
}

int bfaintb_prepack(void* packed, const void* b, uint32_t n, uint32_t k, uint32_t ldb, int weight_bits, void* stream)
{
    return repack(packed, b, n, k, ldb, weight_bits, stream, false);
}

int bfaintb_unpack(void* b, const void* packed, uint32_t n, uint32_t k, uint32_t ldb, int weight_bits, void* stream)
{
    return repack(b, packed, n, k, ldb, weight_bits, stream, true);
}

int bfaintb_prepack_colmajor(void* packed, const void* b, uint32_t n, uint32_t k, uint32_t ldb, int weight_bits, void* stream)
{
    if (weight_bits != 8 && weight_bits != 4) return BFAINTB_ERR_UNSUPPORTED;
    const int e = check_packed_shape(n, k, weight_bits);
    if (e) return e;
    if (ldb < k || ldb % 16u != 0) return BFAINTB_ERR_BAD_LD;  // elements between columns
    if (n == 0) return BFAINTB_OK;
    if (packed == nullptr || b == nullptr) return BFAINTB_ERR_NULL_POINTER;
    if (misaligned16(packed) || misaligned16(b)) return BFAINTB_ERR_ALIGNMENT;
    return (int)bfaintb::launch_pack_colmajor(static_cast<uint8_t*>(packed), static_cast<const uint8_t*>(b), n, k,
                                              weight_bits == 8 ? ldb : ldb / 2u, weight_bits, static_cast<hipStream_t>(stream));
}

// Packed weights, "DECODE": the slab-streaming kernel (one workgroup per 16 columns over all of k, no split, every block
// of 16 rows of A converts the slab again) or the decode family reading packed slabs (128 or 256 columns per workgroup,
// split along k).  The slab kernel wins while the rows are few; how few depends on the shape, so packed_uses_slab
// compares what each was measured to take.
static DecodePlan packed_family_plan(uint32_t m, uint32_t n, uint32_t k, int bits, bool fitted = true);

// The slab kernel against the family, by what each was measured to take: 28 weight shapes from 256 x 7168 to 28672 x 8192,
// m = 1 .. 32, both code widths; least-squares fits, 7 - 9 % rms (us).
// The slab kernel: a workgroup walks its 16 columns alone, two workgroups that share a CU at half the pace each, so a
// launch takes as many walks as the fullest CU has slabs — n / 16 over 256 CUs, rounded up (4-bit codes, 5120 x 5120,
// 320 slabs: 7.3 us, what 8192 x 5120 would take; 4096 x 4096: 3.5).  4-bit codes are bound by the CUs' vector
// arithmetic (1975 rows per us and walk); 8-bit codes by that (1544 rows per us) or by memory (6.2 TB/s).  Each
// further row of A costs 1.4 - 3.6 % of the walk up to 6 rows and 6 - 8 % from there (two blocks of 16 rows from m = 17).
// The family's 128-column form streams at about 4.4 TB/s (4-bit) or 5.6 TB/s (8-bit) with every CU busy, pays the
// split's hand-over, and hardly grows with m up to 16 rows (11 - 26 % more from 17).
// Where the two are close either choice is within a few per cent; where they are not the gap is up to 80 % (4-bit codes,
// 5120 x 13824, m = 16: slab 31.0, family 17.2; 13824 x 5120: 26.0 / 15.5; 4096 x 2048, m = 32: 5.5 / 6.9; 1024 x 16384,
// m = 1: 10.5 / 9.0.  8-bit codes, m = 8: 5120 x 13824 23.2 / 16.3; 13824 x 5120 20.2 / 15.0; 5120 x 5120 11.3 / 9.2;
// 2048 x 4096, m = 12: 5.5 / 6.9).  Picks on the scan, weights cold: 4-bit 9 of 252 more than 5 % off the faster kernel
// (worst 12 %), 8-bit 12 of 252 (worst 14 %); fixed row limits, as before: 22 of 196, up to 42 %.  With the conversion by halves both
// 4-bit kernels are 1 - 9 % faster than fitted, and the picks hold: over the 28 shapes, 10 row counts and groups of 128 or none, 16 of 560 more
// than 5 % off, 0.4 % over the faster kernel on average (worst 8192 x 28672, 1 row: slab 35.9, family 29.0).
static double packed_slab_walks(uint32_t n)
{
    const double cus = (double)machine_cus();
    const double slabs = n / 16.0;
    return slabs <= 4.0 * cus ? (double)(uint64_t)((slabs + cus - 1.0) / cus) : slabs / cus;
}
static double packed_family_fill(uint32_t m, uint32_t n, const DecodePlan& pl)
{
    const double cus = (double)machine_cus();
    const double wgs = (double)((n + pl.cols - 1u) / pl.cols) * pl.splits * ((m + 16u * pl.mb - 1u) / (16u * pl.mb));
    const double rounds = (double)(uint64_t)((wgs + cus - 1.0) / cus);
    return wgs / (rounds * cus);
}
static double packed8_slab_time_us(uint32_t m, uint32_t n, uint32_t k)
{
    const double walks = packed_slab_walks(n);
    const double rows = m <= 6u ? 1.0 + 0.0136 * (m - 1.0) : m <= 16u ? 1.068 + 0.0578 * (m - 6.0) : 0.856 + 0.0608 * m;
    // (from the third walk on a walk never takes less than 2.2 us: its start and its reduction weigh as much as 1300 rows —
    // k = 2048, m = 8 / 12: 10496 columns 10.2 us, 16384 columns 15.3, where rows alone would say 7.2 and 10.6; one or two
    // walks of a short k hide them behind the launch: 4096 x 2048 stays at 3.7 us)
    const double per_walk = (k / 1544.0 > 2.2 || walks <= 2.0) ? k / 1544.0 : 2.2;
    const double walk_us = walks * per_walk, stream_us = (double)n * k / 6.16e6;
    return 2.07 + 0.017 * m * walks + (walk_us > stream_us ? walk_us : stream_us) * rows;
}
static double packed8_family_time_us(uint32_t m, uint32_t n, uint32_t k, const DecodePlan& pl)
{
    // (a long k streams faster, the workgroups' starts and hand-overs weighing less: 6 x 15104 x 11008 28.8 us, 6 x 7168 x 14336
    // 20.6, where 5.63 TB/s would say 34.1 and 23.3)
    const double long_k = k <= 4096u ? 0.0 : k >= 12288u ? 1.0 : (k - 4096.0) / 8192.0;
    // (many splits: the hand-over, not the stream, is what narrower workgroups leave — 5 x 1456 x 6912, 14 splits, 8.7 us with eight column blocks,
    // 8.9 with six; 4 x 1296 x 6400 8.6 / 8.1, five; the slab kernel 7.7 and 7.5)
    DecodePlan at = pl;
    if (pl.splits > 8u) at.cols = 128u;
    const double stream_us = (double)n * k / 1.0e6 / (5.63 * (1.0 + 0.12 * long_k) * pow(packed_family_fill(m, n, at), 0.638));
    return 3.0 + 0.0885 * m + 0.118 * (pl.splits - 1.0) + stream_us * (1.0 - 0.0037 * m + (m > 16u ? 0.1076 : 0.0)) * (pl.cols == 256u ? 1.1 : 1.0);
}
static double packed4_slab_time_us(uint32_t m, uint32_t n, uint32_t k, bool charge_large)
{
    const double rows = m <= 6u ? 1.0 + 0.031 * (m - 1.0) : m <= 16u ? 1.155 + 0.078 * (m - 6.0) : 1.267 + 0.0776 * m;
    // (more than seven slabs per CU: 5 % less than that — 32000 / 50304 / 128256 / 151936 x 4096, m = 1: 17.6 / 26.2 / 63.4 / 74.8 us;
    // 28672 x 8192, seven, is as the formula says: 31.1)
    const double many = n / 16.0 > 7.0 * (double)machine_cus() ? 0.95 : 1.0;
    // (from the third walk on a walk never takes less than 1.45 us, as for 8-bit codes: k = 2048, 12 x 10240 9.6 us, 8 x 9984 8.3)
    const double walks = packed_slab_walks(n);
    const double per_walk = (k / 1975.0 > 1.45 || walks <= 2.0) ? k / 1975.0 : 1.45;
    // (more than 96 Mi weights: 10 % more on average over 310 shapes, and up to 25 % — 24272 x 9216, m = 1: 35.6 us, 31392 x 8960, m = 3: 43.6)
    const double large = charge_large && (uint64_t)n * k > (96ull << 20) ? 1.1 : 1.0;
    return 2.58 + many * large * walks * per_walk * rows;
}
static double packed4_family_time_us(uint32_t m, uint32_t n, uint32_t k, const DecodePlan& pl)
{
    // (more than one round of workgroups: 8 % more than the fill says — 50304 / 128256 / 151936 x 4096, m = 1: 35.6 / 71.6 / 86.8 us,
    // m = 16: 37.4 / 75.4 / 91.5)
    const double wgs = (double)((n + pl.cols - 1u) / pl.cols) * pl.splits * ((m + 16u * pl.mb - 1u) / (16u * pl.mb));
    const double stream_us = (double)n * k / 2.0e6 / (4.37 * pow(packed_family_fill(m, n, pl), 0.58)) * (wgs > (double)machine_cus() ? 1.08 : 1.0);
    // (narrower workgroups on few weights: what they gain is the stream's, not the start's — 1 x 9296 x 1408 6.4, the slab kernel 6.0; 2 x 10576 x 1408
    // 7.1 / 6.3; 21 x 3584 x 4224 9.9 / 8.7)
    const double few = pl.cols < 128u && (uint64_t)n * k < (24ull << 20) ? 1.08 : 1.0;
    return 4.71 + 0.067 * m + 0.144 * (pl.splits - 1.0) + few * stream_us * (1.0 + 0.0003 * m + (m > 16u ? 0.258 : 0.0));
}
static bool packed_slab_leads(uint32_t m, uint32_t n, uint32_t k, int bits, const DecodePlan& pl, bool large)
{
    if (m > kDecodeAutoMaxM) return false;
    if (bits == 8) return packed8_slab_time_us(m, n, k) <= packed8_family_time_us(m, n, k, pl);
    if (pl.cols > 128u) return m <= 8u;
    return packed4_slab_time_us(m, n, k, large) <= packed4_family_time_us(m, n, k, pl);
}
// Whether the slab kernel leads the family with eight column blocks: what the choice was before there were fewer.  Such a call has no scratch to
// ask for and may be a first one under capture, and stays one.
static bool packed_slab_leads_eight_blocks(uint32_t m, uint32_t n, uint32_t k, int bits)
{
    return packed_slab_leads(m, n, k, bits, packed_family_plan(m, n, k, bits, false), false);
}
static bool packed_uses_slab(uint32_t m, uint32_t n, uint32_t k, int bits)
{
    if (m > kDecodeAutoMaxM) return false;
    const DecodePlan pl = packed_family_plan(m, n, k, bits);
    return packed_slab_leads(m, n, k, bits, pl, true) || (pl.splits > 1u && packed_slab_leads_eight_blocks(m, n, k, bits));
}

// Columns of a workgroup over packed weights, by whole column blocks of 16: eight, or as few as make the launch shorter by the fullest CU's share,
// rounds of workgroups times columns.  A workgroup has one CU's LDS and waves to itself while it runs, and eight blocks fill the CUs where
// n / 128 times the splits happens to be 256 or a little less (us, eight blocks / the rule's, 16 rows: 22016 x 4096 4-bit g128 18.8 / 16.5, six;
// 8-bit 20.3 / 17.5, six; 11008 x 4096 4-bit 11.5 / 10.3, six; 28672 x 8192 4-bit 31.6 / 29.2, seven; more
// than a round of eight: 34560 x 7936 4-bit, 4 rows, 53.7 / 36.2, five).  Over 3900 random shapes of 1 to 32 rows the family is faster by 15 % where it takes
// five blocks, 11 % six, 3 % seven; against the best of the four at each shape the rule is 0.5 % off.
// Two limits have no measurement behind them: seven only unsplit and from 13 rows, and eight for a split of more than 128 Mi weights.  The plan query's
// answers for 12 x 28672 x 8192 and 16 x 12288 x 12288 packed 4-bit are fixed (tests/test_capi_cpu.py), although fewer blocks would take 3 %
// and 8 to 15 % less there.  Within them seven serve little beside 24592 to 28672 unsplit columns at 13 to 32 rows: up to 7 % (28672 x 8192).
// (k up to 1024, which is over before its workgroups have filled: 13 x 16336 x 1024 8-bit 7.5 with eight, 8.1 with five; and more than 12 splits, where the
// hand-over is most of it: 8 x 1024 x 15872 4-bit 9.9 / 10.7.)
// (More than 32 rows take their row blocks again for every workgroup: not looked at.)
static DecodePlan fitted_to_cus(DecodePlan pl, uint32_t m, uint32_t n, uint32_t k)
{
    if (m > kDecodeAutoMaxM || pl.mb > 2u || pl.waves != 8u || (pl.splits > 1u && (uint64_t)n * k > (128ull << 20)) || k <= 1024u || pl.splits > 12u) return pl;
    const uint64_t blocks = n / 16u, others = (uint64_t)pl.splits * ((m + 16u * pl.mb - 1u) / (16u * pl.mb)), cus = machine_cus();
    auto share = [&](uint32_t c) { return ((blocks + c - 1u) / c * others + cus - 1u) / cus * c; };
    // (a tenth less at least: three rounds of five blocks are no better than two of eight — 59680 x 1024 4-bit, 6 rows, 14.6 / 13.2)
    uint64_t least = share(8u) * 9u / 10u + 1u;
    for (uint32_t c = 7u; c >= 5u; --c) {
        if (share(c) >= least || (c == 7u && (m <= 12u || pl.splits > 1u))) continue;
        least = share(c), pl.cols = 16u * c;
    }
    return pl;
}

// The family's plan over packed weights.  8-bit codes: the one row-major weights get, as long as it uses the 128 columns
// per workgroup the packed kernels are built for.  4-bit codes: the row-block plan also below 33 rows of A (measured
// against the small-m plan: 8192 x 8192, m = 32: 28.9 / 36.4 us; 28672 x 8192, m = 24: 56.9 / 65.6 us).
static DecodePlan packed_family_plan(uint32_t m, uint32_t n, uint32_t k, int bits, bool fitted)
{
    if (bits == 8) {
        const DecodePlan pl = decode_plan(m, n, k, bits, 0, true);
        if (pl.cols == 128u) return fitted ? fitted_to_cus(pl, m, n, k) : pl;
    }
    // 4-bit codes: the 128-column form (8 column blocks of 16 per workgroup, 8 waves) with the launch shape 8-bit codes
    // would get, wherever that shape has 128 columns.  Against the 256-column form, whose kernels over packed 4-bit codes
    // run 4 waves (us, 128 / 256 columns): 1024 x 8192, m = 64 / 128: 8.9 / 18.3, 11.4 / 17.5; 4096 x 4096: 10.6 / 15.7,
    // 14.9 / 20.7; 8192 x 8192, m = 16 / 32: 15.5 / 19.9, 18.3 / 24.1; 28672 x 8192, m = 12 / 32 / 48: 37.0 / 49.4, 42.3 / 47.1,
    // 52.0 / 70.6; 8192 x 28672: 37.0 / 41.4, 43.9 / 50.3, 52.8 / 68.5; 8192 x 11008, m = 16 / 64: 19.0 / 23.9, 30.5 / 36.2; the
    // other way round at most 6 % (16384 x 8192, m = 12: 29.5 / 27.8; 32000 x 4096: 27.6 / 26.3).
    if (bits == 4) {
        const DecodePlan pl = decode_plan(m, n, k, 8, 0, true, true);
        if (pl.cols == 128u) return fitted ? fitted_to_cus(pl, m, n, k) : pl;
    }
    return decode_plan_row_blocks(m, n, k, bits, 0, true);
}

// The family's estimate against the tiles', over packed weights, corrected as decode_family_time_us corrects it for
// row-major weights, with what a scan of 11 weight shapes x 12 values of m (40 .. 2048) x both code widths fits.  8-bit
// codes: the family's kernels over packed weights run at 0.72 (row blocks up to 32 rows) to 0.78 (64 rows) of the
// estimate's stream and arithmetic, and the hand-over costs 0.35 and 0.7 of its term; the factors in use (0.76, 0.84)
// sit a little above that, where the pick on the scan's shapes is best.  4-bit codes: the family measures 0.69 - 0.84 of
// the whole estimate (their packed kernels have no 8-wave form) and the tiles over packed 4-bit codes 0.82 - 0.98 of
// theirs; 0.84 against the tiles' estimate as it stands picks best (2 of 116 shapes more than 3 % off, worst 9 %;
// 8-bit: 3 of 128, worst 15 % at 40 x 11008 x 4096).  Up to 64 rows the family used to be the rule, as it once was
// for row-major weights: 4-bit codes against 11008 and 28672 columns then ran 22 - 39 % over the tiles' time.
static double packed_family_time_us(uint32_t m, uint32_t n, uint32_t k, int bits, const DecodePlan& pl)
{
    FamilyEstimate e;
    const double ranked = decode_family_estimate_us(m, n, k, bits, pl, &e) - e.serial;
    // Beyond 256 rows, unsplit, more than two rounds of workgroups (five row blocks and more against very many columns):
    // all the estimate says (us, family / tiles: 320 x 44032 x 2048 8-bit 132 / 87; 384 x 37120 x 2048 4-bit 132 / 76).  With
    // fewer workgroups than that the factors below stand: 640 x 1024 x 2048 12.3 / 16.3.
    if (m > 256u && pl.splits == 1u) {
        const double wgs_ = (double)((n + pl.cols - 1u) / pl.cols) * (double)((m + 16u * pl.mb - 1u) / (16u * pl.mb));
        if (wgs_ > 2.0 * (double)machine_cus()) return 5.0 + e.core;
    }
    if (bits == 4) return (pl.cols <= 128u ? 0.70 : 0.84) * ranked;  // (the 128-column form measures 0.52 - 0.79 of its estimate)
    // (a row block that is not full costs less: 64-row blocks at m = 40 / 48 / 64 measure 0.87 / 0.91 / 1.0 of the tiles' time
    // over 11 weight shapes where the estimate had them level — the rows past m are neither converted for nor multiplied)
    const double block_rows = 16.0 * pl.mb;
    const double fill = m < block_rows ? m / block_rows : 1.0;  // (with more blocks than one the estimate is right as it stands: 96 x 8192 x 8192)
    // (and a round of workgroups that leaves CUs idle slows the stream less than in proportion: 172 and 192 workgroups of 64
    // rows x 128 columns run at 0.80 and 0.85 of the pace of 256, not 0.67 and 0.75 — 11008 x 8192, 22016 x 4096, 12288 x 12288)
    const double wgs = (double)((n + pl.cols - 1u) / pl.cols) * pl.splits * (double)(uint64_t)((m + block_rows - 1.0) / block_rows);
    const double cus = (double)machine_cus();
    const double idle = wgs < cus ? pow(wgs / cus, 0.45) : 1.0;
    // (a single block, since its kernels start each workgroup's walk over k at a step of its own: 0.92 of that — at 64 rows
    // the family leads the tiles by 5 - 8 % on 11008 x 8192, 28672 x 8192, 32000 x 4096, 14336 x 8192, 12288 x 12288)
    const double base = m <= block_rows ? 0.57 : 0.65;
    return (pl.mb == 4u ? 0.84 : 0.76) * (base + 0.35 * fill) * (5.0 + e.core * idle + (pl.mb == 4u ? 0.7 : 0.35) * e.partial);
}
// Which kernel multiplies by packed weights: the decode kernels (the slab-streaming one while packed_uses_slab, the
// row-blocked family without a split along k beyond) or the tiled kernel, by the estimates that choose for row-major weights.
static int packed_variant(uint32_t m, uint32_t n, uint32_t k, int bits, int variant, bool second_launch = true)
{
    if (variant == BFAINTB_VARIANT_DECODE) return m <= kDecodeMaxM ? variant : BFAINTB_ERR_BAD_VARIANT;
    if (is_prefill(variant)) return variant;
    if (variant != BFAINTB_VARIANT_AUTO) return BFAINTB_ERR_BAD_VARIANT;
    if (packed_uses_slab(m, n, k, bits) || m <= kDecodeAutoMaxM) return BFAINTB_VARIANT_DECODE;
    if (m > kDecodeFamilyAutoMaxM || wide_tiles_run(m, n, k, bits, second_launch)) return BFAINTB_VARIANT_PREFILL;
    const DecodePlan pl = packed_family_plan(m, n, k, bits);
    return family_leads_tiles(packed_family_time_us(m, n, k, bits, pl), m, n, k, bits, true, second_launch) ? BFAINTB_VARIANT_DECODE : BFAINTB_VARIANT_PREFILL;
}

int bfaintb_gemm_prepacked_variant(uint32_t m, uint32_t n, uint32_t k, int weight_bits, uint32_t group_size)
{
    int e = check_format(k, weight_bits, group_size);
    if (e) return e;
    e = check_shape(m, n, k);
    if (e) return e;
    e = check_packed_shape(n, k, weight_bits);
    if (e) return e;
    return packed_variant(m, n, k, weight_bits, BFAINTB_VARIANT_AUTO);
}

// Scratch of the packed path: the decode family (where the slab kernel is not used) and the small tiles split along k.
static size_t packed_workspace_need(uint32_t m, uint32_t n, uint32_t k, int bits, int v, bool second_launch = true)
{
    if (m == 0 || n == 0) return 0;
    if (is_prefill(v)) return tiled_may_split(v, m, n, k, bits) ? tile_workspace_bytes(tile128_plan(m, n, k, bits, 0, second_launch), m, n) : 0;
    if (v != BFAINTB_VARIANT_DECODE || packed_uses_slab(m, n, k, bits)) return 0;
    const DecodePlan pl = packed_family_plan(m, n, k, bits);
    if (pl.splits <= 1) return 0;
    return bfaintb::kWorkspaceHeaderBytes + ((((size_t)(pl.splits - 1u) * m * n * sizeof(float)) + 255u) & ~(size_t)255u);
}

// ---- A product in two launches, by rows of A.  The tiled kernels take the time of whole rounds of tiles: a few rows more than
//      fill one cost up to a round.  Where the times below say so, the rows that fill their tiles go first and the rest is a
//      product of its own, by whatever kernel suits it (packed weights, us, one launch / two: 528 x 22016 x 4096 4-bit, 258 large
//      tiles, 162 / 114; 577 rows 164 / 127; 1040 x 13824 x 5120 4-bit 203 / 141; 784 x 5120 x 13824 4-bit 186 / 126; 640 x 28672 x
//      8192 4-bit 313 / 253; 1040 x 4096 x 4096 8-bit 57 / 44; 2176 x 8192 x 8192 8-bit 294 / 230).

// What one launch of the library's own choice takes, in microseconds, for more rows than the estimates that choose between
// kernels are asked about: the large tiles by their number (a round at a load below one CU each runs at a higher clock; us per
// K-step at 162 / 216 / 256 tiles, 4-bit 1.39 / 1.49 / 1.55, 8-bit, at 172 / 256, 1.26 / 1.52), the thin last round as the half tiles
// it runs as; up to 32 rows the stream of the weights.
// (17 to 32 rows on tiles: by the tiles' estimate, 0.88 - 1.07 of the measured time by kind of weights, 9 % rms over 340 shapes; the stream at
// this rate would be 1.15 (4-bit) to 1.69 (8-bit) times it.  For rows of B that lie n codes apart, as the scratch is asked for.)
static double launch_time_us(uint32_t m, uint32_t n, uint32_t k, int bits, bool packed, bool grouped)
{
    if (few_rows_on_tiles(m, n, k, bits, grouped, packed, n)) return tile128_plan(m, n, k, bits, 1).us;
    if (m <= kDecodeAutoMaxM) return 6.0 + (double)n * k * bits / 8.0 / 3.3e6 * (m <= 16u ? 1.0 : 1.25);
    const WideTiles wide = wide_tiles(m, n, k, bits);
    if (wide.blocks != 0u) return wide.us;
    if (m <= kDecodeFamilyAutoMaxM) {  // (beyond 32 rows the library's own choice asks just this)
        const DecodePlan pl = packed ? packed_family_plan(m, n, k, bits) : decode_plan(m, n, k, bits, 0);
        const double family = packed ? packed_family_time_us(m, n, k, bits, pl) : decode_family_time_us(m, n, k, bits, pl);
        if (family_leads_tiles(family, m, n, k, bits, packed, true)) {
            // (a short k: the start of a round of workgroups, 5.2 to 6.6 us at k = 128 to 640, which the estimate leaves out)
            const double rounds = (double)((n + pl.cols - 1u) / pl.cols) * pl.splits * ((m + 16u * pl.mb - 1u) / (16u * pl.mb)) / machine_cus();
            const double starts = k <= 1024u && rounds > 1.0 ? 6.0 * (rounds - 1.0) : 0.0;
            return starts + (prefill_small_tiles(m, n, k, bits) ? family_beside_tiles_us(family, m, n, bits, packed) : family);
        }
    }
    // (tall tiles of one chain are estimated 4.9 us short, which the choice against the family is fitted with and which does not matter there; next to
    // tiles of 256 columns at what they take it would send products with a short k to two launches: 50 shapes of k = 128 to 1792, 4.4 to 5.5 on nearly all)
    if (prefill_tall_tiles(m, n, k, bits)) return prefill_estimate_us(m, n, k, bits) + (tall_tiles_in_one_chain(m, k) ? 4.9 : 0.0);
    if (prefill_small_tiles(m, n, k, bits)) return prefill_estimate_us(m, n, k, bits);
    return square_tiles_us(m, n, k, bits);
}

static size_t row_split_workspace(uint32_t head, uint32_t rest, uint32_t n, uint32_t k, int bits, bool packed)
{
    size_t need = 0;
    for (const uint32_t rows : {head, rest}) {
        const size_t part = packed ? packed_workspace_need(rows, n, k, bits, packed_variant(rows, n, k, bits, BFAINTB_VARIANT_AUTO))
                                   : workspace_need(rows, n, k, bits, resolve_variant(rows, n, k, bits, BFAINTB_VARIANT_AUTO), 0);
        if (part > need) need = part;
    }
    return need;
}

// Rows of the first launch, or 0 for one launch over all of them.
static uint32_t row_split_rule(uint32_t m, uint32_t n, uint32_t k, int bits, bool packed, bool grouped)
{
    if (m <= 256u || n < 16u || g_force_row_block.load(std::memory_order_relaxed) != 0u) return 0;
    const uint64_t cus = machine_cus();
    const uint32_t cols256 = (n + 255u) / 256u, cols128 = (n + 127u) / 128u;
    // the rows that whole rounds of large tiles hold; one round of tall tiles; one of small ones; and all whole large tiles, or
    // all but one row of them
    const uint64_t rounds = (uint64_t)((m + 255u) / 256u) * cols256 / cus;
    const uint64_t candidates[] = {rounds * cus / cols256 * 256u, cus / cols128 * 256u, cus / cols128 * 128u, (m - 1u) / 256u * 256u,
                                   (m - 1u) / 256u * 256u - 256u};
    const double one = launch_time_us(m, n, k, bits, packed, grouped);
    // (0.94: the estimates' error.  Of 200 shapes, m = 257 .. 4096, 25 go in two launches so, 1.25 times
    // as fast on average and none slower; at 0.97 three of 49 are, by 4 - 9 %)
    // (0.985 where the one launch is of tiles of 256 columns and as many rows as suit it, whose estimate is nearer)
    const bool wide = m > kDecodeFamilyAutoMaxM || (packed ? packed_variant(m, n, k, bits, BFAINTB_VARIANT_AUTO) : resolve_variant(m, n, k, bits, BFAINTB_VARIANT_AUTO)) == BFAINTB_VARIANT_PREFILL;
    double best = (wide && wide_tiles(m, n, k, bits).blocks != 0u ? 0.985 : 0.94) * one;
    uint32_t head = 0;
    for (size_t i = 0; i < sizeof(candidates) / sizeof(candidates[0]); ++i) {
        const uint64_t c = candidates[i];
        if (c == 0u || c >= m) continue;
        bool asked = false;
        for (size_t j = 0; j < i; ++j) asked = asked || candidates[j] == c;
        if (asked) continue;
        const uint32_t rows = (uint32_t)c;
        // (no launch is estimated at less than 2 us: most candidates need no look at their rest)
        const double first = launch_time_us(rows, n, k, bits, packed, grouped) + 1.0;
        if (first + 2.0 >= best) continue;
        const double two = first + launch_time_us(m - rows, n, k, bits, packed, grouped);
        if (two >= best) continue;
        if (row_split_workspace(rows, m - rows, n, k, bits, packed) > BFAINTB_STATIC_SCRATCH_BYTES) continue;
        best = two;
        head = rows;
    }
    return head;
}

// (a call asks two or three times, for its scratch and for its launch, and a model asks about the same few shapes: each
// thread keeps the last answers, one per slot of a hash of the question.  A new question costs 1.5 - 3.2 us of host time; a known one
// 0.07 where tiles of 256 columns run, 0.2 otherwise, and 0.7 - 1 if the answer is two launches.  A prompt of a new length asks once per
// shape of its layers, as long as no two of them share a slot)
static uint32_t row_split_head(uint32_t m, uint32_t n, uint32_t k, int bits, bool packed, bool grouped)
{
    if (m <= 256u) return 0;
    struct Answer {
        uint32_t m, n, k, kind, cus, row_block, head;
    };
    static thread_local Answer answers[256] = {};
    const uint32_t kind = (uint32_t)bits * 4u + (packed ? 2u : 0u) + (grouped ? 1u : 0u), cus = machine_cus(), row_block = g_force_row_block.load(std::memory_order_relaxed);
    Answer& a = answers[((m * 2654435761u) ^ (n * 2246822519u) ^ (k * 3266489917u) ^ kind) >> 24];
    if (a.m != m || a.n != n || a.k != k || a.kind != kind || a.cus != cus || a.row_block != row_block)
        a = Answer{m, n, k, kind, cus, row_block, row_split_rule(m, n, k, bits, packed, grouped)};
    return a.head;
}

size_t bfaintb_gemm_prepacked_workspace_bytes_ex(uint32_t m, uint32_t n, uint32_t k, int weight_bits, uint32_t group_size, int variant)
{
    if (check_format(k, weight_bits, group_size) || check_shape(m, n, k) || check_packed_shape(n, k, weight_bits)) return 0;
    const int v = packed_variant(m, n, k, weight_bits, variant);
    if (v < 0) return 0;
    if (variant == BFAINTB_VARIANT_AUTO) {
        const uint32_t head = row_split_head(m, n, k, weight_bits, true, group_size != 0);
        if (head != 0u) return row_split_workspace(head, m - head, n, k, weight_bits, true);
    }
    return packed_workspace_need(m, n, k, weight_bits, v);
}

size_t bfaintb_gemm_prepacked_workspace_bytes(uint32_t m, uint32_t n, uint32_t k, int weight_bits, uint32_t group_size)
{
    return bfaintb_gemm_prepacked_workspace_bytes_ex(m, n, k, weight_bits, group_size, BFAINTB_VARIANT_AUTO);
}

static int gemm_prepacked_impl(void* c, const void* a, const void* packed_b, const void* scale, const Epilogue& ep, uint32_t m,
                               uint32_t n, uint32_t k, uint32_t lda, uint32_t ldc, int weight_bits, uint32_t group_size,
                               void* workspace, size_t workspace_bytes, void* stream, int variant, bool whole = false, bool second_launch = true)
{
    const void* bias = ep.bias;
    int e = check_format(k, weight_bits, group_size);
    if (e) return e;
    e = check_shape(m, n, k);
    if (e) return e;
    e = check_packed_shape(n, k, weight_bits);
    if (e) return e;
    if (lda < k || ldc < ep.out_cols(n) || lda % 8u != 0 || ldc % 8u != 0) return BFAINTB_ERR_BAD_LD;
    const int v = packed_variant(m, n, k, weight_bits, variant, second_launch);
    if (v < 0) return v;
    if (m == 0 || n == 0) return BFAINTB_OK;
    if (c == nullptr || a == nullptr || packed_b == nullptr || scale == nullptr) return BFAINTB_ERR_NULL_POINTER;
    if (misaligned16(c) || misaligned16(a) || misaligned16(packed_b) || misaligned16(scale) || misaligned16(bias) ||
        misaligned16(ep.residual))
        return BFAINTB_ERR_ALIGNMENT;
    if (!whole && variant == BFAINTB_VARIANT_AUTO) {
        const uint32_t head = row_split_head(m, n, k, weight_bits, true, group_size != 0);
        if (head != 0u && row_split_served(workspace, workspace_bytes, row_split_workspace(head, m - head, n, k, weight_bits, true), false,
                                           static_cast<hipStream_t>(stream))) {
            e = gemm_prepacked_impl(c, a, packed_b, scale, ep, head, n, k, lda, ldc, weight_bits, group_size, workspace, workspace_bytes, stream, variant,
                                    true);
            if (e) return e;
            return gemm_prepacked_impl(static_cast<uint16_t*>(c) + (size_t)head * ldc, static_cast<const uint16_t*>(a) + (size_t)head * lda, packed_b,
                                       scale, ep.from_row(head), m - head, n, k, lda, ldc, weight_bits, group_size, workspace, workspace_bytes, stream,
                                       variant, true);
        }
    }
    GemmParams p{};
    p.residual = static_cast<const uint16_t*>(ep.residual);
    p.ldr = ep.ldr;
    p.activation = ep.activation;
    p.c = static_cast<uint16_t*>(c);
    p.a = static_cast<const uint16_t*>(a);
    p.b = static_cast<const uint8_t*>(packed_b);
    p.scale = static_cast<const uint16_t*>(scale);
    p.bias = static_cast<const uint16_t*>(bias);
    p.m = m; p.n = n; p.k = k;
    p.lda = lda;
    p.ldc = ldc;
    p.lds = n;
    p.group_size = group_size;
    bfaintb::set_group_division(p);
    p.cus = machine_cus();
    hipStream_t st = static_cast<hipStream_t>(stream);
    auto attach = [&] { return attach_workspace(p, workspace, workspace_bytes, packed_workspace_need(m, n, k, weight_bits, v, second_launch)); };
    auto without_second_launch = [&] {  // (as in gemm_impl)
        return gemm_prepacked_impl(c, a, packed_b, scale, ep, m, n, k, lda, ldc, weight_bits, group_size, workspace, workspace_bytes, stream, variant, true, false);
    };
    if (is_prefill(v)) {
        // a tile's 16 column blocks and a 256-row panel of A are addressed through 32-bit buffer extents
        if ((uint64_t)k * 256u * (uint32_t)weight_bits / 8u >= (1ull << 31) || (uint64_t)256 * lda * 2u >= (1ull << 31))
            return BFAINTB_ERR_BAD_SHAPE;
        if (tiled_may_split(v, m, n, k, weight_bits) && bfaintb::prefill128_wreg_serves(p)) {
            // small tiles: the kernel that keeps the weights in registers, with the plan (split along k included) and the
            // workspace protocol of the row-major path
            const TilePlan tp = tile128_plan(m, n, k, weight_bits, 0, second_launch);
            p.k_per_wg = tp.k_per_wg;
            p.splits = tp.splits;
            p.tile_blocks = tp.blocks;
            p.finish_launch = tp.finish_launch;
            std::unique_lock<std::mutex> in_order;
            if (p.splits > 1) {
                e = attach();
                if (e) return second_launch ? without_second_launch() : e;
                in_order = std::unique_lock<std::mutex>(workspace_order(p.ws_header));
            }
            return (int)bfaintb::launch_prefill128_wreg(p, weight_bits, true, st);
        }
        if (v == BFAINTB_VARIANT_PREFILL) {
            p.tile_blocks = wide_tiles(m, n, k, weight_bits).blocks;
            if (p.tile_blocks != 0u) return (int)bfaintb::launch_prefill_packed(p, weight_bits, st, true);
        }
        if (v == BFAINTB_VARIANT_PREFILL_256X128 || (v == BFAINTB_VARIANT_PREFILL && prefill_tall_tiles(m, n, k, weight_bits))) {
            p.k_per_wg = k;
            p.splits = 1;
            if (v == BFAINTB_VARIANT_PREFILL && !tall_tiles_in_one_chain(m, k)) {
                p.tile_blocks = tall_tile_blocks(m);
                return (int)bfaintb::launch_prefill128_wreg(p, weight_bits, true, st);
            }
            return (int)bfaintb::launch_prefill256x128_wreg(p, weight_bits, true, st);
        }
        if (use_small_tiles(v, m, n, k, weight_bits)) return (int)bfaintb::launch_prefill128(p, weight_bits, true, st);
        return (int)bfaintb::launch_prefill_packed(p, weight_bits, st, v != BFAINTB_VARIANT_PREFILL_256_LDS);
    }
    if (!packed_uses_slab(m, n, k, weight_bits)) {
        // beyond a few dozen rows the row-blocked decode family (A reused across 128 or 256 columns) reads the packed
        // slabs: measured at n = k = 4096 and m = 64, 128, 256: 16, 20, 22 us against 18, 34, 63 us for the slab kernel.
        // Same plan as for row-major weights, split along k and workspace protocol included.
        if (m > kDecodeMaxM) return BFAINTB_ERR_BAD_VARIANT;
        const DecodePlan pl = packed_family_plan(m, n, k, weight_bits);
        p.k_per_wg = pl.k_per_wg;
        p.splits = pl.splits;
        p.decode_waves = pl.waves;
        p.decode_cols = pl.cols;
        p.decode_mb = pl.mb;
        if (p.splits > 1) {
            e = attach();
            if (e) return second_launch ? without_second_launch() : e;
        }
        DeviceState* dev = nullptr;
        e = device_state(st, &dev);
        if (e) return packed_slab_leads_eight_blocks(m, n, k, weight_bits) ? (int)bfaintb::launch_decode_packed(p, weight_bits, st) : e;
        if (variant == BFAINTB_VARIANT_AUTO && few_rows_on_tiles(m, n, k, weight_bits, group_size != 0, true, n) && (uint64_t)256 * lda * 2u < (1ull << 31))
            return (int)launch_few_rows_on_tiles(p, weight_bits, true, st);
        std::unique_lock<std::mutex> in_order;
        if (p.splits > 1) in_order = std::unique_lock<std::mutex>(workspace_order(p.ws_header));
        return (int)bfaintb::launch_decode_family_packed(p, weight_bits, st);
    }
    return (int)bfaintb::launch_decode_packed(p, weight_bits, st);
}

int bfaintb_gemm_prepacked_ex(void* c, const void* a, const void* packed_b, const void* scale, const void* bias, uint32_t m,
                              uint32_t n, uint32_t k, uint32_t lda, uint32_t ldc, int weight_bits, uint32_t group_size,
                              void* workspace, size_t workspace_bytes, void* stream, int variant)
{
    Epilogue ep;
    ep.bias = bias;
    return gemm_prepacked_impl(c, a, packed_b, scale, ep, m, n, k, lda, ldc, weight_bits, group_size, workspace, workspace_bytes,
                               stream, variant);
}

int bfaintb_gemm_prepacked_fused(void* c, const void* a, const void* packed_b, const void* scale, const bfaintb_epilogue* epilogue,
                                 uint32_t m, uint32_t n, uint32_t k, uint32_t lda, uint32_t ldc, int weight_bits, uint32_t group_size,
                                 void* workspace, size_t workspace_bytes, void* stream)
{
    Epilogue ep;
    const int e = read_epilogue(ep, epilogue, n);
    if (e) return e;
    return gemm_prepacked_impl(c, a, packed_b, scale, ep, m, n, k, lda, ldc, weight_bits, group_size, workspace, workspace_bytes,
                               stream, BFAINTB_VARIANT_AUTO);
}

int bfaintb_gemm_prepacked(void* c, const void* a, const void* packed_b, const void* scale, const void* bias, uint32_t m, uint32_t n,
                           uint32_t k, uint32_t lda, uint32_t ldc, int weight_bits, uint32_t group_size, void* workspace,
                           size_t workspace_bytes, void* stream)
{
    return bfaintb_gemm_prepacked_ex(c, a, packed_b, scale, bias, m, n, k, lda, ldc, weight_bits, group_size, workspace,
                                     workspace_bytes, stream, BFAINTB_VARIANT_AUTO);
}

int bfaintb_gemm_ex(void* c, const void* a, const void* b, const void* scale, uint32_t m, uint32_t n, uint32_t k,
                    uint32_t lda, uint32_t ldb, uint32_t ldc, int weight_bits, uint32_t group_size, void* workspace,
                    size_t workspace_bytes, void* stream, int variant, uint32_t split_k)
{
    return gemm_impl(c, a, b, scale, Epilogue{}, m, n, k, lda, ldb, ldc, weight_bits, group_size, workspace, workspace_bytes, stream,
                     variant, split_k);
}

int bfaintb_gemm_bias(void* c, const void* a, const void* b, const void* scale, const void* bias, uint32_t m, uint32_t n,
                      uint32_t k, uint32_t lda, uint32_t ldb, uint32_t ldc, int weight_bits, uint32_t group_size, void* workspace,
                      size_t workspace_bytes, void* stream)
{
    Epilogue ep;
    ep.bias = bias;
    return gemm_impl(c, a, b, scale, ep, m, n, k, lda, ldb, ldc, weight_bits, group_size, workspace, workspace_bytes, stream,
                     BFAINTB_VARIANT_AUTO, 0);
}

int bfaintb_gemm_fused(void* c, const void* a, const void* b, const void* scale, const bfaintb_epilogue* epilogue, uint32_t m,
                       uint32_t n, uint32_t k, uint32_t lda, uint32_t ldb, uint32_t ldc, int weight_bits, uint32_t group_size,
                       void* workspace, size_t workspace_bytes, void* stream)
{
    Epilogue ep;
    const int e = read_epilogue(ep, epilogue, n);
    if (e) return e;
    return gemm_impl(c, a, b, scale, ep, m, n, k, lda, ldb, ldc, weight_bits, group_size, workspace, workspace_bytes, stream,
                     BFAINTB_VARIANT_AUTO, 0);
}

int bfaintb_gemm_reference_ex(void* c, const void* a, const void* b, const float* scale, uint32_t m, uint32_t n, uint32_t k, uint32_t lda,
                              uint32_t ldb, uint32_t ldc, void* workspace, size_t workspace_bytes, void* stream, int variant, uint32_t split_k)
{
    Epilogue ep;
    ep.reference_arith = true;
    return gemm_impl(c, a, b, scale, ep, m, n, k, lda, ldb, ldc, 8, 0, workspace, workspace_bytes, stream, variant, split_k);
}

int bfaintb_gemm_reference(void* c, const void* a, const void* b, const float* scale, uint32_t m, uint32_t n, uint32_t k, uint32_t lda,
                           uint32_t ldb, uint32_t ldc, void* workspace, size_t workspace_bytes, void* stream)
{
    return bfaintb_gemm_reference_ex(c, a, b, scale, m, n, k, lda, ldb, ldc, workspace, workspace_bytes, stream, BFAINTB_VARIANT_AUTO, 0);
}

int bfaintb_gemm(void* c, const void* a, const void* b, const void* scale, uint32_t m, uint32_t n, uint32_t k,
                 uint32_t lda, uint32_t ldb, uint32_t ldc, int weight_bits, uint32_t group_size, void* workspace,
                 size_t workspace_bytes, void* stream)
{
    return bfaintb_gemm_ex(c, a, b, scale, m, n, k, lda, ldb, ldc, weight_bits, group_size, workspace, workspace_bytes,
                           stream, BFAINTB_VARIANT_AUTO, 0);
}

int bfaintb_gemm_static(void* c, const void* a, const void* b, const void* scale, uint32_t m, uint32_t n, uint32_t k, uint32_t lda,
                        uint32_t ldb, uint32_t ldc, int weight_bits, uint32_t group_size, void* stream)
{
    return gemm_impl(c, a, b, scale, Epilogue{}, m, n, k, lda, ldb, ldc, weight_bits, group_size, nullptr, 0, stream, BFAINTB_VARIANT_AUTO,
                     0, true);
}

size_t bfaintb_gemm_static_scratch_bytes(void) { return BFAINTB_STATIC_SCRATCH_BYTES; }

int bfaintb_dequant(void* w, const void* b, const void* scale, uint32_t n, uint32_t k, uint32_t ldb, uint32_t ldw,
                    int weight_bits, uint32_t group_size, void* stream)
{
    int e = check_format(k, weight_bits, group_size);
    if (e) return e;
    if (k == 0 || n % (weight_bits == 4 ? 16u : 8u) != 0 || k % 2u != 0) return BFAINTB_ERR_BAD_SHAPE;
    if (ldb < n || ldw < n || ldb % 16u != 0 || ldw % 8u != 0) return BFAINTB_ERR_BAD_LD;
    if (n == 0) return BFAINTB_OK;
    if (w == nullptr || b == nullptr || scale == nullptr) return BFAINTB_ERR_NULL_POINTER;
    if (misaligned16(w) || misaligned16(b) || misaligned16(scale)) return BFAINTB_ERR_ALIGNMENT;
    return (int)bfaintb::launch_dequant(static_cast<uint16_t*>(w), static_cast<const uint8_t*>(b),
                                        static_cast<const uint16_t*>(scale), n, k, weight_bits == 8 ? ldb : ldb / 2u, ldw,
                                        weight_bits, group_size, static_cast<hipStream_t>(stream));
}

int bfaintb_probe_read(const void* src, size_t bytes, void* sink, void* stream)
{
    if (bytes == 0) return BFAINTB_OK;
    if (src == nullptr) return BFAINTB_ERR_NULL_POINTER;
    if (misaligned16(src)) return BFAINTB_ERR_ALIGNMENT;
    if (bytes / 16 / 512 / 4 >= (1ull << 31)) return BFAINTB_ERR_BAD_SHAPE;
    return (int)bfaintb::launch_probe_read(src, bytes, sink, static_cast<hipStream_t>(stream));
}

// One launch of a checked question's answer (two where a kernel's own last round or hand-over is one): see bfaintb_gemm_plan.
static int plan_whole(uint32_t m, uint32_t n, uint32_t k, int weight_bits, uint32_t group_size, int packed, int variant, uint32_t split_k,
                      bfaintb_plan* out)
{
    memset(out, 0, sizeof(*out));
    const int v = packed ? packed_variant(m, n, k, weight_bits, variant) : resolve_variant(m, n, k, weight_bits, variant);
    if (v < 0) return v;
    out->compute_units = machine_cus();
    out->launches = 1;
    out->splits = 1;
    out->k_per_workgroup = k;
    if (m == 0 || n == 0) return BFAINTB_OK;
    auto tiles_of_128_columns = [&](uint32_t blocks, uint32_t splits, uint32_t k_per_wg) {
        GemmParams p{};
        p.m = m;
        p.group_size = group_size;
        p.tile_blocks = blocks;
        p.splits = splits;
        p.k_per_wg = k_per_wg;
        out->kernel = BFAINTB_KERNEL_TILES_128;
        out->tile_rows = 16u * blocks;
        out->tile_cols = 128u;
        out->waves = bfaintb::prefill128_wreg_copier(p, weight_bits, packed != 0) ? 9u : 8u;
        out->splits = splits;
        out->k_per_workgroup = k_per_wg;
        out->workgroups = ((m + out->tile_rows - 1u) / out->tile_rows) * ((n + 127u) / 128u) * splits;
    };
    if (v == BFAINTB_VARIANT_DECODE) {
        out->variant = v;
        if (packed && packed_uses_slab(m, n, k, weight_bits)) {
            out->kernel = BFAINTB_KERNEL_DECODE_SLAB;
            out->tile_rows = m <= 16u ? 16u : 32u;
            out->tile_cols = 16u;
            out->waves = 8u;
            out->workgroups = n / 16u * ((m + out->tile_rows - 1u) / out->tile_rows);
            return BFAINTB_OK;
        }
        const DecodePlan pl = packed ? packed_family_plan(m, n, k, weight_bits) : decode_plan(m, n, k, weight_bits, split_k);
        out->workspace_bytes = split_workspace_bytes(pl.splits, m, n);
        if (variant == BFAINTB_VARIANT_AUTO && (packed || split_k == 0) && few_rows_on_tiles(m, n, k, weight_bits, group_size != 0, packed != 0, n)) {
            tiles_of_128_columns(2u, 1u, (k + 63u) / 64u * 64u);
            out->tiles_instead = out->workgroups;
            return BFAINTB_OK;
        }
        out->kernel = BFAINTB_KERNEL_DECODE_FAMILY;
        out->tile_rows = 16u * pl.mb;
        out->tile_cols = pl.cols;
        out->waves = pl.waves;
        out->splits = pl.splits;
        out->k_per_workgroup = pl.k_per_wg;
        out->workgroups = ((n + pl.cols - 1u) / pl.cols) * pl.splits * ((m + 16u * pl.mb - 1u) / (16u * pl.mb));
        return BFAINTB_OK;
    }
    // the tiled kernels
    if (v == BFAINTB_VARIANT_PREFILL) {
        const WideTiles w = wide_tiles(m, n, k, weight_bits, packed ? 0u : split_k);
        if (w.blocks != 0u) {
            out->variant = v;  // (no variant names these tiles)
            out->kernel = BFAINTB_KERNEL_TILES_256;
            out->tile_rows = 16u * w.blocks;
            out->tile_cols = 256u;
            out->waves = 4u;
            out->workgroups = w.rows_of_tiles * ((n + 255u) / 256u);
            return BFAINTB_OK;
        }
    }
    if (use_small_tiles(v, m, n, k, weight_bits)) {
        out->variant = BFAINTB_VARIANT_PREFILL_128;
        if (v != BFAINTB_VARIANT_PREFILL_128_LDS) {
            const TilePlan tp = tile128_plan(m, n, k, weight_bits, packed ? 0u : split_k);
            tiles_of_128_columns(tp.blocks, tp.splits, tp.k_per_wg);
            out->launches = 1u + tp.finish_launch;
            out->workspace_bytes = tile_workspace_bytes(tp, m, n);
            return BFAINTB_OK;
        }
        out->kernel = BFAINTB_KERNEL_TILES_128_LDS;
        out->tile_rows = out->tile_cols = 128u;
        out->waves = 8u;
        out->workgroups = ((m + 127u) / 128u) * ((n + 127u) / 128u);
        return BFAINTB_OK;
    }
    if (v == BFAINTB_VARIANT_PREFILL_256X128 || (v == BFAINTB_VARIANT_PREFILL && prefill_tall_tiles(m, n, k, weight_bits))) {
        if (v == BFAINTB_VARIANT_PREFILL && !tall_tiles_in_one_chain(m, k)) {
            out->variant = v;  // (no variant names these tiles)
            tiles_of_128_columns(tall_tile_blocks(m), 1u, (k + 63u) / 64u * 64u);
            return BFAINTB_OK;
        }
        out->variant = BFAINTB_VARIANT_PREFILL_256X128;
        out->kernel = BFAINTB_KERNEL_TILES_256X128;
        out->tile_rows = 256u;
        out->tile_cols = 128u;
        out->waves = 4u;
        out->workgroups = ((m + 255u) / 256u) * ((n + 127u) / 128u);
        return BFAINTB_OK;
    }
    out->variant = v == BFAINTB_VARIANT_PREFILL_256_LDS ? v : BFAINTB_VARIANT_PREFILL_256;
    out->kernel = v == BFAINTB_VARIANT_PREFILL_256_LDS ? BFAINTB_KERNEL_TILES_256_LDS : BFAINTB_KERNEL_TILES_256;
    out->tile_rows = out->tile_cols = 256u;
    out->waves = v == BFAINTB_VARIANT_PREFILL_256_LDS ? 8u : 4u;
    {
        const uint32_t tiles = ((m + 255u) / 256u) * ((n + 255u) / 256u);
        const uint32_t halves = bfaintb::thin_round_tiles(tiles, m, machine_cus());
        out->workgroups = tiles - halves;
        out->tail_workgroups = 2u * halves;
        out->launches = (tiles - halves != 0u ? 1u : 0u) + (halves != 0u ? 1u : 0u);
    }
    return BFAINTB_OK;
}

// What a call would launch, without launching it: the queries above rolled into one description, for callers that want
// to log or check the library's choice and for the scans that hold the choice against measurements.
int bfaintb_gemm_plan(uint32_t m, uint32_t n, uint32_t k, int weight_bits, uint32_t group_size, int packed, int variant, uint32_t split_k,
                      bfaintb_plan* out)
{
    if (out == nullptr) return BFAINTB_ERR_NULL_POINTER;
    memset(out, 0, sizeof(*out));
    int e = check_format(k, weight_bits, group_size);
    if (e) return e;
    e = check_shape(m, n, k, packed ? 8 : weight_bits);
    if (e) return e;
    if (packed) {
        e = check_packed_shape(n, k, weight_bits);
        if (e) return e;
    }
    const int v = packed ? packed_variant(m, n, k, weight_bits, variant) : resolve_variant(m, n, k, weight_bits, variant);
    if (v < 0) return v;
    if (variant == BFAINTB_VARIANT_AUTO && (packed || split_k == 0)) {
        const uint32_t head = row_split_head(m, n, k, weight_bits, packed != 0, group_size != 0);
        if (head != 0u) {  // the first launch, described as such; of the second one its workgroups
            bfaintb_plan rest;
            e = plan_whole(head, n, k, weight_bits, group_size, packed, variant, 0, out);
            if (e == 0) e = plan_whole(m - head, n, k, weight_bits, group_size, packed, variant, 0, &rest);
            if (e) return e;
            out->tail_workgroups += rest.workgroups + rest.tail_workgroups;
            out->launches += rest.launches;
            out->workspace_bytes = row_split_workspace(head, m - head, n, k, weight_bits, packed != 0);
            return BFAINTB_OK;
        }
    }
    return plan_whole(m, n, k, weight_bits, group_size, packed, variant, split_k, out);
}

uint32_t bfaintb_prefill_tile(uint32_t m, uint32_t n) { return prefill_small_tiles(m, n, 4096u, 8) ? 128u : 256u; }
uint32_t bfaintb_prefill_tile_cols(uint32_t m, uint32_t n) { return (prefill_small_tiles(m, n, 4096u, 8) || prefill_tall_tiles(m, n, 4096u, 8)) ? 128u : 256u; }

const char* bfaintb_kernel_name(int variant, int weight_bits, uint32_t group_size, uint32_t m)
{
    int v = variant;
    if (v == BFAINTB_VARIANT_AUTO) v = m <= kDecodeAutoMaxM ? BFAINTB_VARIANT_DECODE : BFAINTB_VARIANT_PREFILL;
    if (v == BFAINTB_VARIANT_DECODE) return "bfaintb_decode_kernel";
    // (row-major weights, plain or bias epilogue; the forms with both operands in LDS serve the rest)
    if (v == BFAINTB_VARIANT_PREFILL || v == BFAINTB_VARIANT_PREFILL_256) return "bfaintb_prefill_wreg_kernel";
    if (v == BFAINTB_VARIANT_PREFILL_256_LDS) return "bfaintb_prefill_kernel";
    if (v == BFAINTB_VARIANT_PREFILL_128) return "bfaintb_prefill128_wreg_kernel";
    if (v == BFAINTB_VARIANT_PREFILL_128_LDS) return "bfaintb_prefill128_kernel";
    if (v == BFAINTB_VARIANT_PREFILL_256X128) return "bfaintb_prefill256x128_wreg_kernel";
    (void)weight_bits;
    (void)group_size;
    return "";
}

}  // extern "C"
