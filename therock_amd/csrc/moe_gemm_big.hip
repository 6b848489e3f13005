// Large-tile grouped GEMM for prefill-sized expert batches (gfx950).
//
// Same math and epilogues as moe_gemm_kernel, different machinery:
//   * 512 threads = 8 waves as 2 (token halves) x 4 (weight-row quarters); the workgroup owns up to
//     320 sorted rows of one expert (ten 32-row blocks, interleaved between the two token halves)
//     and 256 weight rows.  320 rather than 256 so that an expert of the DeepSeek-V3-shaped
//     workload (about 270 rows) is one tile and its weights are fetched once.
//   * Both operands go global -> LDS with global_load_lds_dwordx4 (no staging registers).  The K loop
//     advances in 64-byte steps.  Tokens (re-read from L2 by every column tile) arrive one 64-byte
//     step at a time through a ring of three to six stages (step_stages).  Weights are streamed from HBM exactly once, as
//     full 128-byte lines, half of the tile's rows per unit (unit u = rows (u&1)*128.., K bytes
//     [128*(u>>1), +128)), through a ring of six units issued four steps ahead.
//   * The loads are issued from inline assembly so that their completion is tracked by hand:
//     s_waitcnt vmcnt(n) with n = the DMA instructions this wave issued after the data about to be
//     consumed, then one workgroup barrier per step, which also frees the buffers the next issues
//     write into.  Loads of one wave return in order, so the two streams are issued by different
//     waves (0..3 weights, 4..7 tokens): mixed in one wave, the L2-hit token loads would queue
//     behind the HBM-miss weight loads.
//   * What bounds the kernel is the compute unit's vector memory path: L2 hits queued behind HBM misses do
//     not overtake them, so the token stream costs its stand-alone time on top of the weight stream (about
//     19 bytes per clock together; a step of this tile needs up to 36.9 KB for 1400 clocks of MFMA work).
//   * LDS rows are swizzled: 64-byte token rows keep chunk c of row r at c ^ ((r >> 2) & 3), 128-byte
//     token rows at c ^ ((r >> 1) & 7), 128-byte weight rows at c ^ weight_row_swizzle(r); both the linear DMA
//     writes and the ds_read_b128 operand fetches are then conflict-free on the 64-bank LDS.  Weight rows sit in
//     LDS in channel order (row r of a 32-row block = channel r; the lane whose MFMA row is m reads row
//     chan_of_row(m)), so that the eight rows of a DMA instruction are eight consecutive channels: eight full
//     128-byte lines in the row-major layout and in ck_tile's pre-shuffled one alike.  Token rows past the tile's last row inside a
//     fetched 64-row group (and padding ids) fetch some real row instead - their MFMA columns are never
//     stored; whole groups the tile does not have are not fetched.
//   * The K loop is specialised on the number of token blocks a wave owns, on the number of 64-row token
//     groups the tile has and on whether the weight DMA is non-temporal, so that the MFMA region is
//     straight-line code and every wait count a compile-time constant: scalar branches in the issue path
//     cost 5 % of the kernel's time when tried.
//   * The int8 path runs here too: i8 MFMAs for the gate+up GEMM; for the down GEMM bf16 tokens against
//     int8 weights that are converted after the LDS read, one 128-byte weight line lasting four K steps.
//   * Work items go to the XCDs in chunks of 32 (see lookup_tile).
#include "moe_gemm_device.hpp"

#include <algorithm>
#include <mutex>
#include <type_traits>

namespace mi355 {
using namespace gemm;
namespace {

constexpr int kBigThreads   = 512;
constexpr int kStepKB       = 64;  // bytes of K per compute step and row
constexpr int kBigWRows     = 256;
constexpr int kBigXRows     = 320;
constexpr int kMaxNB        = kBigXRows / 64; // token blocks per wave (5)
constexpr int kWHalfRows    = kBigWRows / 2;
constexpr int kWUnitBytes   = kWHalfRows * 2 * kStepKB; // 128 rows x 128 B
constexpr int kWSlots       = 6;
constexpr int kYsRows       = 512;                      // padded rows per K block of a scale stage
constexpr int kYsStageBytes = (kStepKB / 32) * kYsRows; // fp8 gemm1: e8m0 scales of 2 K blocks
constexpr int kXOffset      = kWSlots * kWUnitBytes;
constexpr int kLdsBytes     = 160 * 1024; // of a gfx950 compute unit
// Gate+up GEMM (token rows gathered by id): a token stage holds 128 bytes of K per row, two compute steps, so that a
// token DMA instruction fetches eight whole 128-byte lines instead of sixteen half lines (a compute unit's address
// path moves 100 GB/s in whole lines and 58 GB/s in halves).  Two such stages of a full tile and a weight ring of five slots.
constexpr int kWSlotsPair   = 5;
constexpr int kXOffsetPair  = kWSlotsPair * kWUnitBytes;

// Token stages of a tile of `groups` 64-row token groups: as many as fit beside the weight ring.  A compute unit's requests
// return in order, so a token stage arrives with the HBM latency of the weights ahead of it (1.4 us and more under load),
// and a step of a tile of few rows, whose MFMAs take 0.2 .. 0.4 us, took half of that with the two stages a full tile has
// room for (0.7 .. 0.9 us whatever the operand type or the rows).  More weight units in flight (seven slots) changed nothing.
// Passes, two -> as many stages as fit: 900 tokens x 8 of 64 bf16 experts 2560 x 1536 363 -> 339 us, 1881 x 3 of 39 bf16 experts
// 6976 x 2880 1080 -> 1038, 2048 x 8 of 128 int8 experts 4096 x 1536 743 -> 697, 777 x 4 of 32 fp16 experts 2880 x 2880 382 -> 372.
constexpr int pair_stage_bytes(int groups) { return groups * 64 * 2 * kStepKB; }
constexpr int pair_stages(int groups) { return groups <= 2 ? 4 : groups == 3 ? 3 : 2; }
constexpr int step_stage_bytes(int groups) { return groups * 64 * kStepKB; }
constexpr int step_stages(int groups, bool scales) { return groups <= 2 ? 6 : groups == 3 ? (scales ? 4 : 5) : groups == 4 ? (scales ? 3 : 4) : 3; }
constexpr bool stages_fit(int groups)
{
    return kXOffsetPair + pair_stages(groups) * pair_stage_bytes(groups) <= kLdsBytes &&
           kXOffset + step_stages(groups, false) * step_stage_bytes(groups) <= kLdsBytes &&
           kXOffset + step_stages(groups, true) * (step_stage_bytes(groups) + kYsStageBytes) <= kLdsBytes;
}
static_assert(stages_fit(1) && stages_fit(2) && stages_fit(3) && stages_fit(4) && stages_fit(kMaxNB), "LDS budget");

// Epilogue operands of a gate+up tile of 8-bit operands, fetched into LDS ahead of the first stages, where a tile of up to four
// token groups leaves room: the 256 weight rows' scales, the token rows' scales and their sorted ids, 1 KiB each.  Loaded behind
// the K loop they were two dependent round trips, one past L2, with nothing else of the compute unit in flight (4300 clocks
// of a tile's 35000 where K is 640 bytes).  Passes: 8541 tokens x 7 of 166 int8 experts 640 x 12544 3310 -> 3139 us, 3526 x 5 of 111
// int8 experts 512 x 1792 194 -> 189, 4054 x 8 of 47 int8 experts 3072 x 896 499 -> 484.
constexpr int kEpiGroups   = 4;
constexpr int kEpiRows     = kEpiGroups * 64;
constexpr int kEpiOffset   = kLdsBytes - 3 * 1024;
constexpr int kEpiChannels = kEpiOffset, kEpiScales = kEpiOffset + 1024, kEpiIds = kEpiOffset + 2048;
constexpr bool epilogue_fits(int groups) { return kXOffsetPair + pair_stages(groups) * pair_stage_bytes(groups) <= kEpiOffset; }
static_assert(epilogue_fits(1) && epilogue_fits(2) && epilogue_fits(3) && epilogue_fits(kEpiGroups) && kBigWRows * 4 <= 1024 && kEpiRows * 4 <= 1024,
              "LDS budget of the epilogue's operands");

typedef __attribute__((address_space(3))) unsigned char lds_byte_t;

// Chunk swizzle of the 128-byte weight rows in LDS.  The 16 lanes that a ds_read_b128 serves together read the rows
// chan_of_row(16 i .. 16 i + 15) = {0..3, 16..19, 4..7, 20..23} (+ 8 for i = 1): among the rows of equal parity (two
// rows span the 64 banks) bits 1, 2 and 4 of the row number take all eight values.
__device__ __host__ constexpr int weight_row_swizzle(int r) { return ((r >> 1) & 3) | (((r >> 4) & 1) << 2); }


__device__ inline uint32_t lds_offset(const void* p)
{
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const lds_byte_t*)p));
}

__device__ inline const unsigned char* uniform_ptr(const unsigned char* p)
{
    const uint64_t v  = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
    return reinterpret_cast<const unsigned char*>((static_cast<uint64_t>(hi) << 32) | lo);
}

// lane i of the wave copies 16 (4) bytes from base + off (a wave-uniform base, a per-lane 32-bit offset)
// to LDS byte m0 + 16*i (4*i)
__device__ inline void dma16(const unsigned char* base_uniform, uint32_t off, uint32_t m0_uniform)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m0_uniform), "v"(off), "s"(uniform_ptr(base_uniform))
                 : "memory");
}
__device__ inline void dma16nt(const unsigned char* base_uniform, uint32_t off, uint32_t m0_uniform)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(m0_uniform), "v"(off), "s"(uniform_ptr(base_uniform))
                 : "memory");
}
__device__ inline void dma4(const unsigned char* base_uniform, uint32_t off, uint32_t m0_uniform)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(m0_uniform), "v"(off), "s"(uniform_ptr(base_uniform))
                 : "memory");
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>): indices that are constants before any loop pass runs
template <int N, typename F>
__device__ __attribute__((always_inline)) inline void static_for(F&& f)
{
    if constexpr(N > 0)
    {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

template <int N>
__device__ inline void wait_vmcnt()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// WPERM: the weights are in ck_tile's pre-shuffled layout, where 128 contiguous bytes are one 16-byte chunk of eight
// consecutive rows.  The eight rows x eight chunks of a weight DMA instruction then sit in LDS chunk-major - lane
// 8 c' + r fetches chunk c' ^ s of row r, s = bit 1 of the instruction's number, and lands at byte 128 c' + 16 r of
// the instruction's 1 KiB - so that eight consecutive lanes fetch one whole line, as they do for row-major weights
// in the row-major LDS layout (eight chunks of one row).  The operand fetches of sixteen lanes (rows 0..7 of one
// instruction, rows 16..23 of the one two further on, same chunk) cover 256 contiguous bytes modulo the bank span
// thanks to s.
template <int MODE, bool GEMM0, bool WPERM>
__global__ __launch_bounds__(kBigThreads) void moe_gemm_big_kernel(const GemmParams p)
{
    using MT  = ModeTraits<MODE>;
    using Acc = typename MT::Acc;
    constexpr int kOpB   = MT::kOpB;
    constexpr int kSteps = kStepKB / (2 * kOpB); // MFMAs along K per compute step: 1 (fp8) or 2 (bf16, i8)
    // int8 weights against bf16 tokens (down GEMM of the int8 path): a 64-byte token step is 32 elements = 32
    // weight bytes, so the 128-byte lines of a weight unit last four steps instead of two
    constexpr bool kW8 = MODE == kBf16W8;
    constexpr bool kMx   = MODE == kFp8 && !GEMM0;
    static_assert(MODE == kBf16 || MODE == kF16 || MODE == kFp8 || MODE == kI8 || (MODE == kBf16W8 && !GEMM0),
                  "no large-tile kernel for this mode");
    // Software-pipelined K loop (kPipe): the operands of step k+1 are fetched from LDS into registers during step
    // k, each fragment right behind the last MFMA that reads its register, so that after a barrier the MFMAs start
    // at once instead of waiting for operand fetches that all eight waves issue at the same moment.  The barrier of
    // step k then has to guarantee the data of step k+1: every transfer runs one step further ahead.
    constexpr bool kPipe  = !kMx;
    constexpr bool kXPair = kPipe && GEMM0; // 128-byte token stages
    // 8-bit rows of an odd number of 64-byte steps (hidden sizes that are odd multiples of 64): the last 128-byte window
    // has only its first half.  Lanes that would fetch the second half (the next row's bytes, past the tensor's end in its
    // last row) fetch the first one again, and the last step has no partner, so nothing reads what they fetched.
    constexpr bool kOddK = kXPair && (MODE == kI8 || MODE == kFp8);
    // Down GEMM weights of one byte a value, rows of an odd number of 64-byte pieces: the last 128-byte window begins 64 bytes
    // earlier, inside the row, and the steps it serves read its second half.
    constexpr bool kOddW = !GEMM0 && (MODE == kI8 || kW8);
    constexpr int kWS     = kXPair ? kWSlotsPair : kWSlots;
    // token stages (steps, or pairs of steps) of a tile, and the LDS offset of its scale stages
    constexpr auto x_stages  = [](int groups) { return kXPair ? pair_stages(groups) : step_stages(groups, kMx); };
    constexpr auto ys_offset = [](int groups) { return kXOffset + step_stages(groups, kMx) * step_stage_bytes(groups); };

    extern __shared__ __align__(16) unsigned char lds[];

    const int tid  = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r32  = lane & 31;
    const int kg   = lane >> 5;
    // waves w and w+4 share a SIMD: give them the two token halves of the same weight quarter, so
    // that every SIMD carries the same number of token blocks
    const int wt   = wave >> 2; // token half: blocks wt, wt+2, ...
    const int ww   = wave & 3;  // weight-row quarter

    // ---- work item (same XCD-aware order as moe_gemm_kernel)
    const TileRef tile = lookup_tile<true>(p.tile_map, p.n_ntiles, p.max_tiles, blockIdx.x, p.tile_rows);
    if(!tile.ok)
        return;
    const int expert = tile.expert;
    const int row0   = tile.row0;
    const int slice  = !GEMM0 && p.k_cols > 0 ? tile.nt / p.k_cols : 0; // slice of K (down GEMM)
    const int nt     = tile.nt - slice * p.k_cols;
    const int nrows  = tile.nrows;
    const int nmb    = ceil_div(nrows, 32);
    const bool paired = GEMM0 && !p.gate_only; // gate rows paired with up rows (see run_epilogue)
    const int n_base  = nt * (paired ? 128 : 256);

    // ---- DMA assignments.
    // Loads of one wave return in order, so a wave that mixed the two streams would see its L2-hit
    // token loads queue behind HBM-miss weight loads.  The streams are therefore issued by different
    // waves: waves 0..3 the weights, waves 4..7 the tokens (and, on the fp8 down-GEMM, the e8m0 scales).
    // Weights: unit u = rows (u & 1) * 128 .. + 127 of the tile, K bytes [128 * (u >> 1), + 128).  One unit
    // is 16 instructions of 8 rows x 128 B (full cache lines); wave w issues instructions w, w+4, w+8, w+12.
    // Tokens: step x = the tile's rows, K bytes [64 x, + 64), up to 20 slabs of 16 rows x 64 B; wave 4+q fills
    // slabs q, q+4, .. as far as the tile has rows (one instruction per 64 rows of the tile) and fetches 256
    // scale bytes.  The count is a template argument of the K loop: selecting the instructions and the
    // matching wait with scalar branches inside the loop cost 5 % of the kernel's time.
    // Every source address is a wave-uniform base (operand base + K offset of the unit, kept in
    // scalar registers) plus a per-lane 32-bit row offset doff[] that never changes: weights
    // doff[4 * half + j]; tokens doff[0..4], scales doff[5].  Token rows that do not exist (padding
    // ids, rows past the tile) read row 0 instead: their MFMA columns are never stored.
    const bool w_role = wave < 4;
    const int q4      = wave & 3;
    uint32_t doff[kXPair ? 10 : 8];
    const unsigned char* dbase;
    if(w_role)
    {
        dbase = uniform_ptr(p.w + (int64_t)expert * p.w_expert_bytes);
#pragma unroll
        for(int h = 0; h < 2; h++)
#pragma unroll
            for(int j = 0; j < 4; j++)
            {
                const int inst   = q4 + 4 * j;                      // instruction of the unit: LDS rows 8 inst .. + 7
                const int rih    = inst * 8 + (WPERM ? lane & 7 : lane >> 3); // LDS row inside the half
                const int trow   = h * kWHalfRows + rih;
                const int blk    = trow >> 5;
                const int c      = trow & 31; // LDS row r of a 32-row block holds weight channel r (see weight_row_swizzle)
                const int cchunk = WPERM ? (lane >> 3) ^ ((inst >> 1) & 1) : (lane & 7) ^ weight_row_swizzle(rih);
                int grow;
                if(paired)
                    grow = (blk & 1) * p.n_out + min(n_base + (blk >> 1) * 32 + c, p.n_out - 1);
                else
                    grow = min(n_base + blk * 32 + c, p.n_total - 1);
                doff[h * 4 + j] = weight_offset(p, p.w_permuted != 0, grow, cchunk);
            }
    }
    else
    {
        dbase = uniform_ptr(p.x);
        if constexpr(kXPair)
        {
            // instruction j of wave 4 + q: rows (q + 4 j) * 8 .. + 7 of the tile, 128 bytes each, chunks swizzled
            // like the weight rows
#pragma unroll
            for(int j = 0; j < 10; j++)
            {
                const int lrow = (q4 + 4 * j) * 8 + (lane >> 3);
                int sid        = p.tokens;
                if(lrow < nrows)
                    sid = p.sorted_ids[row0 + lrow];
                const uint32_t src = real_id(sid, p.tokens, p.topk) ? token_row(p, sid) : 0u;
                doff[j]            = src * (uint32_t)p.x_row_bytes + ((lane & 7) ^ ((lrow >> 1) & 7)) * 16;
            }
        }
        else
        {
            const int lrow16 = lane >> 2;
            const int cchunk = (lane & 3) ^ ((lane >> 4) & 3);
#pragma unroll
            for(int j = 0; j < 5; j++)
            {
                const int lrow = (q4 + 4 * j) * 16 + lrow16;
                uint32_t src   = lrow < nrows ? row0 + lrow : row0;
                if(GEMM0 || p.slot_rows > 0)
                {
                    int sid = p.tokens;
                    if(lrow < nrows)
                        sid = p.sorted_ids[row0 + lrow];
                    const bool ok = real_id(sid, p.tokens, GEMM0 ? p.topk : p.slot_rows);
                    src           = !ok ? 0u : GEMM0 ? token_row(p, sid) : (uint32_t)slot_row(sid, p.slot_rows);
                }
                doff[j] = src * (uint32_t)p.x_row_bytes + cchunk * 16;
                if(!GEMM0 && p.y_slab > 0) // slab-major Y: whole slabs; slabs past the tile's rows read its first
                    doff[j] = (uint32_t)(((row0 >> 4) + ((q4 + 4 * j) * 16 < nrows ? q4 + 4 * j : 0)) * p.y_slab) * 1024u +
                              lrow16 * 64 + cchunk * 16;
            }
            // scales: K block (q >> 1) of the step, rows (q & 1) * 256 .. + 255 (the rows are padded)
            doff[5] = (uint32_t)((q4 >> 1) * p.ys_kb_stride + row0 + (q4 & 1) * 256 + lane * 4);
            doff[6] = doff[7] = 0;
        }
    }
    const int64_t ys_step = (kStepKB / 32) * p.ys_kb_stride;
    const int x_step      = (!GEMM0 && p.y_slab > 0) ? 1024 : kStepKB; // bytes between token steps

    const uint32_t lds_base = lds_offset(lds);
    // compute steps of this workgroup's slice of K, whose first bytes the base addresses point at (a slice is a multiple of
    // 512 weight bytes): even, but for 8-bit rows of an odd number of 64-byte steps (kOddK, kOddW)
    int kt_count = p.k_bytes_x / kStepKB;
    const unsigned char* ys_base = p.y_scale;
    if(!GEMM0 && p.k_cols > 0)
    {
        const int slice_steps = p.k_slice / (kW8 ? kStepKB / 2 : kStepKB);
        const int step0       = slice * slice_steps;
        kt_count              = min(kt_count - step0, slice_steps);
        dbase = uniform_ptr(dbase + (w_role ? (int64_t)slice * weight_k_advance(p, p.k_slice) : (int64_t)step0 * x_step));
        if constexpr(kMx)
            ys_base += step0 * ys_step;
    }
    const bool odd_k        = (kOddK || kOddW) && (kt_count & (kW8 ? 2 : 1)) != 0; // (kW8: 64 bytes of weights are two steps)
    const int n_wunits      = kW8 ? (kt_count + (odd_k ? 2 : 0)) / 2 : kt_count + (odd_k ? 1 : 0); // two units (row halves) per 128 bytes of weight K
    // Where the walk over K begins.  The 256 weight rows of a tile lie a row pitch apart, so that with a pitch of whole
    // 4 KiB (hidden 4096 or 2048 in 16 bits, 4096 or 8192 in 8) every row of a K window sits behind the same L2 channel,
    // and the workgroups of an XCD, started together, walk the channels in step.  Column tile i begins a
    // share of K further on instead, the fractional part of i * golden ratio, and wraps around: any run of consecutive
    // tiles, the 32 an XCD runs together, spreads evenly over the row and its channels.  (Steps of 3, 5, 9, 11 and 13
    // windows of 128 bytes measured the same; 4 windows reach 16 of the start points of an 8 KiB row and are as slow as
    // none.  Tiles are numbered over the experts, as a narrow layer has few columns.)  Gate+up
    // GEMM at 83 rows per expert: bf16 8 x 4096 x 16384 462 -> 350 us (4.7 -> 6.1 TB/s), fp8 / int8 16 x 4096 x 8192
    // 255 -> 190 / 262 -> 200 us; at other pitches up to 4 % (int8, 64 x 7168 x 2048 at 84 rows: pass 713 -> 684 us).
    // Which layers do: big_k_spread, by sizes alone, so that the order of a token's sums does not depend on how many rows other
    // tokens bring its expert.  (int8 sums are exact in any order: there experts of several row tiles, which fetch each
    // weight slice together and each token slice for eight column tiles at a time, keep one place to begin at.)
    constexpr uint32_t kGolden = 0x9e3779b9u; // its fractional part in units of 2^-32
    const int n_win   = n_wunits >> 1; // 128-byte windows of weight K
    const bool rotate = !odd_k && p.k_spread != 0 && (MODE != kI8 || tile.expert_tiles == 1);
    const uint32_t at = (uint32_t)expert * (uint32_t)p.n_ntiles + (uint32_t)tile.nt;
    const int rot     = rotate ? (int)__umulhi(at * kGolden, (uint32_t)n_win) : 0; // < n_win
    // the wave's stream (weights or tokens): address of the window it is in, moved on by its issue functions
    const int w_kadv            = weight_k_advance(p, 2 * kStepKB); // bytes between the 128-byte K windows of two weight units
    const int64_t window_bytes  = w_role ? w_kadv : (int64_t)x_step * (kW8 ? 4 : 2);
    const unsigned char* stream = dbase + window_bytes * rot;
    ys_base += rot * 2 * ys_step; // (moves along with the tokens)
    // windows until the stream goes back, and by how much: to the start of K, or (kOddW) the half window
    const bool half_window = kOddW && odd_k && w_role;
    int windows_left       = half_window ? n_win - 1 : n_win - rot;
    const int64_t back     = half_window ? w_kadv / 2 : window_bytes * n_win;
    if(half_window && windows_left == 0) // (a slice of 64 bytes: the window begins in the slice before)
        stream -= back;
    // (selects, not a branch: branches in the issue path cost time)
    auto end_window = [&](int64_t bytes) __attribute__((always_inline)) {
        const bool end = --windows_left == 0;
        stream += bytes - (end ? back : 0);
        if constexpr(kMx)
            ys_base -= end ? n_win * 2 * ys_step : 0;
    };

    // weight role: unit u (half u & 1) -> ring slot u % 6
    // Weights no other row tile re-reads (the expert has a single one) are fetched non-temporal: measured
    // -8 % on the gate+up GEMM at 32 rows per expert, -2 % at 256; with several row tiles per expert the
    // re-reads should hit L2, and non-temporal fetches cost 3 % there.  NT is a template argument like the
    // slab-group count, for the same reason.  8-bit rows of an odd number of 64-byte pieces are left out: a 128-byte piece of
    // every second row lies in two lines there, the pieces before and after in the same two, and with the hint each is fetched
    // twice.  Passes, with -> without it: 1600 tokens x 8 of 64 int8 experts 4160 x 3008 870 -> 786 us, 1150 x 4 of 20 fp8 experts
    // 6336 x 9344 1054 -> 995, 680 x 4 of 16 int8 experts 2112 x 14272 580 -> 542; at 90 rows per expert no difference.
    const bool w_nt = tile.expert_tiles == 1 && (WPERM || p.w_row_bytes % 128 == 0);
    auto issue_w = [&](int u, auto half_tag, auto nt_tag) __attribute__((always_inline)) {
        constexpr int H = decltype(half_tag)::value;
        constexpr bool NT = decltype(nt_tag)::value;
        if(u >= n_wunits)
            return;
        const uint32_t sbase     = lds_base + ((uint32_t)u % kWS) * kWUnitBytes + q4 * 1024;
        const unsigned char* src = stream;
#pragma unroll
        for(int j = 0; j < 4; j++)
        {
            // H < 0: the row half is not known at compile time (int8 weights: one unit every other step); the
            // choice is spelled as arithmetic, a select between two elements of doff[] turns the array into an
            // indexed one in scratch memory
            const uint32_t off = H >= 0 ? doff[(H >= 0 ? H : 0) * 4 + j]
                                        : doff[j] ^ ((doff[j] ^ doff[4 + j]) & (0u - (uint32_t)(u & 1)));
            if constexpr(NT)
                dma16nt(src, off, __builtin_amdgcn_readfirstlane(sbase + j * 4096));
            else
                dma16(src, off, __builtin_amdgcn_readfirstlane(sbase + j * 4096));
        }
        if(H < 0 ? (u & 1) : H)
        {
            end_window(w_kadv);
        }
    };
    // token role: step x -> ring stage x % x_stages(groups)
    auto issue_x = [&](int x, int stage, int groups) __attribute__((always_inline)) {
        if(x >= kt_count)
            return;
        const uint32_t sbase     = lds_base + kXOffset + stage * step_stage_bytes(groups) + q4 * 1024;
        const unsigned char* src = stream;
#pragma unroll
        for(int j = 0; j < 5; j++)
            if(j < groups)
                dma16(src, doff[j], __builtin_amdgcn_readfirstlane(sbase + j * 4096));
        if constexpr(kMx)
        {
            dma4(ys_base, doff[5],
                 __builtin_amdgcn_readfirstlane(lds_base + ys_offset(groups) + stage * kYsStageBytes +
                                                (q4 >> 1) * kYsRows + (q4 & 1) * 256));
            ys_base += ys_step;
        }
        if((x & (kW8 ? 3 : 1)) == (kW8 ? 3 : 1))
            end_window(x_step);
        else
            stream += x_step;
    };

    // (kOddK) token lanes of the half the last pair does not have fetch the other half from here on
    auto halve_x = [&]() __attribute__((always_inline)) {
        if constexpr(kXPair)
        {
#pragma unroll
            for(int j = 0; j < 10; j++)
            {
                const int lrow = (q4 + 4 * j) * 8 + (lane >> 3);
                doff[j] -= (((lane & 7) ^ ((lrow >> 1) & 7)) & 4) ? 64u : 0u;
            }
        }
    };
    // 128-byte token stages: pair m = steps 2 m and 2 m + 1 -> stage m % x_stages(groups); two instructions per 64 rows of the
    // tile
    auto issue_x_pair = [&](int m, int stage, int groups) __attribute__((always_inline)) {
        if constexpr(kXPair)
        {
            if(2 * m >= kt_count)
                return;
            const uint32_t sbase     = lds_base + kXOffsetPair + stage * pair_stage_bytes(groups) + q4 * 1024;
            const unsigned char* src = stream;
#pragma unroll
            for(int j = 0; j < 10; j++)
                if(j < 2 * groups)
                    dma16(src, doff[j], __builtin_amdgcn_readfirstlane(sbase + j * 4096));
            end_window(2 * kStepKB);
        }
    };

    // token blocks of this wave (blocks wt, wt + 2, ..) and 64-row slab groups that hold rows of the tile
    const int nb_w     = __builtin_amdgcn_readfirstlane(max(0, min(kMaxNB, (nmb - wt + 1) / 2)));
    const int x_groups = __builtin_amdgcn_readfirstlane(max(1, (nmb + 1) / 2));

    // the epilogue's operands: ahead of all other transfers of these waves, so that the first wait covers them
    constexpr bool kEpi = kXPair && (MODE == kI8 || MODE == kFp8);
    const bool epi_lds  = kEpi && x_groups <= kEpiGroups && p.w_scale != nullptr && p.x_scale != nullptr;
    if constexpr(kEpi)
    {
        if(epi_lds && w_role)
        {
            // scale of weight row i of the tile, 64 a wave
            const int i   = q4 * 64 + lane;
            const int row = paired ? (i >> 7) * p.n_out + min(n_base + (i & 127), p.n_out - 1) : min(n_base + i, p.n_total - 1);
            dma4(reinterpret_cast<const unsigned char*>(p.w_scale + (int64_t)expert * p.n_total), (uint32_t)row * 4u,
                 __builtin_amdgcn_readfirstlane(lds_base + kEpiChannels + q4 * 256));
        }
        else if(epi_lds)
        {
            const int r   = min(q4 * 64 + lane, nrows - 1);
            const int sid = p.sorted_ids[row0 + r];
            dma4(reinterpret_cast<const unsigned char*>(p.sorted_ids + row0), (uint32_t)r * 4u,
                 __builtin_amdgcn_readfirstlane(lds_base + kEpiIds + q4 * 256));
            dma4(reinterpret_cast<const unsigned char*>(p.x_scale), real_id(sid, p.tokens, p.topk) ? token_row(p, sid) * 4u : 0u,
                 __builtin_amdgcn_readfirstlane(lds_base + kEpiScales + q4 * 256));
        }
    }

    Acc acc[kMaxNB][2];
#pragma unroll
    for(int i = 0; i < kMaxNB; i++)
#pragma unroll
        for(int b = 0; b < 2; b++)
#pragma unroll
            for(int v = 0; v < 16; v++)
                acc[i][b][v] = 0;

    // prologue: weight units 0..3 (0..4 when pipelined with six slots, unless a unit lasts four steps), all token
    // stages (but one when not pipelined)
    using H0 = std::integral_constant<int, 0>;
    using H1 = std::integral_constant<int, 1>;
    if(w_role)
    {
        auto units = [&](auto nt_tag) __attribute__((always_inline)) {
            static_for<(kPipe && !kXPair && !kW8) ? 5 : 4>([&](auto u_tag) __attribute__((always_inline)) {
                constexpr int u = decltype(u_tag)::value;
                using Half      = std::integral_constant<int, (u & 1)>;
                issue_w(u, Half{}, nt_tag);
            });
        };
        if(w_nt)
            units(std::true_type{});
        else
            units(std::false_type{});
    }
    else if constexpr(kXPair)
    {
        const int stages = x_stages(x_groups);
        for(int m = 0; m < stages; m++)
        {
            if(odd_k && m == kt_count >> 1)
                halve_x();
            issue_x_pair(m, m, x_groups);
        }
    }
    else
    {
        const int stages = x_stages(x_groups) - (kPipe ? 0 : 1);
        for(int x = 0; x < stages; x++)
            issue_x(x, x, x_groups);
    }

    // per-lane LDS read offsets (swizzled chunk positions are per-lane constants)
    const int sw_w  = (r32 >> 1) & 7; // 128-byte token rows of the gate+up GEMM
    const int w_row = chan_of_row(r32); // LDS row that holds the channel of this lane's MFMA row
    const int sw_wr = WPERM ? (w_row >> 4) & 1 : weight_row_swizzle(w_row);
    constexpr int kWChunkB = WPERM ? 128 : 16; // LDS bytes between two chunks of a weight row
    const int sw_x  = (r32 >> 2) & 3; // 64-byte token rows
    const int w_off = WPERM ? ((ww & 1) * 8 + (w_row >> 3)) * 1024 + (w_row & 7) * 16 : ((ww & 1) * 64 + w_row) * (2 * kStepKB);
    const int w_h   = ww >> 1;
    const int x_off = kXOffset + (wt * 32 + r32) * kStepKB;

    // NB: token blocks of this wave; XG: slab groups a token-role wave issues per step (0 in a weight-role wave)
    auto k_loop = [&](auto nb_tag, auto xg_tag, auto nt_tag) __attribute__((always_inline)) {
        constexpr int NB = decltype(nb_tag)::value;
        constexpr int XG = decltype(xg_tag)::value;
        constexpr int NF = NB > 0 ? NB : 1;
        // (a weight-role wave owns blocks 0, 2, .., as many as the tile has token groups)
        constexpr int kGroups = XG > 0 ? XG : NB > 0 ? NB : 1;
        constexpr int kXS     = x_stages(kGroups);
        if constexpr(kPipe)
        {
            // operand registers of the step about to run
            Frag wf[kSteps][2];
            Frag xf[kSteps][NF];
            // first step of the last window where only its second half is new (kOddW)
            [[maybe_unused]] const int half_from = kOddW && odd_k ? kt_count - (kW8 ? 2 : 1) : INT32_MAX;
            // weight fragment b of sub-step s of step kk (parity P), token fragment i of sub-step s of step kk
            auto load_wf = [&](int kk, auto p_tag, int s, int b) __attribute__((always_inline)) {
                constexpr int P          = decltype(p_tag)::value;
                constexpr int kh         = P * 4; // first chunk of the step inside the 128-byte weight row
                const unsigned char* wp  = lds + ((uint32_t)(big_pair_of_step(kk, kW8) + w_h) % kWS) * kWUnitBytes + w_off + b * 32 * (2 * kStepKB);
                const int cw_lo          = kOpB == 16 ? ((kh + 2 * s + kg) ^ sw_wr) * kWChunkB : ((kh + kg) ^ sw_wr) * kWChunkB;
                const int cw_hi          = ((kh + 2 + kg) ^ sw_wr) * kWChunkB;
                Frag f;
                if constexpr(kW8)
                {
                    // 8 int8 of this lane's K group, not converted yet: 16-byte chunk (kk & 3) * 2 + s of the row, half kg
                    const int q   = (kk >= half_from ? kk + 2 : kk) & 3;
                    const int c8  = (((q << 1) + s) ^ sw_wr) * kWChunkB + kg * 8;
                    const uint2 v = *reinterpret_cast<const uint2*>(wp + c8);
                    f.lo.x        = v.x;
                    f.lo.y        = v.y;
                    return f;
                }
                if constexpr(kOddW)
                {
                    f.lo = *reinterpret_cast<const uint4*>(wp + (cw_lo ^ (kk >= half_from ? 4 * kWChunkB : 0)));
                    return f;
                }
                f.lo = *reinterpret_cast<const uint4*>(wp + cw_lo);
                if constexpr(kOpB == 32)
                    f.hi = *reinterpret_cast<const uint4*>(wp + cw_hi);
                return f;
            };
            auto load_xf = [&](int kk, int s, int i) __attribute__((always_inline)) {
                Frag f;
                if constexpr(kXPair)
                {
                    const unsigned char* xp = lds + kXOffsetPair + ((uint32_t)(kk >> 1) % kXS) * pair_stage_bytes(kGroups) + (wt * 32 + r32 + i * 64) * (2 * kStepKB);
                    const int kh            = (kk & 1) * 4;
                    const int cx_lo         = kOpB == 16 ? ((kh + 2 * s + kg) ^ sw_w) * 16 : ((kh + kg) ^ sw_w) * 16;
                    const int cx_hi         = ((kh + 2 + kg) ^ sw_w) * 16;
                    f.lo                    = *reinterpret_cast<const uint4*>(xp + cx_lo);
                    if constexpr(kOpB == 32)
                        f.hi = *reinterpret_cast<const uint4*>(xp + cx_hi);
                }
                else
                {
                    const unsigned char* xp = lds + x_off + ((uint32_t)kk % kXS) * step_stage_bytes(kGroups) + i * 64 * kStepKB;
                    const int cx_lo         = kOpB == 16 ? ((2 * s + kg) ^ sw_x) * 16 : (kg ^ sw_x) * 16;
                    const int cx_hi         = ((2 + kg) ^ sw_x) * 16;
                    f.lo                    = *reinterpret_cast<const uint4*>(xp + cx_lo);
                    if constexpr(kOpB == 32)
                        f.hi = *reinterpret_cast<const uint4*>(xp + cx_hi);
                }
                return f;
            };
            // own transfers of the data named `need` have landed (the instructions issued after them may be
            // pending), everyone's are visible after the barrier, and nobody reads the buffers of the step before
            auto sync = [&](bool w_counted, bool x_counted, auto w_tag, auto x_tag) __attribute__((always_inline)) {
                if(w_role ? w_counted : x_counted)
                {
                    if(w_role)
                        wait_vmcnt<decltype(w_tag)::value>();
                    else
                        wait_vmcnt<decltype(x_tag)::value>();
                }
                else
                    wait_vmcnt<0>();
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // own operand fetches are complete
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
            };
            // step 0's data: weight units 0 and 1 (2, 3, 4 may be pending; with 128-byte token stages, or where a unit lasts
            // four steps, 2 and 3) and the first token stage (the others may be pending)
            const bool six = kt_count >= 6;
            if constexpr(kXPair)
                sync(six, kt_count >= 2 * kXS, std::integral_constant<int, 8>{}, std::integral_constant<int, 2 * XG * (kXS - 1)>{});
            else
                sync(kW8 ? n_wunits >= 4 : six, kt_count >= kXS, std::integral_constant<int, (kW8 ? 8 : 12)>{},
                     std::integral_constant<int, XG * (kXS - 1)>{});
            static_for<kSteps>([&](auto s_tag) __attribute__((always_inline)) {
                constexpr int s = decltype(s_tag)::value;
                wf[s][0]        = load_wf(0, H0{}, s, 0);
                wf[s][1]        = load_wf(0, H0{}, s, 1);
                if constexpr(kW8)
                {
                    wf[s][0].lo = int8x8_to_bf16x8(make_uint2(wf[s][0].lo.x, wf[s][0].lo.y));
                    wf[s][1].lo = int8x8_to_bf16x8(make_uint2(wf[s][1].lo.x, wf[s][1].lo.y));
                }
                static_for<NB>([&](auto i_tag) __attribute__((always_inline)) {
                    constexpr int i = decltype(i_tag)::value;
                    xf[s][i]        = load_xf(0, s, i);
                });
            });
            auto step = [&](int k, auto par_tag) __attribute__((always_inline)) {
                constexpr int PAR = decltype(par_tag)::value;
                using NPAR        = std::integral_constant<int, 1 - PAR>;
                // The barrier of step k guarantees step k+1: token step k+1 (the kXS - 2 after it may be pending) and the
                // weight pair of step k+1, that is units up to k+1 for even k (k+2 .. k+4 pending) or up to k+2 for odd k.
                // 128-byte token stages: a weight unit less is in flight (unit k+3 may be pending at odd k), and the
                // token pair of steps k+1 and k+2 is due at odd k (the kXS - 2 after it may be pending; at even k one more,
                // its pair was due the step before).
                // Steps 2 m and 2 m + 1 read the same weight pair and the same token stage, so only the barrier of
                // the odd step has anything to guarantee, and what the even step overwrites (the slot of weight unit
                // k - 1) was last read before the barrier of step k - 1: the even step has no barrier.
                // Measured: without it the bf16 and int8 GEMMs (two MFMA sub-steps per step) run 2 % faster, the fp8
                // GEMM (one) 5 % slower, so that one keeps it.
                // Units of int8 weights, one every other step and read for four: the pair of step k + 1 has landed once at most
                // two units are in flight, while there are later ones (big_units_may_fly).
                const bool counted = k + 4 < kt_count;
                if constexpr(kXPair)
                {
                    // (all of them have been issued if the last step is further off)
                    if constexpr(PAR == 1 || kSteps == 1)
                        sync(counted, k + 2 * kXS - 2 < kt_count, std::integral_constant<int, (PAR ? 4 : 8)>{},
                             std::integral_constant<int, 2 * XG * (kXS - (PAR ? 2 : 1))>{});
                }
                else if constexpr(kW8)
                    sync(big_units_may_fly(k + 1, kt_count, kW8), k + kXS <= kt_count, std::integral_constant<int, 8>{},
                         std::integral_constant<int, XG * (kXS - 2)>{});
                else
                    sync(counted, k + kXS <= kt_count, std::integral_constant<int, (PAR ? 8 : 12)>{},
                         std::integral_constant<int, XG * (kXS - 2)>{});
                // the transfers of the step go out behind the MFMAs of the second token block (measured: 1 to 2 %
                // faster than right after the barrier, where all eight waves queue up at the address unit while the
                // MFMA pipe has nothing to do; one instruction behind every block is 5 % slower)
                auto issue_next = [&]() __attribute__((always_inline)) {
                    if constexpr(kXPair)
                    {
                        // slot (k + 4) % 5 held unit k - 1, the stage of pair (k - 1) / 2 the tokens of steps k - 1 and k:
                        // both were last read during step k - 1, into registers, before this step's barrier
                        if(w_role)
                            issue_w(k + 4, par_tag, nt_tag);
                        else if constexpr(PAR == 1)
                            issue_x_pair(((k - 1) >> 1) + kXS, (uint32_t)((k - 1) >> 1) % kXS, XG);
                    }
                    else if(w_role)
                    {
                        if constexpr(!kW8)
                            issue_w(k + 5, NPAR{}, nt_tag);
                        else if constexpr(PAR == 0)
                            issue_w(big_unit_of_step(k, kW8), std::integral_constant<int, -1>{}, nt_tag);
                    }
                    else
                        issue_x(k + kXS, (uint32_t)k % kXS, XG);
                };
                constexpr int kIssueAfter = 1;
                if constexpr(NB <= kIssueAfter)
                    issue_next();
                static_for<kSteps>([&](auto s_tag) __attribute__((always_inline)) {
                    constexpr int s = decltype(s_tag)::value;
                    // int8 weights of the next step travel under this one's MFMAs and are converted behind them
                    [[maybe_unused]] Frag raw[2];
                    if constexpr(kW8)
                    {
                        raw[0] = load_wf(k + 1, NPAR{}, s, 0);
                        raw[1] = load_wf(k + 1, NPAR{}, s, 1);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    static_for<NB>([&](auto i_tag) __attribute__((always_inline)) {
                        constexpr int i = decltype(i_tag)::value;
                        if constexpr(MODE == kFp8 && GEMM0)
                        {
                            acc[i][0] = mfma_fp8_unscaled(wf[s][0], xf[s][i], acc[i][0]);
                            acc[i][1] = mfma_fp8_unscaled(wf[s][1], xf[s][i], acc[i][1]);
                        }
                        else
                        {
                            acc[i][0] = mfma<MODE>(wf[s][0], xf[s][i], 0u, acc[i][0]);
                            acc[i][1] = mfma<MODE>(wf[s][1], xf[s][i], 0u, acc[i][1]);
                        }
                        // the fragment's registers are free: fetch its successor (stale data after the last step)
                        __builtin_amdgcn_sched_barrier(0);
                        xf[s][i] = load_xf(k + 1, s, i);
                        if constexpr(NB > kIssueAfter && s == 0 && i == kIssueAfter)
                            issue_next();
                        __builtin_amdgcn_sched_barrier(0);
                    });
                    if constexpr(kW8)
                    {
                        wf[s][0].lo = int8x8_to_bf16x8(make_uint2(raw[0].lo.x, raw[0].lo.y));
                        wf[s][1].lo = int8x8_to_bf16x8(make_uint2(raw[1].lo.x, raw[1].lo.y));
                    }
                    else
                    {
                        wf[s][0] = load_wf(k + 1, NPAR{}, s, 0);
                        wf[s][1] = load_wf(k + 1, NPAR{}, s, 1);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
            };
            if constexpr(kOddK)
            {
                // the last window's units go out in steps kt_count - 5 and kt_count - 4 (rows of five steps or more: see
                // big_tile_supported) and its tokens in step kt_count - 2 kXS, each the wave's last: from there on the lanes of
                // the missing half fetch the other one
                int k   = 0;
                int end = !odd_k ? kt_count : kt_count - (w_role ? 5 : 2 * kXS + 1);
                for(;;)
                {
                    for(; k < end; k += 2)
                    {
                        step(k, H0{});
                        step(k + 1, H1{});
                    }
                    if(!odd_k || end == kt_count - 1)
                        break;
                    end = kt_count - 1;
                    if(w_role)
                    {
#pragma unroll
                        for(int j = 0; j < 4; j++)
                        {
                            const int rih   = (q4 + 4 * j) * 8 + (WPERM ? lane & 7 : lane >> 3);
                            const int chunk = WPERM ? (lane >> 3) ^ (((q4 + 4 * j) >> 1) & 1) : (lane & 7) ^ weight_row_swizzle(rih);
                            const uint32_t back = (chunk & 4) ? (WPERM ? 1024u : 64u) : 0u;
                            doff[j] -= back;
                            doff[4 + j] -= back;
                        }
                    }
                    else if(kt_count > 2 * kXS) // (otherwise the last pair has gone out already)
                        halve_x();
                }
                if(odd_k)
                    step(k, H0{});
                return;
            }
            if constexpr(kOddW && !kW8)
            {
                for(int k = 0; k + 1 < kt_count; k += 2)
                {
                    step(k, H0{});
                    step(k + 1, H1{});
                }
                if(odd_k)
                    step(kt_count - 1, H0{});
                return;
            }
            for(int k = 0; k < kt_count; k += 2)
            {
                step(k, H0{});
                step(k + 1, H1{});
            }
        }
        else
        {
            // fp8 down GEMM.  One compute step; PAR = k & 1
            auto step = [&](int k, auto par_tag) __attribute__((always_inline)) {
                constexpr int PAR = decltype(par_tag)::value;
                // Needed now: token step k and the weight units of pair k >> 1.  Issued after them and allowed to stay pending:
                // kXS - 2 token steps; two weight units (even k) or three (odd k), until the last pair is the one needed.
                if(w_role ? big_units_may_fly(k, kt_count, false) : k + kXS - 2 < kt_count)
                {
                    if(w_role)
                        wait_vmcnt<PAR ? 12 : 8>();
                    else
                        wait_vmcnt<(XG + 1) * (kXS - 2)>(); // token-role instructions of the steps after it
                }
                else
                    wait_vmcnt<0>();
                // data of step k visible to all waves; everyone is done reading step k-1 (a bare barrier:
                // the DMA completion was awaited above and LDS reads are consumed by MFMAs before a
                // wave gets here)
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                // The transfers of the step, whose buffers are free from the barrier on (behind the first MFMAs, as in the
                // pipelined loop, needs a scheduling fence for which there is no register to spare)
                if(w_role)
                    issue_w(big_unit_of_step(k, false), par_tag, nt_tag);
                else
                    issue_x(k + kXS - 1, (uint32_t)(k + kXS - 1) % kXS, XG);

                // first unit of the pair that holds this step's weight bytes
                const int pair0          = big_pair_of_step(k, false);
                const unsigned char* wst = lds + ((uint32_t)(pair0 + w_h) % kWSlots) * kWUnitBytes + w_off;
                const unsigned char* xst = lds + x_off + ((uint32_t)k % kXS) * step_stage_bytes(kGroups);
                const unsigned char* ysl = lds + ys_offset(kGroups) + ((uint32_t)k % kXS) * kYsStageBytes + kg * kYsRows + wt * 32 + r32;
                constexpr int kh         = PAR * 4; // first chunk of this step inside the 128-byte weight row
                Frag wf[2];
                Frag xf[NF];
                uint32_t xs[NF];
#pragma unroll
                for(int b = 0; b < 2; b++)
                {
                    const unsigned char* wp = wst + b * 32 * (2 * kStepKB);
                    wf[b].lo                = *reinterpret_cast<const uint4*>(wp + ((kh + kg) ^ sw_wr) * kWChunkB);
                    wf[b].hi                = *reinterpret_cast<const uint4*>(wp + ((kh + 2 + kg) ^ sw_wr) * kWChunkB);
                }
#pragma unroll
                for(int i = 0; i < NB; i++)
                {
                    const unsigned char* xp = xst + i * 64 * kStepKB;
                    xf[i].lo                = *reinterpret_cast<const uint4*>(xp + (kg ^ sw_x) * 16);
                    xf[i].hi                = *reinterpret_cast<const uint4*>(xp + ((2 + kg) ^ sw_x) * 16);
                    xs[i]                   = ysl[i * 64];
                }
#pragma unroll
                for(int i = 0; i < NB; i++)
                {
                    acc[i][0] = mfma<MODE>(wf[0], xf[i], xs[i], acc[i][0]);
                    acc[i][1] = mfma<MODE>(wf[1], xf[i], xs[i], acc[i][1]);
                }
            };
            for(int k = 0; k < kt_count; k += 2)
            {
                step(k, H0{});
                step(k + 1, H1{});
            }
        }
    };
    // weight-role waves own blocks 0, 2, .. (ceil(nmb / 2) of them), token-role waves blocks 1, 3, ..
    // (floor(nmb / 2)) and issue ceil(nmb / 2) slab groups: the same count, or one more when nmb is odd
    using I0 = std::integral_constant<int, 0>;
    auto run = [&](auto nb_tag) {
        constexpr int NB = decltype(nb_tag)::value;
        if(w_role && w_nt)
            k_loop(nb_tag, I0{}, std::true_type{});
        else if(w_role)
            k_loop(nb_tag, I0{}, std::false_type{});
        else if(x_groups == NB)
            k_loop(nb_tag, std::integral_constant<int, (NB > 0 ? NB : 1)>{}, std::false_type{});
        else
            k_loop(nb_tag, std::integral_constant<int, (NB < kMaxNB ? NB + 1 : kMaxNB)>{}, std::false_type{});
    };
    switch(nb_w)
    {
    case 5: run(std::integral_constant<int, 5>{}); break;
    case 4: run(std::integral_constant<int, 4>{}); break;
    case 3: run(std::integral_constant<int, 3>{}); break;
    case 2: run(std::integral_constant<int, 2>{}); break;
    case 1: run(std::integral_constant<int, 1>{}); break;
    default: run(std::integral_constant<int, 0>{}); break;
    }

    // ---- epilogue
    if constexpr(kEpi)
    {
        EpilogueOperands<kMaxNB> o;
        if(epi_lds)
        {
            o.cols = epilogue_columns<GEMM0>(p, n_base, ww, kg);
            // (rows of a column group the tile does not have hold another row's scale; nothing is stored for them)
            const float* sc = reinterpret_cast<const float*>(lds + kEpiChannels) + (paired ? ww * 32 : ww * 64) + 16 * kg;
            load_channel_scales(sc, o.sc0);
            load_channel_scales(sc + (paired ? 128 : 32), o.sc1);
#pragma unroll
            for(int i = 0; i < kMaxNB; i++)
            {
                const int r      = wt * 32 + i * 64 + r32;
                const int at     = min(min(r, nrows - 1), kEpiRows - 1);
                const int sid    = reinterpret_cast<const int*>(lds + kEpiIds)[at];
                o.rows.real[i]   = real_id(sid, p.tokens, p.topk);
                o.rows.sa[i]     = o.rows.real[i] ? reinterpret_cast<const float*>(lds + kEpiScales)[at] : 0.0f;
                o.rows.orow[i]   = p.slot_rows <= 0 ? row0 + r : o.rows.real[i] ? (int)slot_row(sid, p.slot_rows) : 0;
            }
        }
        else
            load_epilogue<MODE, GEMM0, kMaxNB>(p, o, expert, row0, nrows, wt * 32, 64, n_base, ww, r32, kg, slice);
        pin_epilogue(o);
        apply_epilogue<MODE, GEMM0, kMaxNB>(p, acc, o, row0, nrows, wt * 32, 64, nb_w, r32, kg, expert);
    }
    else
        run_epilogue<MODE, GEMM0, kMaxNB>(p, acc, expert, row0, nrows, wt * 32, 64, nb_w, n_base, ww, r32, kg, slice);
}

template <int MODE, bool GEMM0, bool WPERM>
int launch_big_w(const GemmParams& p, int max_tiles, hipStream_t stream)
{
    const size_t lds    = kLdsBytes;
    // the dynamic LDS limit is an attribute of the function on one device: set once per device, whichever host
    // thread gets there first (the others wait for it)
    static std::once_flag attr_once[64];
    int dev = 0;
    (void)hipGetDevice(&dev);
    hipError_t attr = hipSuccess;
    auto set_attr   = [&] {
        attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&moe_gemm_big_kernel<MODE, GEMM0, WPERM>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    };
    if(dev >= 0 && dev < 64)
        std::call_once(attr_once[dev], set_attr);
    else
        set_attr();
    MI355_HIP_TRY(attr);
    const int grid = round_up(max_tiles * p.n_ntiles, 256); // whole rounds of 32-item chunks over the 8 XCDs
    if(grid <= 0)
        return MI355_MOE_OK;
    KernelTimer timer(GEMM0 ? MI355_MOE_K_GEMM0 : MI355_MOE_K_GEMM1, stream);
    hipLaunchKernelGGL((moe_gemm_big_kernel<MODE, GEMM0, WPERM>), dim3(grid), dim3(kBigThreads), lds, stream, p);
    MI355_HIP_TRY(hipGetLastError());
    return MI355_MOE_OK;
}

template <int MODE, bool GEMM0>
int launch_big_t(const GemmParams& p, int max_tiles, hipStream_t stream)
{
    return p.w_permuted ? launch_big_w<MODE, GEMM0, true>(p, max_tiles, stream) : launch_big_w<MODE, GEMM0, false>(p, max_tiles, stream);
}

} // namespace

int big_tile_rows() { return kBigXRows; }

bool big_tile_supported(int prec, int k_bytes0, int k_bytes1, bool y_i8)
{
    // K in whole pairs of 64-byte steps; the int8 path's down GEMM in whole 64-byte pieces of its weight rows, two at
    // least (kOddW); the
    // 8-bit gate+up GEMM also in odd numbers of steps, from five on (kOddK)
    const bool k0_odd = k_bytes0 % (2 * kStepKB) == kStepKB && k_bytes0 >= 5 * kStepKB;
    if(prec == MI355_MOE_FP8 && k0_odd)
        return k_bytes1 % (2 * kStepKB) == 0;
    if(prec == MI355_MOE_INT8)
    {
        const int kw1 = y_i8 ? k_bytes1 : k_bytes1 / 2;
        return (k_bytes0 % (2 * kStepKB) == 0 || k0_odd) && kw1 % kStepKB == 0 && kw1 >= 2 * kStepKB;
    }
    return (prec == MI355_MOE_BF16 || prec == MI355_MOE_FP16 || prec == MI355_MOE_FP8) && k_bytes0 % (2 * kStepKB) == 0 &&
           k_bytes1 % (2 * kStepKB) == 0;
}

int launch_gemm_big(int prec, bool gemm0, const GemmParams& p, int max_tiles, hipStream_t stream, bool y_i8)
{
    if(prec == MI355_MOE_INT8 && !gemm0 && y_i8)
        return launch_big_t<kI8, false>(p, max_tiles, stream);
    if(prec == MI355_MOE_BF16)
        return gemm0 ? launch_big_t<kBf16, true>(p, max_tiles, stream) : launch_big_t<kBf16, false>(p, max_tiles, stream);
    if(prec == MI355_MOE_FP16)
        return gemm0 ? launch_big_t<kF16, true>(p, max_tiles, stream) : launch_big_t<kF16, false>(p, max_tiles, stream);
    if(prec == MI355_MOE_FP8)
        return gemm0 ? launch_big_t<kFp8, true>(p, max_tiles, stream) : launch_big_t<kFp8, false>(p, max_tiles, stream);
    if(prec == MI355_MOE_INT8)
        return gemm0 ? launch_big_t<kI8, true>(p, max_tiles, stream) : launch_big_t<kBf16W8, false>(p, max_tiles, stream);
    return fail(MI355_MOE_E_UNSUPPORTED, "no large-tile kernel for precision %d", prec);
}

} // namespace mi355
