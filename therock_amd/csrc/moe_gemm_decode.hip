// Grouped GEMM for decode-sized expert batches (one or two 32-row blocks per expert tile; gfx950).
//
// With a handful of tokens per expert the two GEMMs are pure weight streaming, and what decides
// the rate is the shape of the HBM requests: 128-byte pieces of 256 different rows (the tile shape
// of moe_gemm_kernel) reach about 5.3 TB/s on rows of 4 KB, 512 contiguous bytes per row about
// 6.9 TB/s.  So here a workgroup owns only 64 weight rows (gate+up GEMM: 32 gate + 32 up rows = 32 Y
// columns) and walks K in steps of 512 bytes per row.  The four waves split each step along K: wave
// w multiplies bytes [128 w, 128 w + 128) of every row with the matching token columns, and the four
// partial accumulators are added through LDS at the end (in wave order, so the result is
// deterministic).  Same MFMA orientation (weight rows on the M side), operand layouts and epilogues
// as moe_gemm_kernel; operand tiles are staged through LDS with the next step prefetched into
// registers, weights with non-temporal loads where the expert has a single row tile.  NXB = 2 multiplies every weight tile with two token
// blocks (tiles of up to 64 sorted rows), so that experts with 33 .. 64 rows still stream their
// weights once.
#include "moe_gemm_device.hpp"

#include <algorithm>
#include <type_traits>

namespace mi355 {
using namespace gemm;
namespace {

constexpr int kDecWRows = 64;  // weight rows per workgroup
constexpr int kDecWKB   = 512; // weight bytes per row and step

// How a tile's weights are fetched (the two walks of the tile): as data that only this workgroup reads, as data that others read
// too, or whichever the tile's entry says.
enum Weights
{
    kOnce,
    kSeveral,
    kByTile
};

template <int MODE, bool GEMM0, int NXB, bool WPERM, Weights WEIGHTS>
__device__ __attribute__((always_inline)) inline void decode_tile(const GemmParams p, const TileRef tile, unsigned char* lds)
{
#include "moe_gemm_decode_tile.inl"
}

template <int MODE, bool GEMM0, int NXB, bool WPERM>
__global__ __launch_bounds__(kBlock, (NXB > 1 || MODE == kBf16W8 || MODE == kFp8) ? 2 : 3) void moe_gemm_decode_kernel(const GemmParams p)
{
    extern __shared__ __align__(16) unsigned char lds[];
    // ---- work item (same XCD-aware order as moe_gemm_kernel)
    const TileRef tile = lookup_tile(p.tile_map, p.n_ntiles, p.max_tiles, blockIdx.x, p.tile_rows);
    if(!tile.ok)
        return;
    // Pre-shuffled weights, one token block: the two walks each have a tile to themselves.  In one tile, the other forms' way, they
    // take all 168 registers of three workgroups a compute unit and spill up to three more (8 to 16 bytes of scratch memory, which
    // every workgroup sets up); apart they take 164.  Passes over 8 bf16 experts 1024 x 1024, 8 / 20 / 33 tokens, together -> apart:
    // 28.0 -> 26.7, 27.7 -> 27.0, 27.8 -> 26.9 us; 128 experts 4096 x 1536: 256 Zipf-routed tokens in int8 230.9 -> 228.8, in bf16
    // 394.8 -> 390.9, 4 tokens in fp16 193.7 -> 192.8; 64 experts 4096 x 2048, 1 / 2 / 4 bf16 tokens 56.1 -> 55.6, 82.7 -> 83.2, 138.4 ->
    // 137.8.  The other forms spill nothing, and with a tile for each walk batches of two-block tiles were up to 2 % slower
    // (200 x 2 tokens of the small layer 29.7 -> 30.4 us).  They hold the text of the tile itself and not the function: through it
    // the compiler orders the same instructions otherwise (128 x 2 tokens of that layer 32.9 -> 33.2 us).
    if constexpr(WPERM && NXB == 1)
    {
        if(tile.expert_tiles == 1)
            decode_tile<MODE, GEMM0, NXB, WPERM, kOnce>(p, tile, lds);
        else
            decode_tile<MODE, GEMM0, NXB, WPERM, kSeveral>(p, tile, lds);
    }
    else
    {
        constexpr Weights WEIGHTS = kByTile;
#include "moe_gemm_decode_tile.inl"
    }
}

template <int MODE, bool GEMM0, int NXB, bool WPERM>
int launch_decode_w(const GemmParams& p, int max_tiles, hipStream_t stream)
{
    using MT            = ModeTraits<MODE>;
    constexpr int kXMul = MT::kXKB / MT::kWKB;
    constexpr size_t lds = kDecWRows * (kDecWKB + kPadB) + NXB * 32 * (kDecWKB * kXMul + kPadB);
    static_assert(3 * NXB * 2 * 16 * 64 * 4 <= lds, "the reduction buffer fits in the operand tiles");
    const int grid = round_up(max_tiles * p.n_ntiles, 8);
    if(grid <= 0)
        return MI355_MOE_OK;
    KernelTimer timer(GEMM0 ? MI355_MOE_K_GEMM0 : MI355_MOE_K_GEMM1, stream);
    if constexpr(lds > 64 * 1024)
    {
        // the dynamic LDS limit is an attribute of the function on one device: set once per device
        static bool attr_ok[64] = {};
        int dev = 0;
        (void)hipGetDevice(&dev);
        if(dev < 0 || dev >= 64 || !attr_ok[dev])
        {
            MI355_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(&moe_gemm_decode_kernel<MODE, GEMM0, NXB, WPERM>),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            if(dev >= 0 && dev < 64)
                attr_ok[dev] = true;
        }
    }
    hipLaunchKernelGGL((moe_gemm_decode_kernel<MODE, GEMM0, NXB, WPERM>), dim3(grid), dim3(kBlock), lds, stream, p);
    MI355_HIP_TRY(hipGetLastError());
    return MI355_MOE_OK;
}

template <int MODE, bool GEMM0, int NXB>
int launch_decode_n(const GemmParams& p, int max_tiles, hipStream_t stream)
{
    return p.w_permuted ? launch_decode_w<MODE, GEMM0, NXB, true>(p, max_tiles, stream)
                        : launch_decode_w<MODE, GEMM0, NXB, false>(p, max_tiles, stream);
}

// blocks: 32-row token blocks per tile (1 or 2)
template <int MODE, bool GEMM0>
int launch_decode_t(int blocks, const GemmParams& p, int max_tiles, hipStream_t stream)
{
    return blocks == 1 ? launch_decode_n<MODE, GEMM0, 1>(p, max_tiles, stream) : launch_decode_n<MODE, GEMM0, 2>(p, max_tiles, stream);
}

} // namespace

int decode_tile_cols(bool gemm0) { return gemm0 ? 32 : 64; }

// byte offsets inside the token buffer, Y and one expert's weights must fit 32 bits
bool decode_supported(int64_t x_bytes, int64_t y_bytes, int64_t w_expert_bytes)
{
    const int64_t lim = (int64_t)1 << 32;
    return x_bytes < lim && y_bytes < lim && w_expert_bytes < lim;
}

int launch_gemm_decode(int prec, bool gemm0, int blocks, const GemmParams& p, int max_tiles, hipStream_t stream, bool y_i8)
{
    if(blocks != 1 && blocks != 2)
        return fail(MI355_MOE_E_UNSUPPORTED, "decode kernel: %d token blocks per tile", blocks);
    const int b = blocks;
    if(prec == MI355_MOE_INT8 && !gemm0 && y_i8)
        return launch_decode_t<kI8, false>(b, p, max_tiles, stream);
    if(prec == MI355_MOE_BF16)
        return gemm0 ? launch_decode_t<kBf16, true>(b, p, max_tiles, stream) : launch_decode_t<kBf16, false>(b, p, max_tiles, stream);
    if(prec == MI355_MOE_FP16)
        return gemm0 ? launch_decode_t<kF16, true>(b, p, max_tiles, stream) : launch_decode_t<kF16, false>(b, p, max_tiles, stream);
    if(prec == MI355_MOE_FP8 && b == 1) // (with two token blocks the fp8 kernels spill and the other families are faster)
        return gemm0 ? launch_decode_n<kFp8, true, 1>(p, max_tiles, stream) : launch_decode_n<kFp8, false, 1>(p, max_tiles, stream);
    if(prec == MI355_MOE_INT8 && gemm0)
        return launch_decode_t<kI8, true>(b, p, max_tiles, stream);
    if(prec == MI355_MOE_INT8 && b == 1) // (two token blocks of bf16 Y per int8 weight tile do not fit the register budget)
        return launch_decode_n<kBf16W8, false, 1>(p, max_tiles, stream);
    return fail(MI355_MOE_E_UNSUPPORTED, "no decode kernel for precision %d with %d token blocks per tile", prec, b);
}

} // namespace mi355
