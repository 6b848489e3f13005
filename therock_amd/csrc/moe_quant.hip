// Data-preparation kernels around the fused-MoE GEMMs for gfx950: per-row dynamic quantisation, ck_tile's
// MoE smooth-quant, and the conversion to and from ck_tile's pre-shuffled weight layout.  All of them are
// HBM-bound byte movers: one pass over the input, coalesced 16-byte accesses, no LDS beyond the row reductions.
#include "moe_gemm_device.hpp"

#include <algorithm>
#include <type_traits>

namespace mi355 {
using namespace gemm;
namespace {

// one value -> e4m3 (round to nearest even, saturating) or int8 (saturate, then ck_tile's float -> int8
// static_cast: truncation toward zero)
template <bool FP8>
__device__ inline unsigned char quantise_one(float v)
{
    if constexpr(FP8)
    {
        const float cl = fminf(fmaxf(v, -448.f), 448.f);
        return static_cast<unsigned char>(__builtin_amdgcn_cvt_pk_fp8_f32(cl, cl, 0, false) & 0xff);
    }
    else
    {
        const float cl = fminf(fmaxf(v, -128.f), 127.f);
        return static_cast<unsigned char>(static_cast<signed char>(static_cast<int>(cl)));
    }
}

// Four integers -> their low bytes in one dword.
__device__ inline uint32_t pack_low_bytes(int a, int b, int c, int d)
{
    const uint32_t ab = __builtin_amdgcn_perm(static_cast<uint32_t>(b), static_cast<uint32_t>(a), 0x0c0c0400u);
    const uint32_t cd = __builtin_amdgcn_perm(static_cast<uint32_t>(d), static_cast<uint32_t>(c), 0x04000c0cu);
    return ab | cd;
}

// A row's quantisation by its largest magnitude.  scale() is what the codes stand for: amax / qmax, 1 for a row of zeros.
// lo and hi bracket its reciprocal: v_rcp_f32 is within 1 ulp and the roundings that follow (of the scale itself, the two
// products here and the one with the element) add 2^-22 at most, so that x * lo and x * hi enclose fp32(x / scale()), and with
// them every monotone conversion of it.  Outside the range where none of these can overflow or lose bits to subnormals
// (rows of zeros and infinities among them) both are NaN.
template <bool FP8>
struct RowScale
{
    static constexpr float kMax = FP8 ? 448.0f : 127.0f;
    float amax, lo, hi;
    __device__ explicit RowScale(float m) : amax(m)
    {
        const float r = m >= 0x1p-100f && m <= 0x1p100f ? kMax * __builtin_amdgcn_rcpf(m) : __builtin_nanf("");
        lo            = r * (1.0f - 0x1p-20f);
        hi            = r * (1.0f + 0x1p-20f);
    }
    __device__ float scale() const { return amax > 0.f ? amax / kMax : 1.0f; }
};

__device__ inline uint32_t fp8x4(float a, float b, float c, float d)
{
    const int w = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
    return static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(c, d, w, true));
}

// v_cvt_i32_f32: toward zero, saturating, 0 for a NaN (which the language leaves undefined)
__device__ inline int float_to_int(float v)
{
    int r;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

// Eight codes in two dwords, each from the quotient rounded like the division; NEAREST: int8 codes rounded to nearest even
// instead of toward zero.
template <bool FP8, bool NEAREST>
__device__ inline uint2 exact_codes_8(const float (&o)[8], double s_rcp)
{
    float q[8];
#pragma unroll
    for(int i = 0; i < 8; i++)
        q[i] = div_by_row_scale(o[i], s_rcp);
    if constexpr(FP8)
    {
#pragma unroll
        for(int i = 0; i < 8; i++)
            q[i] = fminf(fmaxf(q[i], -448.f), 448.f);
        return make_uint2(fp8x4(q[0], q[1], q[2], q[3]), fp8x4(q[4], q[5], q[6], q[7]));
    }
    else
    {
        int c[8];
#pragma unroll
        for(int i = 0; i < 8; i++)
            c[i] = NEAREST ? float_to_int(__builtin_rintf(q[i])) : static_cast<int>(static_cast<signed char>(quantise_one<false>(q[i])));
        return make_uint2(pack_low_bytes(c[0], c[1], c[2], c[3]), pack_low_bytes(c[4], c[5], c[6], c[7]));
    }
}

// The same codes.  A code is right where both ends of the bracket give it, which fails for one quotient in some 2^14 (those
// within 2^-20 of a code's boundary): one piece of eight in 2000 is done again with the fp64 product that rounds like the
// division, and, with codes rounded toward zero, the piece that holds the row's maximum, whose quotient is 127 itself.
// That product, two conversions at a quarter of the fp32 rate, was most of these kernels' instructions.
// A NaN becomes -128 and 0 (e4m3: -448 and NaN) at the two ends, so it goes to the exact form too.  Codes rounded to nearest
// are the low bytes of x * lo + 1.5 * 2^23, one fused instruction that rounds the product to an integer; a NaN, or a row whose
// bracket is one, shows in the sum of x * 0 there.
// Used where a thread has one or two pieces (up to four in the re-quantisation), which are then in registers for the exact
// form as well; with more, the branch costs more than it saves (see kBracketCols).
template <bool FP8, bool NEAREST = false>
__device__ inline uint2 quantise_8(const float (&o)[8], const RowScale<FP8>& row)
{
    uint2 lo, hi;
    float bad = !FP8 && NEAREST ? row.lo : 0.0f;
    if constexpr(FP8)
    {
        float l[8], h[8];
#pragma unroll
        for(int i = 0; i < 8; i++)
        {
            l[i] = __builtin_amdgcn_fmed3f(o[i] * row.lo, -448.f, 448.f);
            h[i] = o[i] * row.hi;
        }
        lo = make_uint2(fp8x4(l[0], l[1], l[2], l[3]), fp8x4(l[4], l[5], l[6], l[7]));
        hi = make_uint2(fp8x4(h[0], h[1], h[2], h[3]), fp8x4(h[4], h[5], h[6], h[7]));
    }
    else
    {
        int l[8], h[8];
#pragma unroll
        for(int i = 0; i < 8; i++)
        {
            if constexpr(NEAREST)
            {
                l[i] = __float_as_int(fmaf(o[i], row.lo, 0x1.8p23f));
                h[i] = __float_as_int(fmaf(o[i], row.hi, 0x1.8p23f));
                bad  = fmaf(o[i], 0.0f, bad);
            }
            else
            {
                l[i] = static_cast<int>(__builtin_amdgcn_fmed3f(o[i] * row.lo, -128.f, 127.f));
                h[i] = float_to_int(o[i] * row.hi);
            }
        }
        lo = make_uint2(pack_low_bytes(l[0], l[1], l[2], l[3]), pack_low_bytes(l[4], l[5], l[6], l[7]));
        hi = make_uint2(pack_low_bytes(h[0], h[1], h[2], h[3]), pack_low_bytes(h[4], h[5], h[6], h[7]));
    }
    if(((lo.x ^ hi.x) | (lo.y ^ hi.y)) != 0 || bad != bad)
        lo = exact_codes_8<FP8, NEAREST>(o, row_reciprocal(row.scale()));
    return lo;
}

// eight bf16 in four dwords -> fp32
__device__ inline void unpack_bf16x8(const uint4& r, float (&o)[8])
{
    const uint32_t d[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for(int i = 0; i < 4; i++)
    {
        o[2 * i]     = __uint_as_float(d[i] << 16);
        o[2 * i + 1] = __uint_as_float(d[i] & 0xffff0000u);
    }
}

template <int WAVES = 4>
__device__ inline float block_max(float v, float* s_red)
{
    v = wave_reduce_max(v, 0.f);
    if((threadIdx.x & 63) == 0)
        s_red[threadIdx.x >> 6] = v;
    __syncthreads();
    float m = s_red[0];
#pragma unroll
    for(int w = 1; w < WAVES; w++)
        m = fmaxf(m, s_red[w]);
    return m;
}

// Per-row dynamic quantisation of one row by one 256-thread workgroup: xr bf16 (times sr fp32 when SMOOTH),
// scale = amax / qmax, q = quantise(value / scale).  With VEC the row is walked in 16-byte pieces of 8 elements
// (cols % 8 == 0, 16-byte aligned rows); the first kCache pieces of every thread stay in registers between the
// two passes, so rows of up to 8192 columns are read once.  Returns the row's amax to every thread.
constexpr int kQuantCache = 4;
// Rows of up to two pieces a thread take their codes from the bracket, longer ones the exact quotients.  Exact -> bracket, us:
// 32768 rows of 1024 / 4096, int8 37.0 -> 32.6 / 77.1 -> 67.8, e4m3 35.2 -> 26.6 / 75.8 -> 67.4; 8192 rows of 7168, int8 28.1 -> 29.3, e4m3
// 27.5 -> 28.8; 3001 x 8 smooth-quantised rows of 7168 grouped by expert, int8 80 -> 92, e4m3 72 -> 83 (with the exact ones
// fewer registers, too: four waves per SIMD instead of three).  These are of calls repeated on one input; within a pass over more
// data than the caches hold, the 8192 e4m3 rows of 7168 take 37.7 -> 35.3 (0.07 % of that pass).
constexpr int kBracketCols = 2 * 256 * 8;
template <bool FP8, bool SMOOTH, bool VEC, bool BRACKET>
__device__ inline float quantise_row(const uint16_t* __restrict__ xr, const float* __restrict__ sr, int cols,
                                     unsigned char* __restrict__ qr, float* s_red, bool unit_scale_when_zero, float* scale_out)
{
    const float qmx = FP8 ? 448.0f : 127.0f;
    if constexpr(VEC)
    {
        const int chunks = cols >> 3;
        float v[kQuantCache][8];
        auto load = [&](int c, float (&o)[8]) {
            const uint4 r = *reinterpret_cast<const uint4*>(xr + c * 8);
            const uint32_t d[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
            for(int i = 0; i < 4; i++)
            {
                o[2 * i]     = __uint_as_float(d[i] << 16);
                o[2 * i + 1] = __uint_as_float(d[i] & 0xffff0000u);
            }
            if constexpr(SMOOTH)
            {
                const float4 s0 = *reinterpret_cast<const float4*>(sr + c * 8);
                const float4 s1 = *reinterpret_cast<const float4*>(sr + c * 8 + 4);
                o[0] *= s0.x; o[1] *= s0.y; o[2] *= s0.z; o[3] *= s0.w;
                o[4] *= s1.x; o[5] *= s1.y; o[6] *= s1.z; o[7] *= s1.w;
            }
        };
        float amax = 0.f;
#pragma unroll
        for(int j = 0; j < kQuantCache; j++)
        {
            const int c = threadIdx.x + 256 * j;
            if(c < chunks)
            {
                load(c, v[j]);
#pragma unroll
                for(int i = 0; i < 8; i++)
                    amax = fmaxf(amax, fabsf(v[j][i]));
            }
        }
        for(int c = threadIdx.x + 256 * kQuantCache; c < chunks; c += 256)
        {
            float t[8];
            load(c, t);
#pragma unroll
            for(int i = 0; i < 8; i++)
                amax = fmaxf(amax, fabsf(t[i]));
        }
        amax          = block_max(amax, s_red);
        // a row of zeros: the scale written is 1 (row-wise quant) or 0 (smooth-quant, as amax / qmax gives);
        // either way the row's codes are 0, never the 0 / 0 the plain formula would convert
        if(threadIdx.x == 0)
            *scale_out = (amax > 0.f || !unit_scale_when_zero) ? amax / qmx : 1.0f;
        const RowScale<FP8> row(amax);
        const double s_rcp = row_reciprocal(row.scale());
        auto store = [&](int c, const float (&o)[8]) {
            *reinterpret_cast<uint2*>(qr + c * 8) = BRACKET ? quantise_8<FP8>(o, row) : exact_codes_8<FP8, false>(o, s_rcp);
        };
#pragma unroll
        for(int j = 0; j < kQuantCache; j++)
        {
            const int c = threadIdx.x + 256 * j;
            if(c < chunks)
                store(c, v[j]);
        }
        for(int c = threadIdx.x + 256 * kQuantCache; c < chunks; c += 256)
        {
            float t[8];
            load(c, t);
            store(c, t);
        }
        return amax;
    }
    else
    {
        float amax = 0.f;
        for(int c = threadIdx.x; c < cols; c += 256)
            amax = fmaxf(amax, fabsf(bf16_bits_to_float(xr[c]) * (SMOOTH ? sr[c] : 1.0f)));
        amax          = block_max(amax, s_red);
        // a row of zeros: the scale written is 1 (row-wise quant) or 0 (smooth-quant, as amax / qmax gives);
        // either way the row's codes are 0, never the 0 / 0 the plain formula would convert
        const float s_out = (amax > 0.f || !unit_scale_when_zero) ? amax / qmx : 1.0f;
        const float s     = amax > 0.f ? s_out : 1.0f;
        if(threadIdx.x == 0)
            *scale_out = s_out;
        const double s_rcp = row_reciprocal(s);
        for(int c = threadIdx.x; c < cols; c += 256)
            qr[c] = quantise_one<FP8>(div_by_row_scale(bf16_bits_to_float(xr[c]) * (SMOOTH ? sr[c] : 1.0f), s_rcp));
        return amax;
    }
}

// per-row dynamic quantisation bf16 -> e4m3 / int8
template <bool FP8, bool VEC, bool BRACKET>
__global__ __launch_bounds__(256) void rowwise_quant_kernel(const uint16_t* __restrict__ x, int cols,
                                                             int64_t stride_x, unsigned char* __restrict__ q,
                                                             float* __restrict__ scale)
{
    __shared__ float s_red[4];
    const int64_t row = blockIdx.x;
    quantise_row<FP8, false, VEC, BRACKET>(x + row * stride_x, nullptr, cols, q + row * cols, s_red, true, scale + row);
}

// The vector form of many short rows: a wave each, four to a workgroup, as 256 threads have half a piece or one each and as long
// a chain of reductions.  Few rows are left to workgroups, whose lanes have fewer pieces one after the other.  Workgroup -> wave, us:
// 24000 rows of 512 / 1024 / 2048 columns, int8 21.2 -> 11.4, 24.7 -> 15.5, 30.1 -> 27.5, e4m3 18.1 -> 9.7, 21.5 -> 14.2, 27.4 -> 27.1;
// 1024 rows 2.6 -> 2.5, 2.9 -> 2.8, 3.5 -> 3.5; 256 rows 2.4 -> 2.5, 2.4 -> 2.7, 2.5 -> 3.3.  Smooth-quant with 4 slots, 24000 tokens,
// int8 75 -> 33, 92 -> 47, 114 -> 80; 1024 tokens 6.2 -> 5.1, 7.4 -> 6.0, 8.8 -> 8.5.
constexpr int kWaveCols = 8 * 64 * kQuantCache;
inline bool wave_per_row(int64_t rows, int cols) { return cols <= kWaveCols && rows >= cols; }
template <bool FP8>
__global__ __launch_bounds__(256) void rowwise_quant_wave_kernel(const uint16_t* __restrict__ x, int cols, int64_t stride_x,
                                                                  unsigned char* __restrict__ q, float* __restrict__ scale, int rows)
{
    const int lane = threadIdx.x & 63;
    const int row  = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); // (uniform)
    if(row >= rows)
        return;
    const int chunks   = cols >> 3;
    const uint16_t* xr = x + row * stride_x;
    float v[kQuantCache][8];
    float amax = 0.f;
#pragma unroll
    for(int j = 0; j < kQuantCache; j++)
        if(lane + 64 * j < chunks)
            unpack_bf16x8(*reinterpret_cast<const uint4*>(xr + (lane + 64 * j) * 8), v[j]);
#pragma unroll
    for(int j = 0; j < kQuantCache; j++)
        if(lane + 64 * j < chunks)
#pragma unroll
            for(int i = 0; i < 8; i++)
                amax = fmaxf(amax, fabsf(v[j][i]));
    amax = wave_reduce_max(amax, 0.f);
    const RowScale<FP8> rs(amax);
    if(lane == 0)
        scale[row] = rs.scale();
#pragma unroll
    for(int j = 0; j < kQuantCache; j++)
        if(lane + 64 * j < chunks)
            *reinterpret_cast<uint2*>(q + (int64_t)row * cols + (lane + 64 * j) * 8) = quantise_8<FP8>(v[j], rs);
}

// MoE smooth-quant: row (slot k, token t) = x[t, :] * smscale[expert(t, k), :], per-row dynamic quantisation.
// Scalar form: one workgroup per (token, slot).
template <bool FP8>
__global__ __launch_bounds__(256) void moe_smoothquant_kernel(const uint16_t* __restrict__ x,
                                                               const float* __restrict__ smscale,
                                                               const int* __restrict__ topk_ids, int tokens, int hidden,
                                                               int experts, int topk, int64_t x_stride, int64_t y_stride,
                                                               unsigned char* __restrict__ qy, float* __restrict__ yscale)
{
    __shared__ float s_red[4];
    const int t = blockIdx.x;
    const int k = blockIdx.y;
    int e       = topk_ids[(int64_t)t * topk + k];
    e           = min(max(e, 0), experts - 1);
    const int64_t r = (int64_t)k * tokens + t;
    quantise_row<FP8, true, false, false>(x + (int64_t)t * x_stride, smscale + (int64_t)e * hidden, hidden, qy + r * y_stride, s_red,
                                   false, yscale + r);
}

// Vector form (hidden % 8 == 0, aligned rows): one workgroup (LANES 256) or wave (64: short rows, up to PIECES pieces a lane) per
// token walks its slots, so the token's row is read once (its first PIECES pieces per thread stay in registers) and only the
// experts' smooth scales and the quantised rows move per slot.
template <bool FP8, int PIECES, int LANES>
__global__ __launch_bounds__(256) void moe_smoothquant_vec_kernel(const uint16_t* __restrict__ x,
                                                                   const float* __restrict__ smscale,
                                                                   const int* __restrict__ topk_ids, int tokens,
                                                                   int hidden, int experts, int topk, int64_t x_stride,
                                                                   int64_t y_stride, unsigned char* __restrict__ qy,
                                                                   float* __restrict__ yscale)
{
    constexpr bool kMore = LANES == 256 && PIECES == kQuantCache; // a row may have more pieces than its threads hold
    __shared__ float s_red[2][4];
    const int lane = threadIdx.x & (LANES - 1);
    const int t    = LANES == 256 ? blockIdx.x : blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); // (uniform)
    if(LANES < 256 && t >= tokens)
        return;
    const uint16_t* xr = x + (int64_t)t * x_stride;
    const int chunks   = hidden >> 3;
    const float qmx    = FP8 ? 448.0f : 127.0f;
    auto load_x = [&](int c, float (&o)[8]) {
        unpack_bf16x8(*reinterpret_cast<const uint4*>(xr + c * 8), o);
    };
    auto times_sm = [&](const float* sr, int c, const float (&in)[8], float (&o)[8]) {
        const float4 s0 = *reinterpret_cast<const float4*>(sr + c * 8);
        const float4 s1 = *reinterpret_cast<const float4*>(sr + c * 8 + 4);
        o[0] = in[0] * s0.x; o[1] = in[1] * s0.y; o[2] = in[2] * s0.z; o[3] = in[3] * s0.w;
        o[4] = in[4] * s1.x; o[5] = in[5] * s1.y; o[6] = in[6] * s1.z; o[7] = in[7] * s1.w;
    };
    auto scales_of_slot = [&](int k) {
        const int e = topk_ids[(int64_t)t * topk + k];
        return smscale + (int64_t)min(max(e, 0), experts - 1) * hidden;
    };
    // the smooth scales of the cached pieces, for the slot about to be processed: fetched one slot ahead, so that
    // their latency passes under the previous slot's reduction, conversions and stores
    float4 sm[PIECES][2];
    auto fetch_scales = [&](const float* sr) {
#pragma unroll
        for(int j = 0; j < PIECES; j++)
            if(lane + LANES * j < chunks)
            {
                sm[j][0] = *reinterpret_cast<const float4*>(sr + (lane + LANES * j) * 8);
                sm[j][1] = *reinterpret_cast<const float4*>(sr + (lane + LANES * j) * 8 + 4);
            }
    };
    float xv[PIECES][8];
#pragma unroll
    for(int j = 0; j < PIECES; j++)
        if(lane + LANES * j < chunks)
            load_x(lane + LANES * j, xv[j]);
    if(topk > 0)
        fetch_scales(scales_of_slot(0));
    for(int k = 0; k < topk; k++)
    {
        const float* sr = scales_of_slot(k);
        float v[PIECES][8];
        float amax = 0.f;
#pragma unroll
        for(int j = 0; j < PIECES; j++)
        {
            const int c = lane + LANES * j;
            if(c < chunks)
            {
                const float4 s0 = sm[j][0], s1 = sm[j][1];
                v[j][0] = xv[j][0] * s0.x; v[j][1] = xv[j][1] * s0.y; v[j][2] = xv[j][2] * s0.z; v[j][3] = xv[j][3] * s0.w;
                v[j][4] = xv[j][4] * s1.x; v[j][5] = xv[j][5] * s1.y; v[j][6] = xv[j][6] * s1.z; v[j][7] = xv[j][7] * s1.w;
#pragma unroll
                for(int i = 0; i < 8; i++)
                    amax = fmaxf(amax, fabsf(v[j][i]));
            }
        }
        if(k + 1 < topk)
            fetch_scales(scales_of_slot(k + 1));
        for(int c = lane + LANES * PIECES; kMore && c < chunks; c += LANES)
        {
            float a[8], b[8];
            load_x(c, a);
            times_sm(sr, c, a, b);
#pragma unroll
            for(int i = 0; i < 8; i++)
                amax = fmaxf(amax, fabsf(b[i]));
        }
        if constexpr(LANES == 256)
            amax = block_max(amax, s_red[k & 1]); // two buffers: one barrier per slot suffices
        else
            amax = wave_reduce_max(amax, 0.f);
        const int64_t r = (int64_t)k * tokens + t;
        if(lane == 0)
            yscale[r] = amax / qmx; // (a row of zeros: scale 0, codes 0)
        unsigned char* qr = qy + r * y_stride;
        const RowScale<FP8> row(amax);
        [[maybe_unused]] const double s_rcp = row_reciprocal(row.scale());
        // (streaming stores: the quantised rows are written once and should not push the experts' scales out of L2)
        auto store = [&](int c, const float (&o)[8]) {
            typedef __attribute__((ext_vector_type(2))) unsigned u32x2_t;
            uint2 q;
            if constexpr(kMore)
                q = exact_codes_8<FP8, false>(o, s_rcp);
            else
                q = quantise_8<FP8>(o, row);
            __builtin_nontemporal_store(u32x2_t{q.x, q.y}, reinterpret_cast<u32x2_t*>(qr + c * 8));
        };
#pragma unroll
        for(int j = 0; j < PIECES; j++)
            if(lane + LANES * j < chunks)
                store(lane + LANES * j, v[j]);
        for(int c = lane + LANES * PIECES; kMore && c < chunks; c += LANES)
        {
            float a[8], b[8];
            load_x(c, a);
            times_sm(sr, c, a, b);
            store(c, b);
        }
    }
}

// Expert-grouped form, for expert tables that do not stay in an XCD's L2 beside the rows streaming through it
// (256 experts x 7168 columns of fp32 are 7.3 MB against 4 MB): a workgroup owns one expert and one range of
// kSqRange tokens.  It keeps the expert's smooth scales in registers (read once per workgroup instead of once per
// row), finds the range's routing entries that name its expert, and quantises those rows one after the other, the
// next row's activations fetched while the current one is reduced and stored.  The workgroups of one token range sit
// on one XCD and run together there (workgroup ids go round the eight XCDs: id = (range / 8 * experts + expert) * 8 +
// range % 8), so that the range's activations come from HBM once and from that XCD's L2 for the other slots.  Each row
// is computed by the same expressions as in the per-token form: the results are the same bits.
constexpr int kSqRange   = 128;  // tokens per range
constexpr int kSqMaxList = 8192; // routing entries of a range (kSqRange x topk)
template <bool FP8, int PIECES>
__global__ __launch_bounds__(256) void moe_smoothquant_grouped_kernel(const uint16_t* __restrict__ x,
                                                                       const float* __restrict__ smscale,
                                                                       const int* __restrict__ topk_ids, int tokens,
                                                                       int hidden, int experts, int topk, int64_t x_stride,
                                                                       int64_t y_stride, unsigned char* __restrict__ qy,
                                                                       float* __restrict__ yscale)
{
    __shared__ float s_red[2][4];
    __shared__ int s_count;
    __shared__ int s_list[kSqMaxList];
    const int xcd   = blockIdx.x & 7;
    const int e     = (blockIdx.x >> 3) % experts;
    const int range = (blockIdx.x >> 3) / experts * 8 + xcd;
    const int t0    = range * kSqRange;
    if(t0 >= tokens)
        return;
    const int nt     = min(kSqRange, tokens - t0);
    const int chunks = hidden >> 3;
    const float qmx  = FP8 ? 448.0f : 127.0f;
    if(threadIdx.x == 0)
        s_count = 0;
    __syncthreads();
    // entries of the range that name this expert (ids outside [0, experts) are clamped like in the other forms)
    const int* ids = topk_ids + (int64_t)t0 * topk;
    for(int i = threadIdx.x; i < nt * topk; i += 256)
        if(min(max(ids[i], 0), experts - 1) == e)
            s_list[atomicAdd(&s_count, 1)] = i;
    __syncthreads();
    const int n = s_count;
    if(n == 0)
        return;
    const float* sr = smscale + (int64_t)e * hidden;
    float4 sm[PIECES][2];
#pragma unroll
    for(int j = 0; j < PIECES; j++)
        if(threadIdx.x + 256 * j < chunks)
        {
            sm[j][0] = *reinterpret_cast<const float4*>(sr + (threadIdx.x + 256 * j) * 8);
            sm[j][1] = *reinterpret_cast<const float4*>(sr + (threadIdx.x + 256 * j) * 8 + 4);
        }
    auto unpack = [&](const uint4& r, float (&o)[8]) {
        const uint32_t d[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
        for(int i = 0; i < 4; i++)
        {
            o[2 * i]     = __uint_as_float(d[i] << 16);
            o[2 * i + 1] = __uint_as_float(d[i] & 0xffff0000u);
        }
    };
    auto times_sm = [&](int c, const float (&in)[8], float (&o)[8]) {
        const float4 s0 = *reinterpret_cast<const float4*>(sr + c * 8);
        const float4 s1 = *reinterpret_cast<const float4*>(sr + c * 8 + 4);
        o[0] = in[0] * s0.x; o[1] = in[1] * s0.y; o[2] = in[2] * s0.z; o[3] = in[3] * s0.w;
        o[4] = in[4] * s1.x; o[5] = in[5] * s1.y; o[6] = in[6] * s1.z; o[7] = in[7] * s1.w;
    };
    uint4 raw[PIECES];
    auto fetch_row = [&](int entry) {
        const uint16_t* xr = x + (int64_t)(t0 + entry / topk) * x_stride;
#pragma unroll
        for(int j = 0; j < PIECES; j++)
            if(threadIdx.x + 256 * j < chunks)
                raw[j] = *reinterpret_cast<const uint4*>(xr + (threadIdx.x + 256 * j) * 8);
    };
    fetch_row(s_list[0]);
    for(int m = 0; m < n; m++)
    {
        const int entry    = s_list[m];
        const int t        = t0 + entry / topk;
        const int k        = entry - (entry / topk) * topk;
        const uint16_t* xr = x + (int64_t)t * x_stride;
        float v[PIECES][8];
        float amax = 0.f;
#pragma unroll
        for(int j = 0; j < PIECES; j++)
            if(threadIdx.x + 256 * j < chunks)
            {
                float xv[8];
                unpack(raw[j], xv);
                const float4 s0 = sm[j][0], s1 = sm[j][1];
                v[j][0] = xv[0] * s0.x; v[j][1] = xv[1] * s0.y; v[j][2] = xv[2] * s0.z; v[j][3] = xv[3] * s0.w;
                v[j][4] = xv[4] * s1.x; v[j][5] = xv[5] * s1.y; v[j][6] = xv[6] * s1.z; v[j][7] = xv[7] * s1.w;
#pragma unroll
                for(int i = 0; i < 8; i++)
                    amax = fmaxf(amax, fabsf(v[j][i]));
            }
        if(m + 1 < n)
            fetch_row(s_list[m + 1]);
        for(int c = threadIdx.x + 256 * PIECES; PIECES == kQuantCache && c < chunks; c += 256)
        {
            float a[8], b[8];
            unpack(*reinterpret_cast<const uint4*>(xr + c * 8), a);
            times_sm(c, a, b);
#pragma unroll
            for(int i = 0; i < 8; i++)
                amax = fmaxf(amax, fabsf(b[i]));
        }
        amax               = block_max(amax, s_red[m & 1]); // two buffers: one barrier per row suffices
        const int64_t r = (int64_t)k * tokens + t;
        if(threadIdx.x == 0)
            yscale[r] = amax / qmx; // (a row of zeros: scale 0, codes 0)
        unsigned char* qr   = qy + r * y_stride;
        const RowScale<FP8> row(amax);
        [[maybe_unused]] const double s_rcp = row_reciprocal(row.scale());
        auto store = [&](int c, const float (&o)[8]) {
            typedef __attribute__((ext_vector_type(2))) unsigned u32x2_t;
            uint2 q;
            if constexpr(PIECES == kQuantCache)
                q = exact_codes_8<FP8, false>(o, s_rcp);
            else
                q = quantise_8<FP8>(o, row);
            __builtin_nontemporal_store(u32x2_t{q.x, q.y}, reinterpret_cast<u32x2_t*>(qr + c * 8));
        };
#pragma unroll
        for(int j = 0; j < PIECES; j++)
            if(threadIdx.x + 256 * j < chunks)
                store(threadIdx.x + 256 * j, v[j]);
        for(int c = threadIdx.x + 256 * PIECES; PIECES == kQuantCache && c < chunks; c += 256)
        {
            float a[8], b[8];
            unpack(*reinterpret_cast<const uint4*>(xr + c * 8), a);
            times_sm(c, a, b);
            store(c, b);
        }
    }
}

// Re-quantisation of the intermediate activations between the two GEMMs of the int8 path (fused_quant 1 / 2 of
// ck_tile's fused_moe_traits; y_smooth_scale of FusedMoeGemmHostArgs, fused_moegemm_kernel.hpp:103): sorted row r
// of Y (bf16, row-major) times the smooth scale of its expert (SMOOTH), per-row dynamic quantisation to int8:
// scale = amax / 127, codes rounded to nearest even (|value / scale| <= 127 needs no clamp).  ck_tile has no
// instance of these variants to match bit for bit, so the rounding is chosen for accuracy: truncation, which the
// stand-alone smooth-quant kernel above has to use to match ck_tile's, doubles the error of the down GEMM's
// input.  LANES: the threads that hold a row, so that it is read once: a wave up to 2048 columns, a workgroup of 256 up to
// 8192, of 512 up to 16384 (the columns past those are fetched twice, a piece at a time, and take the exact quotients).
// Bound by memory: 59787 rows of 12544 with smooth scales 700 us when 256 threads fetched a third of each row twice and every
// code took its exact quotient, 616 without these, 522 (4.3 TB/s) with a slab's rows on one XCD; 23878 rows of 3904 (a wave each,
// half of it fetched twice) 79 -> 62, 24008 of 1536 28 -> 22.
// Output row-major, or slab-major when segs > 0 (y_slab_offset); padding rows and rows past the sorted prefix are left
// alone.
// FP8 (the fp8 path with fused_quant): e4m3 codes instead, scale = amax / 448, rounded to nearest even by the
// conversion instruction; the workgroups from row_blocks on set the block scales the down GEMM reads (n_ones 16-byte
// pieces) to 2^0, which as a launch of its own took 4.7 us.
template <bool SMOOTH, bool FP8, int LANES>
__global__ __launch_bounds__(LANES < 256 ? 256 : LANES) void moe_requant_y_kernel(const uint16_t* __restrict__ y, int inter,
                                                             const float* __restrict__ smooth,
                                                             const int* __restrict__ sorted_ids,
                                                             const int* __restrict__ sorted_expert_ids,
                                                             const int* __restrict__ total, int unit, int tokens, int topk,
                                                             int segs,
                                                             unsigned char* __restrict__ yq, float* __restrict__ yscale,
                                                             int max_rows, int row_blocks, uint4* __restrict__ ones, int64_t n_ones)
{
    constexpr int kThreads = LANES < 256 ? 256 : LANES;
    constexpr bool kMore   = LANES == 512; // a row may have more columns than its threads hold
    if constexpr(FP8)
    {
        if((int)blockIdx.x >= row_blocks)
        {
            for(int64_t i = (int64_t)(blockIdx.x - row_blocks) * kThreads + threadIdx.x; i < n_ones; i += (int64_t)(gridDim.x - row_blocks) * kThreads)
                ones[i] = make_uint4(0x7f7f7f7fu, 0x7f7f7f7fu, 0x7f7f7f7fu, 0x7f7f7f7fu);
            return;
        }
    }
    const int lane    = threadIdx.x & (LANES - 1);
    // Workgroup ids go round the eight XCDs: the rows of a 16-row slab, whose 64-byte pieces share lines, to one of them.  (Each
    // round of slabs begins one XCD further on, as an expert's padding may leave the same slabs of every round empty.)
    constexpr int kPerSlab = LANES > 64 ? 16 : 4; // workgroups
    const int slot         = blockIdx.x >> 3;
    const int round        = slot / kPerSlab;
    const int64_t group    = (int64_t)(round * 8 + ((blockIdx.x + round) & 7)) * kPerSlab + slot % kPerSlab;
    const int64_t row      = LANES > 64 ? group : group * 4 + (threadIdx.x >> 6);
    if(row >= min(total[0], max_rows)) // (the grid covers whole rounds, up to 127 rows past the buffers)
        return;
    const int chunks = inter >> 3;
    auto dst = [&](int c) {
        return yq + (segs > 0 ? y_slab_offset(row, c * 8, segs) : row * inter + c * 8);
    };
    if(!real_id(sorted_ids[row], tokens, topk))
        return; // padding: no GEMM tile holds the row
    const uint16_t* yr = y + row * inter;
    const float* sr    = SMOOTH ? smooth + (int64_t)sorted_expert_ids[row / unit] * inter : nullptr;
    auto load = [&](int c, float (&o)[8]) {
        const uint4 r = *reinterpret_cast<const uint4*>(yr + c * 8);
        const uint32_t d[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
        for(int i = 0; i < 4; i++)
        {
            o[2 * i]     = __uint_as_float(d[i] << 16);
            o[2 * i + 1] = __uint_as_float(d[i] & 0xffff0000u);
        }
        if constexpr(SMOOTH)
        {
            const float4 s0 = *reinterpret_cast<const float4*>(sr + c * 8);
            const float4 s1 = *reinterpret_cast<const float4*>(sr + c * 8 + 4);
            o[0] *= s0.x; o[1] *= s0.y; o[2] *= s0.z; o[3] *= s0.w;
            o[4] *= s1.x; o[5] *= s1.y; o[6] *= s1.z; o[7] *= s1.w;
        }
    };
    float v[kQuantCache][8];
    float amax = 0.f;
#pragma unroll
    for(int j = 0; j < kQuantCache; j++)
    {
        const int c = lane + LANES * j;
        if(c < chunks)
        {
            load(c, v[j]);
#pragma unroll
            for(int i = 0; i < 8; i++)
                amax = fmaxf(amax, fabsf(v[j][i]));
        }
    }
    for(int c = lane + LANES * kQuantCache; kMore && c < chunks; c += LANES)
    {
        float t[8];
        load(c, t);
#pragma unroll
        for(int i = 0; i < 8; i++)
            amax = fmaxf(amax, fabsf(t[i]));
    }
    if constexpr(LANES > 64)
    {
        __shared__ float s_red[LANES / 64];
        amax = block_max<LANES / 64>(amax, s_red);
    }
    else
        amax = wave_reduce_max(amax, 0.f);
    if(lane == 0)
        yscale[row] = amax / (FP8 ? 448.0f : 127.0f); // (a row of zeros: scale 0, codes 0)
    const RowScale<FP8> rs(amax);
#pragma unroll
    for(int j = 0; j < kQuantCache; j++)
        if(lane + LANES * j < chunks)
            *reinterpret_cast<uint2*>(dst(lane + LANES * j)) = quantise_8<FP8, !FP8>(v[j], rs);
    for(int c = lane + LANES * kQuantCache; kMore && c < chunks; c += LANES)
    {
        float t[8];
        load(c, t);
        *reinterpret_cast<uint2*>(dst(c)) = exact_codes_8<FP8, !FP8>(t, row_reciprocal(rs.scale()));
    }
}

// ck_tile's pre-shuffled weight layout b_nr_kr_kw_nw_kv: the row-major [e, n, k] tensor viewed as
// [e, nr, nw, kr, kw, kv] and permuted to [e, nr, kr, kw, nw, kv].  One thread moves one kv granule.
template <typename G>
__global__ __launch_bounds__(256) void permute_weights_kernel(const G* __restrict__ src, G* __restrict__ dst,
                                                               int64_t granules, int n, int kgran, int nw, int kw,
                                                               int inverse)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if(i >= granules)
        return;
    // i enumerates the permuted layout: (e, nr, kr, kw, nw)
    const int kr_n = kgran / kw;
    int64_t r      = i;
    const int a_nw = (int)(r % nw);
    r /= nw;
    const int a_kw = (int)(r % kw);
    r /= kw;
    const int a_kr = (int)(r % kr_n);
    r /= kr_n;
    const int a_nr = (int)(r % (n / nw));
    const int64_t e = r / (n / nw);
    const int64_t row_major = (e * n + (int64_t)a_nr * nw + a_nw) * kgran + (int64_t)a_kr * kw + a_kw;
    if(inverse)
        dst[row_major] = src[i];
    else
        dst[i] = src[row_major];
}

} // namespace

int launch_permute_weights(const void* src, void* dst, int32_t experts, int32_t n, int32_t k, int32_t elem_bytes,
                           int32_t nw, int32_t kw, int32_t kv, int32_t inverse, hipStream_t stream)
{
    if(!src || !dst || src == dst || experts <= 0 || n <= 0 || k <= 0 || nw <= 0 || kw <= 0 || kv <= 0 ||
       (elem_bytes != 1 && elem_bytes != 2))
        return fail(MI355_MOE_E_INVALID, "permute_weights: bad arguments");
    const int gran = kv * elem_bytes;
    if(n % nw != 0 || k % (kw * kv) != 0 || (gran != 4 && gran != 8 && gran != 16))
        return fail(MI355_MOE_E_UNSUPPORTED,
                    "permute_weights: n %% nw, k %% (kw*kv) must be 0 and kv*elem_bytes 4, 8 or 16 (n=%d k=%d nw=%d kw=%d kv=%d)",
                    n, k, nw, kw, kv);
    const int kgran        = k / kv;
    const int64_t granules = (int64_t)experts * n * kgran;
    const unsigned grid    = (unsigned)ceil_div<int64_t>(granules, 256);
    if(gran == 16)
        hipLaunchKernelGGL(permute_weights_kernel<uint4>, dim3(grid), dim3(256), 0, stream, static_cast<const uint4*>(src),
                           static_cast<uint4*>(dst), granules, n, kgran, nw, kw, inverse);
    else if(gran == 8)
        hipLaunchKernelGGL(permute_weights_kernel<uint2>, dim3(grid), dim3(256), 0, stream, static_cast<const uint2*>(src),
                           static_cast<uint2*>(dst), granules, n, kgran, nw, kw, inverse);
    else
        hipLaunchKernelGGL(permute_weights_kernel<uint32_t>, dim3(grid), dim3(256), 0, stream,
                           static_cast<const uint32_t*>(src), static_cast<uint32_t*>(dst), granules, n, kgran, nw, kw, inverse);
    MI355_HIP_TRY(hipGetLastError());
    return MI355_MOE_OK;
}

int launch_moe_smoothquant(const mi355_moe_smoothquant_args& a, int32_t q_dtype, hipStream_t stream)
{
    if(q_dtype != MI355_MOE_FP8 && q_dtype != MI355_MOE_INT8)
        return fail(MI355_MOE_E_UNSUPPORTED, "moe_smoothquant: q_dtype must be fp8 or int8");
    if(a.tokens < 0 || a.hidden_size <= 0 || a.experts <= 0 || a.topk <= 0 || a.topk > 65535 || a.x_stride < a.hidden_size ||
       a.y_stride < a.hidden_size)
        return fail(MI355_MOE_E_INVALID, "moe_smoothquant: bad sizes (tokens=%d hidden=%d experts=%d topk=%d strides=%d,%d)",
                    a.tokens, a.hidden_size, a.experts, a.topk, a.x_stride, a.y_stride);
    if(a.tokens == 0)
        return MI355_MOE_OK;
    if(!a.p_x || !a.p_smscale || !a.p_topk_ids || !a.p_yscale || !a.p_qy)
        return fail(MI355_MOE_E_INVALID, "moe_smoothquant: null pointer");
    KernelTimer timer(MI355_MOE_K_QUANT, stream);
    // 16-byte pieces of 8 elements when every row starts on a 16-byte (output: 8-byte) boundary
    const bool vec = a.hidden_size % 8 == 0 && a.x_stride % 8 == 0 && a.y_stride % 8 == 0 &&
                     reinterpret_cast<uintptr_t>(a.p_x) % 16 == 0 && reinterpret_cast<uintptr_t>(a.p_smscale) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(a.p_qy) % 8 == 0;
    auto launch = [&](auto kernel, dim3 grid, unsigned lds = 0) {
        hipLaunchKernelGGL(kernel, grid, dim3(256), lds, stream, static_cast<const uint16_t*>(a.p_x),
                           static_cast<const float*>(a.p_smscale), static_cast<const int*>(a.p_topk_ids), a.tokens,
                           a.hidden_size, a.experts, a.topk, (int64_t)a.x_stride, (int64_t)a.y_stride,
                           static_cast<unsigned char*>(a.p_qy), static_cast<float*>(a.p_yscale));
    };
    const dim3 per_token((unsigned)a.tokens), per_wave((unsigned)ceil_div(a.tokens, 4)), per_row((unsigned)a.tokens, (unsigned)a.topk);
    // expert tables beyond 3 MB do not stay in the 4 MB L2 of an XCD: rows grouped by expert, scales in registers
    const int64_t ranges8 = ceil_div<int64_t>(ceil_div(a.tokens, kSqRange), 8);
    const bool grouped    = vec && (int64_t)a.experts * a.hidden_size * (int64_t)sizeof(float) > (3ll << 20) &&
                         kSqRange * a.topk <= kSqMaxList && ranges8 * a.experts * 8 < (1ll << 31);
    // Columns past a thread's registers are fetched again, 6 bytes each, from L2 while the workgroups of an XCD (32 compute
    // units x 4) need no more than it holds; with longer rows 12 KB of LDS more leave three per compute unit: 2048 x 8 int8
    // rows of 13312 129 us with four, 133 with three; of 14336 158, 147; of 16384 242, 210.
    const unsigned grouped_lds = 32 * 4 * 6 * (int64_t)(a.hidden_size - 8 * 256 * kQuantCache) > (4 << 20) ? 12 << 10 : 0;
    auto of_type = [&](auto fp8_tag, auto pieces_tag) {
        constexpr bool FP8   = decltype(fp8_tag)::value;
        constexpr int PIECES = decltype(pieces_tag)::value;
        if(vec && !grouped && wave_per_row(a.tokens, a.hidden_size))
            a.hidden_size <= kWaveCols / 2 ? launch(moe_smoothquant_vec_kernel<FP8, 2, 64>, per_wave) : launch(moe_smoothquant_vec_kernel<FP8, kQuantCache, 64>, per_wave);
        else if(grouped)
            launch(moe_smoothquant_grouped_kernel<FP8, PIECES>, dim3((unsigned)(ranges8 * a.experts * 8)), grouped_lds);
        else if(vec)
            launch(moe_smoothquant_vec_kernel<FP8, PIECES, 256>, per_token);
        else
            launch(moe_smoothquant_kernel<FP8>, per_row);
    };
    // rows of up to 4096 columns need half the registers: six waves per SIMD instead of three (grouped: four, by its list in LDS)
    auto pieces = [&](auto fp8_tag) {
        a.hidden_size <= kBracketCols ? of_type(fp8_tag, std::integral_constant<int, 2>{})
                                     : of_type(fp8_tag, std::integral_constant<int, kQuantCache>{});
    };
    q_dtype == MI355_MOE_FP8 ? pieces(std::true_type{}) : pieces(std::false_type{});
    MI355_HIP_TRY(hipGetLastError());
    return MI355_MOE_OK;
}

int launch_rowwise_quant(const void* x, int64_t rows, int32_t cols, int64_t stride_x, int32_t q_dtype, void* q,
                         void* scale, hipStream_t stream)
{
    if(!x || !q || !scale || rows < 0 || cols <= 0 || stride_x < cols)
        return fail(MI355_MOE_E_INVALID, "rowwise_quant: bad arguments");
    if(q_dtype != MI355_MOE_FP8 && q_dtype != MI355_MOE_INT8)
        return fail(MI355_MOE_E_UNSUPPORTED, "rowwise_quant: q_dtype must be fp8 or int8");
    if(rows == 0)
        return MI355_MOE_OK;
    if(rows > 0x7fffffff)
        return fail(MI355_MOE_E_INVALID, "rowwise_quant: too many rows");
    KernelTimer timer(MI355_MOE_K_QUANT, stream);
    const bool vec = cols % 8 == 0 && stride_x % 8 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(q) % 8 == 0;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)rows), dim3(256), 0, stream, static_cast<const uint16_t*>(x), cols,
                           stride_x, static_cast<unsigned char*>(q), static_cast<float*>(scale));
    };
    auto of_type = [&](auto fp8_tag) {
        constexpr bool FP8 = decltype(fp8_tag)::value;
        if(!vec)
            launch(rowwise_quant_kernel<FP8, false, false>);
        else if(wave_per_row(rows, cols))
            hipLaunchKernelGGL(rowwise_quant_wave_kernel<FP8>, dim3((unsigned)ceil_div<int64_t>(rows, 4)), dim3(256), 0, stream,
                               static_cast<const uint16_t*>(x), cols, stride_x, static_cast<unsigned char*>(q), static_cast<float*>(scale), (int)rows);
        else
            cols <= kBracketCols ? launch(rowwise_quant_kernel<FP8, true, true>) : launch(rowwise_quant_kernel<FP8, true, false>);
    };
    q_dtype == MI355_MOE_FP8 ? of_type(std::true_type{}) : of_type(std::false_type{});
    MI355_HIP_TRY(hipGetLastError());
    return MI355_MOE_OK;
}

int launch_requant_y(const void* y, int32_t inter, const float* smooth, const int* sorted_ids, const int* sorted_expert_ids,
                     const int* total, int32_t unit, int32_t tokens, int32_t topk, int32_t segs, int64_t max_rows, void* yq, float* yscale,
                     hipStream_t stream, bool fp8, void* ones, int64_t ones_bytes)
{
    if(max_rows <= 0)
        return MI355_MOE_OK;
    KernelTimer timer(MI355_MOE_K_QUANT, stream);
    const int lanes      = inter <= 8 * 64 * kQuantCache ? 64 : inter <= 8 * 256 * kQuantCache ? 256 : 512; // (see the kernel)
    const int threads    = std::max(lanes, 256);
    const int row_blocks = (int)round_up<int64_t>(ceil_div<int64_t>(max_rows, threads / lanes), lanes > 64 ? 128 : 32); // whole rounds
    const int64_t n_ones = fp8 ? (ones_bytes + 15) / 16 : 0;
    const dim3 grid((unsigned)(row_blocks + std::min<int64_t>(ceil_div<int64_t>(n_ones, threads), 4096)));
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, stream, static_cast<const uint16_t*>(y), inter, smooth, sorted_ids,
                           sorted_expert_ids, total, unit, tokens, topk, segs, static_cast<unsigned char*>(yq), yscale, (int)max_rows,
                           row_blocks, static_cast<uint4*>(ones), n_ones);
    };
    auto of_type       = [&](auto smooth_tag, auto fp8_tag) {
        constexpr bool S = decltype(smooth_tag)::value, F = decltype(fp8_tag)::value;
        lanes == 64 ? launch(moe_requant_y_kernel<S, F, 64>) : lanes == 256 ? launch(moe_requant_y_kernel<S, F, 256>) : launch(moe_requant_y_kernel<S, F, 512>);
    };
    if(fp8)
        smooth != nullptr ? of_type(std::true_type{}, std::true_type{}) : of_type(std::false_type{}, std::true_type{});
    else
        smooth != nullptr ? of_type(std::true_type{}, std::false_type{}) : of_type(std::false_type{}, std::false_type{});
    MI355_HIP_TRY(hipGetLastError());
    return MI355_MOE_OK;
}

} // namespace mi355
