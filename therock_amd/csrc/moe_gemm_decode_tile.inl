// One tile of the decode GEMM, included in the bodies of moe_gemm_decode_kernel and decode_tile (moe_gemm_decode.hip), where MODE,
// GEMM0, NXB, WPERM, WEIGHTS, p, tile and lds are declared.
    using MT  = ModeTraits<MODE>;
    using Acc = typename MT::Acc;
    constexpr int kOpB     = MT::kOpB;
    constexpr int kXMul    = MT::kXKB / MT::kWKB;     // token bytes per weight byte (2 for bf16 x int8)
    constexpr int kXKB     = kDecWKB * kXMul;         // token bytes per row and step
    constexpr int kWStride = kDecWKB + kPadB;
    constexpr int kXStride = kXKB + kPadB;
    constexpr int kWaveWB  = kDecWKB / 4;             // weight bytes of a row one wave multiplies per step
    constexpr int kSteps   = kWaveWB * kXMul / (2 * kOpB); // MFMAs along K per wave and step
    constexpr int kWLoads  = kDecWRows * (kDecWKB / 16) / kBlock; // 8
    constexpr int kXLoads  = NXB * 32 * (kXKB / 16) / kBlock;     // 4 or 8 per token block
    constexpr int kWRowsPerPass = kBlock / (kDecWKB / 16);        // 8
    constexpr int kXRowsPerPass = kBlock / (kXKB / 16);
    constexpr bool kMx     = MODE == kFp8 && !GEMM0;

    unsigned char* lds_w = lds;
    unsigned char* lds_x = lds + kDecWRows * kWStride;

    const int tid  = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int r32  = lane & 31;
    const int kg   = lane >> 5;

    const int expert = tile.expert;
    const int row0   = tile.row0;
    const int slice  = !GEMM0 && p.k_cols > 0 ? tile.nt / p.k_cols : 0; // slice of K (down GEMM)
    const int nt     = tile.nt - slice * p.k_cols;
    const int nrows  = min(tile.nrows, 32 * NXB);
    // a tile of at most 32 rows leaves the second token block out: no LDS traffic and no MFMAs for it (its loads are
    // masked row by row anyway)
    const bool two   = NXB > 1 && nrows > 32;
    const bool paired = GEMM0 && !p.gate_only; // gate rows paired with up rows (see run_epilogue)
    const int n_base  = nt * (paired ? 32 : 64);

    // ---- global -> register staging assignments: 32 consecutive lanes fetch 512 contiguous bytes
    const int xchunk = tid % (kXKB / 16);
    const int xrow   = tid / (kXKB / 16);
    // The sorted ids of the token rows: fetched first, used only after the first step's weights are on their way.  Nothing
    // of the weights' addresses depends on them, and a workgroup's life is short enough (some 10 us) for a round trip to
    // show: with the epilogue's operands fetched behind the K loop's last step instead of after the reduction, 256
    // Zipf-routed tokens of 128 int8 experts 247.7 -> 242.9 us.  (The second step's weights ahead of the ids as well:
    // two-block tiles lose 1 to 2 %, their first step then waits for both.)
    int sid[kXLoads];
    const bool by_id = GEMM0 || p.slot_rows > 0;
#pragma unroll
    for(int j = 0; j < kXLoads; j++)
    {
        const int r = xrow + kXRowsPerPass * j;
        sid[j]      = r < nrows ? 0 : p.tokens;
        if(by_id && r < nrows)
            sid[j] = p.sorted_ids[row0 + r];
    }
    // Which 16 bytes of the 64 x 512-byte weight tile thread `tid` fetches with load j, as (tile row, 16-byte chunk) =
    // (w_row0 + w_row_add(j), w_chunk0 + w_chunk_add(j)).  Row-major weights: 32 consecutive threads walk the 512
    // contiguous bytes of a row.  ck_tile's pre-shuffled layout (16 rows x 64 bytes per 1 KiB block, the 16-byte
    // pieces of a block ordered by chunk, then row): 16 consecutive threads take the 16 rows of one chunk, 64 a
    // whole block, the four waves four consecutive blocks - a wave's load is 1 KiB of contiguous memory there too.
    // (Bits of the row: 0-1 = tid bits 0-1, 2 = j bit 1, 3-4 = tid bits 2-3, 5 = j bit 2, so that the channels
    // chan_of_row() gives the rows are 16 (j bit 1) + tid % 16; chunk: 0-3 = tid bits 4-7, 4 = j bit 0.)
    // (a template argument: chosen at run time the per-load offsets stop being constants, which costs the registers
    // that three workgroups per compute unit leave no room for)
    constexpr bool wperm = WPERM;
    const int w_chunk0 = wperm ? ((tid >> 6) << 2) | ((tid >> 4) & 3) : tid % (kDecWKB / 16);
    const int w_row0   = wperm ? (((tid >> 3) & 1) << 4) | (((tid >> 2) & 1) << 3) | (tid & 3) : tid / (kDecWKB / 16);
    auto w_row_add     = [&](int j) { return wperm ? ((j >> 2) << 5) | (((j >> 1) & 1) << 2) : kWRowsPerPass * j; };
    auto w_chunk_add   = [&](int j) { return wperm ? (j & 1) << 4 : 0; };
    static_assert(kWLoads == 8 && kWRowsPerPass == 8, "the assignments above cover 64 rows x 32 chunks with 8 loads of 256 threads");
    const unsigned char* wbase = p.w + (int64_t)expert * p.w_expert_bytes;
    // (with both walks in the tile the layout is asked at run time: known to the compiler, it holds more of the offsets' parts in
    // registers and spills 8 of them)
    const bool permuted = WEIGHTS == kByTile ? p.w_permuted != 0 : WPERM;
    uint32_t woff[kWLoads];
#pragma unroll
    for(int j = 0; j < kWLoads; j++)
    {
        const int lrow = w_row0 + w_row_add(j);
        const int blk  = lrow >> 5;
        const int c    = chan_of_row(lrow & 31);
        int grow;
        if(paired)
            grow = blk * p.n_out + min(n_base + c, p.n_out - 1);
        else
            grow = min(n_base + blk * 32 + c, p.n_total - 1);
        woff[j] = weight_offset(p, permuted, grow, w_chunk0 + w_chunk_add(j));
        if constexpr(WEIGHTS == kByTile)
            asm volatile("" : "+v"(woff[j])); // (the upper half of the 64-bit multiply-add it comes from would stay alive beside it)
    }

    const int w_kadv = weight_k_advance(p, kDecWKB); // bytes between the K windows of two steps
    // two steps are kept in flight per workgroup: with three workgroups on a compute unit that is what it
    // takes to have enough bytes outstanding to cover the HBM latency
    uint4 xv_[2][kXLoads];
    uint4 wv_[2][kWLoads];
    uint32_t ys_next_[2][NXB], ys_cur[NXB];
#pragma unroll
    for(int i = 0; i < NXB; i++)
        ys_next_[0][i] = ys_next_[1][i] = ys_cur[i] = 0x7f7f7f7fu;
    const uint4 zero4 = {0u, 0u, 0u, 0u};

    auto load_w = [&](int kt, auto buf_tag, auto once_tag) __attribute__((always_inline)) {
        constexpr int B   = decltype(buf_tag)::value;
        auto& wv          = wv_[B];
        const int kw = kt * kDecWKB + w_chunk0 * 16;
#pragma unroll
        for(int j = 0; j < kWLoads; j++)
        {
            wv[j] = zero4;
            if(kw + w_chunk_add(j) * 16 < p.k_bytes_w)
            {
                typedef __attribute__((ext_vector_type(4))) unsigned u32x4_t;
                const u32x4_t* src = reinterpret_cast<const u32x4_t*>(wbase + (woff[j] + (uint32_t)(kt * w_kadv)));
                const u32x4_t t    = decltype(once_tag)::value ? __builtin_nontemporal_load(src) : *src;
                wv[j]              = make_uint4(t[0], t[1], t[2], t[3]);
            }
        }
    };

    // the steps [kt_first, kt_count) of K are this workgroup's
    const int kt_all   = ceil_div(p.k_bytes_w, kDecWKB);
    const int kt_slice = !GEMM0 && p.k_cols > 0 ? p.k_slice / kDecWKB : kt_all;
    const int kt_first = slice * kt_slice;
    const int kt_count = min(kt_all, kt_first + kt_slice);
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;
    // addresses are a uniform base plus a 32-bit byte offset (the launcher checks that this suffices)
    uint32_t xoff[kXLoads];
    bool xvalid[kXLoads];
    auto resolve_x = [&]() __attribute__((always_inline)) {
#pragma unroll
        for(int j = 0; j < kXLoads; j++)
        {
            const int r   = xrow + kXRowsPerPass * j;
            xvalid[j]     = r < nrows && (!by_id || real_id(sid[j], p.tokens, GEMM0 ? p.topk : p.slot_rows));
            uint32_t src  = row0 + r;
            if constexpr(GEMM0)
                src = token_row(p, sid[j]);
            else if(p.slot_rows > 0)
                src = (uint32_t)slot_row(sid[j], p.slot_rows);
            xoff[j] = (xvalid[j] ? src : 0u) * (uint32_t)p.x_row_bytes + xchunk * 16;
        }
    };
    auto load_x = [&](int kt, auto buf_tag) __attribute__((always_inline)) {
        constexpr int B   = decltype(buf_tag)::value;
        auto& xv          = xv_[B];
        auto& ys_next     = ys_next_[B];
        const int kx = kt * kXKB + xchunk * 16;
#pragma unroll
        for(int j = 0; j < kXLoads; j++)
        {
            xv[j] = zero4;
            if(xvalid[j] && kx < p.k_bytes_x)
                xv[j] = *reinterpret_cast<const uint4*>(p.x + (xoff[j] + (uint32_t)(kt * kXKB)));
        }
        if constexpr(kMx)
        {
            // the four e8m0 scales of this wave's 128 columns of the step, per token block
            const int kb = kt * (kDecWKB / 32) + wave * 4;
#pragma unroll
            for(int i = 0; i < NXB; i++)
            {
                ys_next[i] = 0x7f7f7f7fu;
                if(r32 + 32 * i < nrows && kb * 32 < p.k_bytes_x)
                {
                    const unsigned char* sp = p.y_scale + (int64_t)kb * p.ys_kb_stride + row0 + r32 + 32 * i;
                    ys_next[i] = sp[0] | (sp[p.ys_kb_stride] << 8) | (sp[2 * p.ys_kb_stride] << 16) |
                                 (static_cast<uint32_t>(sp[3 * p.ys_kb_stride]) << 24);
                }
            }
        }
    };

    Acc acc[NXB][2];
#pragma unroll
    for(int i = 0; i < NXB; i++)
#pragma unroll
        for(int b = 0; b < 2; b++)
#pragma unroll
            for(int v = 0; v < 16; v++)
                acc[i][b][v] = 0;

    auto k_step = [&](int kt, auto buf_tag, auto once_tag) __attribute__((always_inline)) {
        constexpr int B = decltype(buf_tag)::value;
        auto& xv        = xv_[B];
        auto& wv        = wv_[B];
#pragma unroll
        for(int j = 0; j < kXLoads; j++)
            if(j < kXLoads / NXB || two)
                *reinterpret_cast<uint4*>(lds_x + (xrow + kXRowsPerPass * j) * kXStride + xchunk * 16) = xv[j];
#pragma unroll
        for(int j = 0; j < kWLoads; j++)
            *reinterpret_cast<uint4*>(lds_w + (w_row0 + w_row_add(j)) * kWStride + (w_chunk0 + w_chunk_add(j)) * 16) = wv[j];
#pragma unroll
        for(int i = 0; i < NXB; i++)
            ys_cur[i] = ys_next_[B][i];
        __syncthreads();
        if(kt + 2 < kt_count)
        {
            load_x(kt + 2, buf_tag);
            load_w(kt + 2, buf_tag, once_tag);
        }
        const unsigned char* xp = lds_x + r32 * kXStride + wave * kWaveWB * kXMul;
#pragma unroll
        for(int s = 0; s < kSteps; s++)
        {
            Frag wf[2];
#pragma unroll
            for(int b = 0; b < 2; b++)
            {
                const unsigned char* wp = lds_w + (b * 32 + r32) * kWStride + wave * kWaveWB;
                if constexpr(MODE == kBf16W8)
                    wf[b].lo = int8x8_to_bf16x8(*reinterpret_cast<const uint2*>(wp + (2 * s + kg) * 8));
                else if constexpr(kOpB == 16)
                    wf[b].lo = *reinterpret_cast<const uint4*>(wp + (2 * s + kg) * 16);
                else
                {
                    wf[b].lo = *reinterpret_cast<const uint4*>(wp + (4 * s + kg) * 16);
                    wf[b].hi = *reinterpret_cast<const uint4*>(wp + (4 * s + 2 + kg) * 16);
                }
            }
#pragma unroll
            for(int i = 0; i < NXB; i++)
            {
                if(i > 0 && !two)
                    continue;
                Frag xf;
                uint32_t xs              = 127;
                const unsigned char* xpi = xp + i * 32 * kXStride;
                if constexpr(kOpB == 16)
                    xf.lo = *reinterpret_cast<const uint4*>(xpi + (2 * s + kg) * 16);
                else
                {
                    xf.lo = *reinterpret_cast<const uint4*>(xpi + (4 * s + kg) * 16);
                    xf.hi = *reinterpret_cast<const uint4*>(xpi + (4 * s + 2 + kg) * 16);
                    if constexpr(kMx)
                        xs = (ys_cur[i] >> (8 * (2 * s + kg))) & 0xffu;
                }
                acc[i][0] = mfma<MODE>(wf[0], xf, xs, acc[i][0]);
                acc[i][1] = mfma<MODE>(wf[1], xf, xs, acc[i][1]);
            }
        }
        __syncthreads();
    };
    auto walk = [&](auto once_tag) __attribute__((always_inline)) {
        load_w(kt_first, B0{}, once_tag);
        __builtin_amdgcn_sched_barrier(0); // (the scheduler would put the ids' wait first)
        resolve_x();
        load_x(kt_first, B0{});
        if(kt_first + 1 < kt_count)
        {
            load_x(kt_first + 1, B1{});
            load_w(kt_first + 1, B1{}, once_tag);
        }
        for(int kt = kt_first; kt < kt_count; kt += 2)
        {
            k_step(kt, B0{}, once_tag);
            if(kt + 1 < kt_count)
                k_step(kt + 1, B1{}, once_tag);
        }
    };
    // Weights that only this workgroup reads are fetched non-temporal: 64 evenly routed tokens of 128 int8 experts 4096 x 1536
    // 371 us, with plain loads 420.  Those of an expert with several row tiles are read by as many workgroups at about the same
    // time, and with the hint some of it goes past L2 again (a Zipf-routed batch of 256 tokens fetched 574 and 272 MB in its two
    // GEMMs, with plain loads there 437 and 229).  Passes: 256 Zipf-routed tokens of that layer 249 -> 218 us (other routing 238 ->
    // 226), in bf16 454 -> 397, 393 x 3 of 53 fp8 experts 6464 x 2560 356 -> 324.  The walk stands here
    // twice because a choice at each load makes the compiler wait for more loads than it has to (decode 1 to 3 % slower); the
    // asm statements differ so that it does not fold the two walks' first loads into one and drop the hint.
    if(WEIGHTS == kOnce || (WEIGHTS == kByTile && tile.expert_tiles == 1))
    {
        asm volatile("; weights read once");
        walk(std::true_type{});
    }
    else
    {
        asm volatile("; weights read by several row tiles");
        walk(std::false_type{});
    }

    // ---- add the four K slices: waves 1..3 park their accumulators in LDS, wave 0 sums in wave order
    using AccElem   = decltype(acc[0][0][0] + acc[0][0][0]);
    AccElem* red    = reinterpret_cast<AccElem*>(lds); // [3][NXB][2][16][64]
    // the epilogue's operands travel while the slices are added
    EpilogueOperands<NXB> eo;
    if(wave == 0)
        load_epilogue<MODE, GEMM0, NXB>(p, eo, expert, row0, nrows, 0, 32, n_base, 0, r32, kg, slice);
    if(wave > 0)
    {
#pragma unroll
        for(int i = 0; i < NXB; i++)
        {
            if(i > 0 && !two)
                continue;
#pragma unroll
            for(int b = 0; b < 2; b++)
#pragma unroll
                for(int v = 0; v < 16; v++)
                    red[((((wave - 1) * NXB + i) * 2 + b) * 16 + v) * 64 + lane] = acc[i][b][v];
        }
    }
    __syncthreads();
    if(wave > 0)
        return;
    // one wave's 32 values at a time: fetching all 96 at once does not fit the register budget of three
    // workgroups per compute unit
#pragma nounroll
    for(int w = 0; w < 3; w++)
#pragma unroll
        for(int i = 0; i < NXB; i++)
        {
            if(i > 0 && !two)
                continue;
#pragma unroll
            for(int b = 0; b < 2; b++)
#pragma unroll
                for(int v = 0; v < 16; v++)
                    acc[i][b][v] += red[(((w * NXB + i) * 2 + b) * 16 + v) * 64 + lane];
        }

    pin_epilogue(eo);
    apply_epilogue<MODE, GEMM0, NXB>(p, acc, eo, row0, nrows, 0, 32, ceil_div(nrows, 32), r32, kg, expert);
