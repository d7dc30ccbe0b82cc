#pragma once
// The conv on 16-row tiles: the form that a launch takes which nobody packs with others (see paella_conv2d_plan, `small`).
// Included by ops_conv.hip, whose FastDiv, quot_fast, PreOp and kPre* it uses.
//
// At batch 1 most layers have too few 32 x 32 tiles for 256 compute units.  The kernel of ops_conv.hip then splits the
// reduction over several workgroups, which exchange partial tiles through memory: a store that is waited for, a counter in
// memory and a read back, 2 to 3 us of the launch's 5 to 8.  Here a tile is (16 * MI) channels x 16 pixels
// (v_mfma_f32_16x16x4_f32, the same rate per cycle), four or two times as many of them, the whole reduction stays in one
// workgroup and its partial tiles, 1 KB each, meet in LDS.  Each wave loads twice the operands per matrix instruction, which a
// launch that fills the device several times over pays for and a lone small layer does not.  By counters, 256->256 3x3 on 14x14: twice the
// look-ups of a compute unit's vector cache (11 600 against 5600), whose data unit is busy for 6.9 of 11.0 us (4.3 of 8.1); 768->192 on 17x17:
// half of them (1900 against 3800), since four times as many compute units have work, and 2.3 of 4.9 us (4.0 of 6.2).
//
// The result has the bits of the 32 x 32 kernel.  The fp32 matrix instructions add their products one after the other, each
// with one rounding, in ascending order of the reduction index they are given; v_mfma_f32_32x32x2 is given the pairs (k, k + 4),
// k = 0..3, of a chunk of eight, so here one instruction is given 0, 4, 1, 5 and the next 2, 6, 3, 7.  A *part* is what one wave
// of the 32 x 32 plan sums (of its `kw` waves in each of its `splits`); parts are summed here in the same pieces and added in the
// same order: waves within a split, then splits.
//
// Operands: lanes (j, kk), j = 0..15, kk = 0..3.  Of a chunk, lane kk needs elements (kk >> 1) and (kk >> 1) + 2 of the four
// reduction values 4 * (kk & 1) ..  -- of the 16 bytes that the packed weights hold for them, half.  So the lower 32 lanes fetch
// the 16 bytes of one chunk, the upper 32 those of the next, and one v_permlane32_swap per pair of registers leaves both chunks'
// operands where the matrix instructions want them.

struct SmallArgs {
    const float* x;
    const float4* wpk;
    const float* bias;
    const float* residual;
    const float* slope;
    float* y;
    int H, W, Q, PQ, sh, sw, ph, pw;
    int K, m_pad, nchunks, S, dh, dw, CB;
    unsigned x_bytes, w_bytes;
    int n_tiles_n, n_tiles_m;
    int slab_major, pointwise, pair_s0;
    int parts, kw_log, chunks_per_split;   // parts = splits << kw_log
    int act;
    float lo, hi;
    FastDiv div_w, div_q, div_cb, div_s;
};

typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kPreZeros = 128;

template <int MI, int NW, bool PW, int PRE = kPreNone>
__device__ __forceinline__ void conv_small_tile(const SmallArgs& p, const unsigned bid, const PreOp pre = PreOp{nullptr, nullptr, 0.f}) {
    constexpr int NE = MI * 4;  // accumulator registers of a tile
    constexpr int D = 2;        // pairs of chunks in flight per wave; three and four measured slower (more registers, longer prologue)
    if (bid >= (unsigned)(p.n_tiles_n * p.n_tiles_m)) return;
    extern __shared__ __align__(16) char smem[];
    float* const red = reinterpret_cast<float*>(smem);       // [part][NE][64]
    char* const ptab = smem + p.parts * (NE * 256);          // input transform: kPreZeros bytes of zeros, then {scale, shift} per channel

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, kk = lane >> 4;
    // Workgroups to tiles: as in conv_tile, every XCD gets a contiguous run of the work list.
    int tile_n, tile_m;
    {
        const unsigned total = (unsigned)(p.n_tiles_n * p.n_tiles_m);
        const unsigned xcd = bid & 7u, q = total >> 3, r = total & 7u;
        const unsigned w = xcd * q + (xcd < r ? xcd : r) + (bid >> 3);
        const unsigned d_w = p.slab_major ? (unsigned)p.n_tiles_n : (unsigned)p.n_tiles_m;
        const unsigned a = quot_fast(w, p.div_w), b = w - a * d_w;
        tile_n = (int)(p.slab_major ? b : a);
        tile_m = (int)(p.slab_major ? a : b);
    }
    const int m0 = tile_m * (16 * MI);
    const int pix = tile_n * 16 + j;
    // The input through a descriptor that starts where tap (0, 0) of output pixel (0, 0) would lie (see conv_tile).
    const unsigned pad_off = (unsigned)(p.ph * p.W + p.pw) * 4u;
    const char* const x_base = reinterpret_cast<const char*>(p.x) - pad_off;
    const unsigned x_len = p.x_bytes + pad_off;
    const int HW4 = p.H * p.W * 4;
    const int chan_lane = (kk >> 1) * HW4;         // this lane's channel within its four
    const int group_lane = (kk & 1) * (4 * HW4);   // ... and which four of a chunk's eight
    int hb = 0, wb = 0, base;
    if (PW) {
        base = pix < p.PQ ? pix * 4 + chan_lane + group_lane : (int)0x80000000u;
    } else {
        const int ho = (int)quot_fast((unsigned)pix, p.div_q);
        const int wo = pix - __mul24(ho, p.Q);
        hb = pix < p.PQ ? __mul24(ho, p.sh) - p.ph : -0x100000;
        wb = __mul24(wo, p.sw) - p.pw;
        base = (__mul24(hb, p.W) + wb) * 4 + (int)pad_off + chan_lane + group_lane;
    }
    const int pair_delta = (kk & 1) * (p.dw * 4) - group_lane;  // paired filter columns: the half selects the column
    const int wlane1 = ((kk & 1) * p.m_pad + m0 + j) * 16;      // weights: both halves of the wave in the same chunk
    const int wstep = p.m_pad * 32;
    const int wlane2 = wlane1 + (kk >> 1) * wstep;              // the upper half one chunk further

    // ---- the wave's parts, one behind the other, each a pipeline of D pairs of chunks.  A lone launch has one or two waves per
    // SIMD, so the scalar instructions of the loop are not hidden: the position is kept by addition, its test is made once per
    // pair, and in the steady state nothing is tested against the part's end.
    struct Slot {
        float4 a[MI];
        float b[2][2];           // [chunk][instruction]
        float sc[2][2], sh[2][2];
        int addr[2];             // of the scales in the table, per chunk (with an input transform)
    };
    int c_left = 0;              // chunks of the part that are not yet requested
    int w_off = 0, x_off = 0;    // byte offsets of the next pair's weights and the next chunk's input
    int cb_left = 0;             // chunks left in the current tap (with paired filter columns: in the current unit)
    int x_step = 8 * HW4;        // from chunk to chunk
    int tap = 0;
    int tap_voff = base;
    int pre_addr = 0, pre_mask = ~0;   // input transform: the lane's place in the table; all zeros where the tap is padding
    const int pre_lane = kPreZeros + ((kk >> 1) + (kk & 1) * 4) * 8;
    // (Row and column by division each time: kept by carries from block to column to row they end up in vector registers, and the
    // 3x3 layers ran a tenth slower.)
    auto open_tap = [&](int t, int cb) {  // position on chunk cb of tap (unit) t
        const int r = (int)quot_fast((unsigned)t, p.div_s);
        int col = t - r * p.S, chan = 0, step = 8;
        bool seg_pair = false;
        if (!PRE && p.pair_s0 >= 0) {  // the packing of stride-2 3-wide filters, see conv_tile
            seg_pair = col != 0;
            chan = col == 2 ? p.CB * 4 : 0;
            step = seg_pair ? 4 : 8;
            col = seg_pair ? p.pair_s0 : 2 - 2 * p.pair_s0;
        }
        const int dy = r * p.dh, dx = col * p.dw;
        const bool ok = ((unsigned)(hb + dy) < (unsigned)p.H) & ((unsigned)(wb + dx) < (unsigned)p.W);
        tap_voff = ok ? (seg_pair ? base + pair_delta : base) : -1;
        chan += cb * step;
        x_off = chan * HW4 + (dy * p.W + dx) * 4;
        x_step = step * HW4;
        cb_left = p.CB - cb;
        tap = t;
        if (PRE) {
            pre_mask = ok ? ~0 : 0;
            pre_addr = pre_lane + chan * 8;
        }
    };
    // full: both chunks of the pair lie in the part
    auto load = [&](Slot& f, auto full) {
        constexpr bool FULL = decltype(full)::value;
        const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void*)p.wpk, 0, FULL || c_left > 0 ? p.w_bytes : 0u, 0x00027000);
        const int wl = FULL || c_left > 1 ? wlane2 : wlane1;  // (the chunk behind the last one may not exist)
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) f.a[mi] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(wr, wl, w_off + mi * 256, 0));
        w_off += 2 * wstep;
        int v0 = tap_voff, v1 = tap_voff, o0 = x_off, o1 = x_off + x_step;
        if (PRE) {
            f.addr[0] = pre_addr & pre_mask;
            f.addr[1] = (pre_addr + 64) & pre_mask;
            pre_addr += 128;
        }
        x_off += 2 * x_step;
        if (!PW) {
            cb_left -= 2;
            if (cb_left <= 0) {  // the tap ends with this pair or inside it
                const bool inside = cb_left < 0;
                open_tap(tap + 1, 0);
                if (inside) {
                    v1 = tap_voff;
                    o1 = x_off;
                    x_off += x_step;
                    cb_left -= 1;
                    if (PRE) {
                        f.addr[1] = pre_addr & pre_mask;
                        pre_addr += 64;
                    }
                    if (cb_left == 0) open_tap(tap + 1, 0);
                }
            }
        }
        const __amdgpu_buffer_rsrc_t xr0 = __builtin_amdgcn_make_buffer_rsrc((void*)x_base, 0, FULL || c_left > 0 ? x_len : 0u, 0x00027000);
        const __amdgpu_buffer_rsrc_t xr1 = __builtin_amdgcn_make_buffer_rsrc((void*)x_base, 0, FULL || c_left > 1 ? x_len : 0u, 0x00027000);
        f.b[0][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr0, v0, o0, 0));
        f.b[0][1] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr0, v0, o0 + 2 * HW4, 0));
        f.b[1][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr1, v1, o1, 0));
        f.b[1][1] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr1, v1, o1 + 2 * HW4, 0));
        if (PRE && !FULL) {
            if (c_left <= 0) f.addr[0] = 0;  // past the table otherwise
            if (c_left <= 1) f.addr[1] = 0;
        }
        c_left -= 2;
    };
    auto load_pre = [&](Slot& f) {
        if (!PRE) return;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const float2* const t = reinterpret_cast<const float2*>(ptab + f.addr[u]);
            const float2 t0 = t[0], t2 = t[2];
            f.sc[u][0] = t0.x; f.sh[u][0] = t0.y;
            f.sc[u][1] = t2.x; f.sh[u][1] = t2.y;
        }
    };
    auto open_part = [&](int part) {
        const int split = part >> p.kw_log, w = part & ((1 << p.kw_log) - 1);
        const int g_begin = split * p.chunks_per_split;
        const int g_end = min(p.nchunks, g_begin + p.chunks_per_split);
        const int cpw = (g_end - g_begin + (1 << p.kw_log) - 1) >> p.kw_log;
        const int c = g_begin + w * cpw;
        c_left = part < p.parts ? max(0, min(g_end - c, cpw)) : 0;
        w_off = c * wstep;
        if (PW) {
            x_off = c * 8 * HW4;
            pre_addr = pre_lane + c * 64;
        } else {
            const int t = (int)quot_fast((unsigned)c, p.div_cb);
            open_tap(t, c - t * p.CB);
        }
    };
    constexpr std::true_type kFull{};
    constexpr std::false_type kAny{};
    f32x4 acc[MI];
    auto compute = [&](Slot& f, bool both) {
        float a[MI][2][2];  // [.][chunk][instruction]
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) {
            const auto s0 = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, f.a[mi].x), __builtin_bit_cast(unsigned, f.a[mi].y), false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, f.a[mi].z), __builtin_bit_cast(unsigned, f.a[mi].w), false, false);
            const unsigned a00 = s0[0], a10 = s0[1], a01 = s1[0], a11 = s1[1];
            a[mi][0][0] = __builtin_bit_cast(float, a00);
            a[mi][1][0] = __builtin_bit_cast(float, a10);
            a[mi][0][1] = __builtin_bit_cast(float, a01);
            a[mi][1][1] = __builtin_bit_cast(float, a11);
        }
        auto chunk = [&](int u) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                float b = f.b[u][i];
                if (PRE) {
                    b = b * f.sc[u][i] + f.sh[u][i];
                    if (PRE == kPreBounded) b = fmaxf(b, pre.lo);
                }
#pragma unroll
                for (int mi = 0; mi < MI; ++mi) acc[mi] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[mi][u][i], b, acc[mi], 0, 0, 0);
            }
        };
        chunk(0);
        if (both) chunk(1);
    };

    int part = wave;
    open_part(part);
    int n = c_left;
    Slot slot[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
        load(slot[d], kAny);
        __builtin_amdgcn_sched_barrier(0);
    }
    // The epilogue's operands travel while the reduction runs: thread (wave w, lane) finishes registers w, w + NW, .. of the tile.
    // Rows past K: a descriptor of the tensor's length and a scalar offset held at that length (see conv_tile).
    constexpr int PER = NE > NW ? NE / NW : 1;
    const bool finishes = wave < NE;
    const unsigned plane = (unsigned)p.PQ * 4u;
    const unsigned y_len = (unsigned)p.K * plane, c_len = (unsigned)p.K * 4u;
    const int lane_off = pix < p.PQ ? (int)((unsigned)(kk * 4) * plane + (unsigned)pix * 4u) : (int)0x80000000u;
    auto rsrc = [](const void* q, unsigned len) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(q), 0, q ? len : 0u, 0x00027000); };
    auto row_of = [&](int i) { const int e = wave + i * NW; return (unsigned)(m0 + (e >> 2) * 16 + (e & 3)); };
    float bias_v[PER], res_v[PER], slope_v[PER];
    if (finishes) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int chan_soff = (int)min(row_of(i) * 4u, c_len), plane_soff = (int)min(row_of(i) * plane, y_len);
            bias_v[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc(p.bias, c_len), kk * 16, chan_soff, 0));
            res_v[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc(p.residual, y_len), lane_off, plane_soff, 0));
            slope_v[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc(p.slope, c_len), kk * 16, chan_soff, 0));
        }
    }
    if (PRE) {
        const int n_chan = p.CB * 8;
        if (threadIdx.x < kPreZeros / 4) reinterpret_cast<float*>(ptab)[threadIdx.x] = 0.f;
        float2* const tab = reinterpret_cast<float2*>(ptab + kPreZeros);
        for (int i = (int)threadIdx.x; i < n_chan; i += 64 * NW) tab[i] = make_float2(pre.scale[i], pre.shift[i]);
        __syncthreads();
#pragma unroll
        for (int d = 0; d < D; ++d) load_pre(slot[d]);
    }
    __builtin_amdgcn_sched_barrier(0);
    while (true) {
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) acc[mi] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto turn = [&](auto full) {  // D pairs are used, D requested
#pragma unroll
            for (int d = 0; d < D; ++d) {
                compute(slot[d], true);
                __builtin_amdgcn_sched_barrier(0);
                load(slot[d], full);
                load_pre(slot[d]);
                __builtin_amdgcn_sched_barrier(0);
            }
            n -= 2 * D;
        };
        while (c_left >= 2 * D) turn(kFull);
        if (c_left > 0) turn(kAny);
        auto flush = [&]() {
#pragma unroll
            for (int mi = 0; mi < MI; ++mi)
#pragma unroll
                for (int e = 0; e < 4; ++e) red[(part * NE + mi * 4 + e) * 64 + lane] = acc[mi][e];
        };
        if (part + NW >= p.parts) {
#pragma unroll
            for (int d = 0; d < D; ++d)  // the rest is in the slots
                if (n > 2 * d) compute(slot[d], n > 2 * d + 1);
            if (part < p.parts) flush();
            break;
        }
        // the next part's first pairs take the slots as they become free
        open_part(part + NW);
        const int n_next = c_left;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (n > 2 * d) compute(slot[d], n > 2 * d + 1);
            __builtin_amdgcn_sched_barrier(0);
            load(slot[d], kAny);
            load_pre(slot[d]);
            __builtin_amdgcn_sched_barrier(0);
        }
        flush();
        part += NW;
        n = n_next;
    }
    __syncthreads();
    if (!finishes) return;
    const int splits = p.parts >> p.kw_log;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = wave + i * NW;
        const float* t = red + e * 64 + lane;
        // the waves of one split of the 32 x 32 plan, then the splits; all of a split's parts are read together
        auto sum = [&](auto count) {
            constexpr int KW = decltype(count)::value;
            float s[KW];
#pragma unroll
            for (int k = 0; k < KW; ++k) s[k] = t[k * (NE * 64)];
            t += KW * (NE * 64);
            float w = s[0];
#pragma unroll
            for (int k = 1; k < KW; ++k) w += s[k];
            return w;
        };
        float v = 0.f;
        for (int s = 0; s < splits; ++s) {
            const float w = p.kw_log == 3 ? sum(std::integral_constant<int, 8>{}) : p.kw_log == 2 ? sum(std::integral_constant<int, 4>{})
                          : p.kw_log == 1 ? sum(std::integral_constant<int, 2>{}) : sum(std::integral_constant<int, 1>{});
            v = splits == 1 ? w : v + w;
        }
        v += bias_v[i];
        v += res_v[i];
        switch (p.act) {
            case PAELLA_ACT_RELU: v = fmaxf(v, 0.f); break;
            case PAELLA_ACT_RELU6: v = fminf(fmaxf(v, 0.f), 6.f); break;
            case PAELLA_ACT_PRELU: v = v > 0.f ? v : v * slope_v[i]; break;
            case PAELLA_ACT_CLIP: v = fminf(fmaxf(v, p.lo), p.hi); break;
            default: break;
        }
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rsrc(p.y, y_len), lane_off, (int)min(row_of(i) * plane, y_len), 16 /* sc1: write through */);
    }
}
