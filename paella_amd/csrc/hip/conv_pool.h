#pragma once
// A small conv and the maximum pooling behind it in one kernel, where no two windows share a pixel.  Included by ops_conv.hip, whose FastDiv, quot_fast
// and activations it uses.
//
// A network of small layers is a chain of launches of 2 to 4 us that compute next to nothing: what a layer takes is its way from the launch to the first
// operand and from the last sum to memory, and the boundary to the next.  A pooling operator is nothing but that.  Here a tile's 16 columns
// (v_mfma_f32_16x16x4_f32, see conv_small.h) are not neighbouring pixels but whole windows -- four of 2x2, one of 3x3 and seven columns idle -- so the maximum
// is taken across a wave's lanes and the conv's output is never written.  The launch is one workgroup per 16 channels and tile of windows, with the waves
// and the chunks per wave of the conv's own plan: the bits are those of the conv's kernel and the pool's.
// The small CNN (28x28, 5x5 convs of 8 and 16 channels, pools 2x2 and 3x3), five launches -> three: one request without a server 27.9 -> 23.1 us, a lone
// client of the server 25.4 -> 18.7 us a request.  What such a kernel takes is the chain of trips in it.  us a launch for its two convs, 2.51 and 4.04
// now, and, in brackets, for a 1x1 8->16 on 48x48 with 2x2, 2.69: the arguments where they are used, six trips, 2.58 and 4.14 (2.75); bias
// and slope behind the sum 2.54 and 4.07 (3.01); four chunks' addresses where there is one chunk 3.17 and 4.01 (3.01); one loop for both
// reduction orders 2.50 and 4.15 (2.74); the maximum in a loop for windows of four and nine too 2.61 and 4.26 (2.91).

struct ConvPoolArgs {
    const float* x;
    const float* wpk;
    const float* bias;
    const float* slope;
    float* y;
    int H, W, HW;                  // of the input
    int K, m_pad, nchunks, kdim, k_order, CB, RS, S;
    int sh, sw, ph, pw, dh, dw;
    int chunks_per_wave;
    int pool_r, pool_s, area;      // the window, which is also the stride
    int wins;                      // windows per tile
    int out_q, out_n;              // pooled columns, pooled outputs of a channel
    int n_tiles_n, n_tiles_m;
    unsigned x_bytes, w_bytes;
    int act;
    float lo, hi;
    FastDiv div_area, div_pool_s, div_out_q, div_rs, div_s, div_cb, div_n;
};

template <int KW>
__device__ __forceinline__ void conv_pool_tile(const ConvPoolArgs& p, const unsigned bid) {
    // The arguments requested together (see conv_tile): read where they are used they are six trips to the scalar cache, one behind the other.
    {
        const unsigned long long x = (unsigned long long)p.x, w = (unsigned long long)p.wpk, b = (unsigned long long)p.bias, l = (unsigned long long)p.slope;
        asm volatile("" ::"s"(x), "s"(w), "s"(b), "s"(l), "s"(p.H), "s"(p.W), "s"(p.HW), "s"(p.K), "s"(p.m_pad), "s"(p.nchunks), "s"(p.kdim), "s"(p.k_order), "s"(p.CB), "s"(p.RS), "s"(p.S),
                     "s"(p.chunks_per_wave), "s"(p.area), "s"(p.wins), "s"(p.n_tiles_n), "s"(p.n_tiles_m), "s"(p.x_bytes), "s"(p.w_bytes), "s"(p.act));
        asm volatile("" ::"s"(p.sh), "s"(p.sw), "s"(p.ph), "s"(p.pw), "s"(p.dh), "s"(p.dw), "s"(p.pool_r), "s"(p.pool_s), "s"(p.out_q), "s"(p.out_n), "s"(p.div_area.mul),
                     "s"(p.div_area.one), "s"(p.div_pool_s.mul), "s"(p.div_pool_s.one), "s"(p.div_out_q.mul), "s"(p.div_out_q.one), "s"(p.div_rs.mul), "s"(p.div_rs.one),
                     "s"(p.div_s.mul), "s"(p.div_s.one), "s"(p.div_cb.mul), "s"(p.div_cb.one), "s"(p.div_n.mul), "s"(p.div_n.one));
    }
    if (bid >= (unsigned)(p.n_tiles_n * p.n_tiles_m)) return;
    __shared__ float red[KW][4][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, kk = lane >> 4;
    const int tile_m = (int)quot_fast(bid, p.div_n), tile_n = (int)bid - tile_m * p.n_tiles_n;
    const int m0 = tile_m * 16;
    const int wi = (int)quot_fast((unsigned)j, p.div_area), pos = j - wi * p.area;
    const int win = tile_n * p.wins + wi;
    const bool valid = wi < p.wins && win < p.out_n;
    const int wy = (int)quot_fast((unsigned)win, p.div_out_q), wx = win - wy * p.out_q;
    const int pr = (int)quot_fast((unsigned)pos, p.div_pool_s), ps = pos - pr * p.pool_s;
    const int h0 = (wy * p.pool_r + pr) * p.sh - p.ph, w0 = (wx * p.pool_s + ps) * p.sw - p.pw;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)p.x, 0, p.x_bytes, 0x00027000);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void*)p.wpk, 0, p.w_bytes, 0x00027000);
    auto rsrc = [](const void* q, unsigned len) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(q), 0, q ? len : 0u, 0x00027000); };
    auto word = [](const __amdgpu_buffer_rsrc_t r, int off) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0)); };

    // What the end needs, requested with the operands.
    constexpr int PER = KW < 4 ? 4 / KW : 1;
    float bias_v[PER], slope_v[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int chan = m0 + 4 * kk + ((wave + i * KW) & 3);
        bias_v[i] = word(rsrc(p.bias, (unsigned)p.K * 4u), chan * 4);
        slope_v[i] = word(rsrc(p.slope, p.act == PAELLA_ACT_PRELU ? (unsigned)p.K * 4u : 0u), chan * 4);
    }

    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    const int begin = wave * p.chunks_per_wave, end = min(p.nchunks, begin + p.chunks_per_wave);
    auto batch = [&](auto count, auto tap_major, int c0) {  // chunks under way together
        constexpr int B = decltype(count)::value;
        constexpr bool TM = decltype(tap_major)::value;
        float a[B][2], b[B][2];
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const int c = c0 + u;
            const bool live = c < end;
            const int tap = TM ? (int)quot_fast((unsigned)c, p.div_cb) : 0;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int kl = 4 * (kk & 1) + (kk >> 1) + 2 * i;  // of the chunk's eight, in the order of the 32 x 32 instruction (conv_small.h)
                int chan, rs;
                bool ok = valid & live;
                if (TM) {
                    chan = (c - tap * p.CB) * 8 + kl;
                    rs = tap;
                } else {
                    const int k = c * 8 + kl;
                    chan = (int)quot_fast((unsigned)k, p.div_rs);
                    rs = k - chan * p.RS;
                    ok = ok & (k < p.kdim);
                }
                const int r = (int)quot_fast((unsigned)rs, p.div_s), s = rs - r * p.S;
                const int h = h0 + r * p.dh, w = w0 + s * p.dw;
                ok = ok & ((unsigned)h < (unsigned)p.H) & ((unsigned)w < (unsigned)p.W);
                b[u][i] = word(xr, ok ? (chan * p.HW + h * p.W + w) * 4 : -1);
                a[u][i] = word(wr, live ? ((c * 2 + (kl >> 2)) * p.m_pad + m0 + j) * 16 + (kl & 3) * 4 : -1);
            }
        }
#pragma unroll
        for (int u = 0; u < B; ++u)
            if (c0 + u < end)
#pragma unroll
                for (int i = 0; i < 2; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][i], b[u][i], acc, 0, 0, 0);
    };
    auto chunks = [&](auto tap_major) {
        if (p.chunks_per_wave == 1) {  // (a first layer: the addresses of chunks that are not there take as long as a trip to memory)
            if (begin < end) batch(std::integral_constant<int, 1>{}, tap_major, begin);
        } else {
            for (int c0 = begin; c0 < end; c0 += 4) batch(std::integral_constant<int, 4>{}, tap_major, c0);
        }
    };
    if (p.k_order) chunks(std::true_type{});
    else chunks(std::false_type{});
#pragma unroll
    for (int e = 0; e < 4; ++e) red[wave][e][lane] = acc[e];
    __syncthreads();
    // Register e of the tile holds, in lane (j, kk), channel m0 + 4 * kk + e at column j; a wave finishes one of them, or two of two waves.
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = wave + i * KW;
        if (e >= 4) break;
        float v = red[0][e][lane];  // wave order, as in conv_tile
#pragma unroll
        for (int w = 1; w < KW; ++w) v += red[w][e][lane];
        const int chan = m0 + 4 * kk + e;
        v += bias_v[i];
        float none = 0.f;  // where conv_tile adds a residual that is not there: -0 becomes +0
        asm volatile("" : "+v"(none));
        v += none;
        v = apply_act(v, p.act, slope_v[i], p.lo, p.hi);
        const int first = (lane & 48) + wi * p.area;
        float m = -FLT_MAX;  // in the order of pool_window
        if (p.area == 4) {
#pragma unroll
            for (int t = 0; t < 4; ++t) m = fmaxf(m, __shfl(v, first + t, 64));
        } else if (p.area == 9) {
#pragma unroll
            for (int t = 0; t < 9; ++t) m = fmaxf(m, __shfl(v, first + t, 64));
        } else {
            for (int t = 0; t < p.area; ++t) m = fmaxf(m, __shfl(v, first + t, 64));
        }
        if (valid && pos == 0 && chan < p.K) store_out(p.y + (size_t)chan * p.out_n + win, m);
    }
}

template <int KW>
__global__ __launch_bounds__(64 * KW) void conv_pool_kernel(ConvPoolArgs args) {
    int idx = 0;  // see conv_mfma_kernel
    asm volatile("" : "+s"(idx));
    conv_pool_tile<KW>((&args)[idx], blockIdx.x);
}

// The same for up to PAELLA_CONV_PACK_MAX requests (launch packing).
struct ConvPoolGroupArgs {
    unsigned grid;                           // workgroups of each
    FastDiv div_grid;
    ConvPoolArgs m[PAELLA_CONV_PACK_MAX];    // only the used entries are written to the argument ring
};

template <int KW>
__global__ __launch_bounds__(64 * KW) void conv_pool_group_kernel(ConvPoolGroupArgs g) {
    const unsigned idx = quot_fast(blockIdx.x, g.div_grid);
    conv_pool_tile<KW>(g.m[idx], blockIdx.x - idx * g.grid);
}
