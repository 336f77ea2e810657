// The general kernel's stride-1 launches of one channel tile and two planes per workgroup (the coarse levels of a network, a tile or two per CU), pipelined.
//
// conv3_mx_k<.., MT 1, NT 2> is a chain there: a chunk's halo through registers into LDS, a barrier, its first weights the same way, a barrier, then pairs that each wait for their
// fragments: 11 K cycles per input block of e4m3, of which 14 pairs x 2 products are 1.8 K. Here the same products in the same order (tap-major inside a chunk of CB blocks) with
// everything requested ahead:
//   * the halo of chunk c + 1 comes by LDS-DMA into the second of two buffers while chunk c is multiplied (positions outside the volume from the constant page);
//   * the weights come by LDS-DMA in stages of seven pairs into a ring of three, two stages ahead;
//   * fragments are fetched two pairs ahead into four register sets; a chunk is unrolled whole, so the sets and the taps' offsets are constants and there is no pair table. A chunk of NP
//     pairs takes the sets in NP % 3 groups of four and then groups of three, so that any three pairs in a row - into the next chunk too - have sets of their own;
//   * one barrier per stage, in front of its first fetch: then every wavefront is done with the stage before, whose ring slot (and with a chunk its halo buffer) takes the next requests.
// What bounds it: 2.1 us per block of e4m3 alone on its CU (256 -> 256 at 2 x 16^3, eight blocks, 25 us in all), of which the products between their barriers take 1.3 (28 in a row per
// wavefront on two accumulators), the fragments' reads 0.45 (three of 2.3 KB per two products and wavefront, 192 cycles of the CU's LDS beside 128 of the matrix pipe), the copies 0.35.
// Counted waits: every wavefront issues NW copies per stage and NHO per chunk, the weights first.
#pragma once

template <int FMT, int CB, int PPS> struct pipe_t {
    static constexpr int HY = 10, HX = 18, TT = 4 * HY * HX, NG = (TT + 63) / 64, TTP = NG * 64, NH = fmt_t<FMT>::NH, WTILE = fmt_t<FMT>::WTILE, KT = WTILE / 1024;
    static constexpr int SC_O = NH * TTP * 16, HB = SC_O + TTP * 4, HBUF = CB * HB;                     // a block's halo: rows [half][position][16 B], then a scale word per position
    static constexpr int NP = (27 * CB + 1) / 2, NSTG = (NP + PPS - 1) / PPS;                  // pairs of a chunk, of a weight stage; stages of a chunk
    static constexpr int NCP = PPS * KT, NPC = NCP + (PPS + 3) / 4, SLOT = NPC * 1024, NS = 3;          // a stage: 1 KiB pieces of codes, then of four pairs' scale words each
    static constexpr int NW = (NPC + 3) / 4, NHO = CB * 3 * (NH + 1);
    static constexpr size_t LDS = (size_t)NS * SLOT + 2 * HBUF;
    static_assert(NG == 12 && NSTG >= 2 && NHO + NW <= 63);
    static constexpr int set(int q) { return q < 4 * (NP % 3) ? q % 4 : (q - 4 * (NP % 3)) % 3; }
    static constexpr int tap_pos(int u) { return ((u / CB / 9) * HY + (u / CB / 3) % 3) * HX + u / CB % 3; }
    static constexpr int row_off(int u) { return u % CB * HB + tap_pos(u) * 16; }
    static constexpr int sc_off(int u) { return u % CB * HB + SC_O + tap_pos(u) * 4; }
};

template <int FMT, int OUT, int CB, int PPS>
__global__ void __launch_bounds__(256, 2) conv3_pipe_k(const conv_args a) {
    using P = pipe_t<FMT, CB, PPS>;
    constexpr int NH = P::NH, WTILE = P::WTILE, NP = P::NP, NSTG = P::NSTG, NW = P::NW, NHO = P::NHO, HX = P::HX, HY = P::HY;
    extern __shared__ __align__(16) unsigned char lds[];
    const unsigned lds0 = (unsigned)(size_t)lds;
    constexpr unsigned halo_o = P::NS * P::SLOT;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 31, h = lane >> 5;
    unsigned tile;                                              // (conv3_mx_k's tile order)
    {
        const unsigned per = (a.ntiles + 7u) / 8u;
        tile = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
        if (tile >= a.ntiles) return;
    }
    int tt = (int)tile;
    const int cs = tt % a.ncs; tt /= a.ncs;
    const int tx = tt % a.ntx; tt /= a.ntx;
    const int ty = tt % a.nty; tt /= a.nty;
    const int tz = tt % a.ntz; const int n = tt / a.ntz;
    const int ox0 = tx * 16, oy0 = ty * 8, oz0 = tz * 2;
    const int lz = wave >> 1, ly0 = (wave & 1) * 4;
    const size_t Sin = (size_t)a.D * a.H * a.W;
    const int nch = a.nbt / CB;

    // ---- requests ----
    const size_t wq_ps = (size_t)a.nmt_all * WTILE, wsc_ps = (size_t)a.nmt_all * 256;
    const uint8_t *wq = a.wq + (size_t)cs * WTILE, *wsc = a.wsc + (size_t)cs * 256;
    unsigned wvo[NW];                                           // the lane's byte offset inside a stage for piece wave + 4 k (pieces past the last: that one again)
    static_for<NW>([&](auto K) {
        constexpr int k = decltype(K)::value;
        const int i = min(wave + 4 * k, P::NPC - 1);
        wvo[k] = i >= P::NCP ? (unsigned)min(4 * (i - P::NCP) + (lane >> 4), PPS - 1) * (unsigned)wsc_ps + (lane & 15) * 16 : (unsigned)(i / P::KT) * (unsigned)wq_ps + (i % P::KT) * 1024 + lane * 16;
    });
    auto wreq = [&](int pair, unsigned so) {
        static_for<NW>([&](auto K) {
            constexpr int k = decltype(K)::value;
            const int i = min(wave + 4 * k, P::NPC - 1);
            dma16s(wvo[k], i >= P::NCP ? wsc + (size_t)pair * wsc_ps : wq + (size_t)pair * wq_ps, lds0 + so + (unsigned)i * 1024u);
        });
    };
    unsigned vox[3]; bool in[3];                                // the lane's halo positions (groups wave, wave + 4, wave + 8): voxel, inside the volume
    static_for<3>([&](auto K) {
        constexpr int k = decltype(K)::value;
        const int pos = (wave + 4 * k) * 64 + lane, pz = pos / (HY * HX), rem = pos - pz * (HY * HX), py = rem / HX, px = rem - py * HX;
        const int gz = oz0 - 1 + a.zi0 + pz, gy = oy0 - 1 + py, gx = ox0 - 1 + px;
        in[k] = pos < P::TT && (unsigned)gz < (unsigned)a.D && (unsigned)gy < (unsigned)a.H && (unsigned)gx < (unsigned)a.W;
        vox[k] = (unsigned)((gz * a.H + gy) * a.W + gx);
    });
    auto hreq = [&](int b0, unsigned hb) {
        static_for<CB>([&](auto B) {
            constexpr int bl = decltype(B)::value;
            const int sb = b0 + bl, seg = sb >= a.nb0p, blk = seg ? sb - a.nb0p : sb, nbs = seg ? a.nbs[1] : a.nbs[0];
            const bool bok = blk < nbs;                         // (uniform) the block holds stored channels
            const size_t plane = ((size_t)n * nbs + (bok ? blk : 0)) * Sin;
            const uint8_t *rb = (seg ? a.xq[1] : a.xq[0]) + plane * (16 * NH), *sp = (seg ? a.xsc[1] : a.xsc[0]) + plane;
            static_for<3>([&](auto K) {
                constexpr int k = decltype(K)::value;
                const bool go = in[k] && bok;
                const uint8_t *row = go ? rb + (size_t)vox[k] * (16 * NH) : a.zpage;
                const unsigned d = lds0 + hb + bl * P::HB + (unsigned)(wave + 4 * k) * 1024u;
                dma16(row, d);
                if constexpr (NH == 2) dma16(row + 16, d + P::TTP * 16);
                dma1(go ? sp + vox[k] : a.zpage + 64, lds0 + hb + bl * P::HB + P::SC_O + (unsigned)(wave + 4 * k) * 256u);
            });
        });
    };
    wreq(0, 0u);
    hreq(0, halo_o);
    wreq(PPS, P::SLOT);
    conv_epi_consts<1, false>(a, lds, cs, tid);

    // ---- fragments ----
    const int p00 = (lz * HY + ly0 + (r >> 4)) * HX + (r & 15);
    const unsigned ab0 = ((NH == 2 ? h * P::TTP : 0) + p00) * 16, sb0 = p00 * 4;
    constexpr unsigned ABJ = 2 * HX * 16, SBJ = 2 * HX * 4;
    v16f acc[1][2];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[0][j][i] = 0.f;
    v8i fb[4][2], fa[4]; int sb[4][2], sa[4];
    unsigned so = 2 * P::SLOT;                                  // the ring slot of the stage being fetched
    auto fetch = [&](auto Q, unsigned hb) {                     // pair Q of the chunk whose halo lies at hb
        constexpr int q = decltype(Q)::value, s = P::set(q), uA = 2 * q, uB = 2 * q + 1 < 27 * CB ? 2 * q + 1 : 2 * q;      // (the unit past the last: zero weights on the one before)
        constexpr int oA = P::row_off(uA), oB = P::row_off(uB), sA = P::sc_off(uA), sB = P::sc_off(uB);
#pragma unroll
        for (int j = 0; j < 2; j++) {
            if constexpr (FMT == 8) {
                const v4i lo = *(const v4i *)(lds + (hb + ab0) + oA + j * ABJ), hi = *(const v4i *)(lds + (hb + ab0) + oB + j * ABJ);
                fb[s][j] = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            } else { const v4i lo = *(const v4i *)(lds + (hb + ab0 + (h ? oB - oA : 0)) + oA + j * ABJ); fb[s][j] = (v8i){lo[0], lo[1], lo[2], lo[3], 0, 0, 0, 0}; }
            sb[s][j] = *(const int *)(lds + (hb + sb0 + (h ? sB - sA : 0)) + sA + j * SBJ);
        }
        const unsigned wo = so + lane * 16;
        const v4i lo = *(const v4i *)(lds + wo + q % PPS * WTILE);
        if constexpr (FMT == 8) { const v4i hi = *(const v4i *)(lds + wo + q % PPS * WTILE + 1024); fa[s] = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}; }
        else fa[s] = (v8i){lo[0], lo[1], lo[2], lo[3], 0, 0, 0, 0};
        sa[s] = *(const int *)(lds + so + lane * 4 + PPS * WTILE + q % PPS * 256);
    };
    // the first fetch of stage LS of chunk c is next: its weights (and the chunk's halo) have landed when at most the copies requested after them are outstanding - the weights of the stage
    // after it, and in the second and third stage of a chunk the next chunk's halo
    auto enter = [&](auto LS, int c) {
        constexpr int ls = decltype(LS)::value;
        const bool more = c + 1 < nch;
        if ((ls == 1 || ls == 2) && more) wait_vm<NW + NHO>(); else wait_vm<NW>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const unsigned prev = so;                               // the stage before's slot takes the stage after next (past the last: the first pairs again, not read)
        so = so + P::SLOT < P::NS * P::SLOT ? so + P::SLOT : 0u;
        if constexpr (ls + 2 < NSTG) wreq(c * NP + (ls + 2) * PPS, prev);
        else wreq(more ? (c + 1) * NP + (ls + 2 - NSTG) * PPS : 0, prev);
        if (ls == 0 && more) hreq((c + 1) * CB, halo_o + ((c + 1) & 1) * P::HBUF);
    };
    enter(std::integral_constant<int, 0>{}, 0);
    fetch(std::integral_constant<int, 0>{}, halo_o);
    fetch(std::integral_constant<int, 1>{}, halo_o);
    for (int c = 0; c < nch; c++) {
        const unsigned hb = halo_o + (c & 1) * P::HBUF, hn = halo_o + ((c + 1) & 1) * P::HBUF;
        static_for<NP>([&](auto Q) {
            constexpr int q = decltype(Q)::value, f = q + 2, s = P::set(q);
            if constexpr (f < NP) {
                if constexpr (f % PPS == 0) enter(std::integral_constant<int, f / PPS>{}, c);
                fetch(std::integral_constant<int, f>{}, hb);
            } else if (c + 1 < nch) {                           // (uniform)
                if constexpr (f == NP) enter(std::integral_constant<int, 0>{}, c + 1);
                fetch(std::integral_constant<int, f - NP>{}, hn);
            }
#pragma unroll
            for (int j = 0; j < 2; j++)
                acc[0][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[s], fb[s][j], acc[0][j], FMT == 8 ? 0 : 4, FMT == 8 ? 0 : 4, 0, sa[s], 0, sb[s][j]);
            asm volatile("" : "+a"(acc[0][0]), "+a"(acc[0][1]) : : "memory");      // (without it the products sink below the chunk's fetches)
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    wait_vm<0>();                                               // (the copies of stages past the last)
    __syncthreads();
    // (conv3_mx_k's epilogues: a divided slice of three tiles keeps the whole one's records)
    if (a.one3) { conv_epilogue<1, 2, OUT, false, false, true, false, true>(a, acc, lds, tile, n, cs, oz0, oy0, ox0, lz, ly0, tid); return; }
    if (a.Co > 16) conv_epilogue<1, 2, OUT, false, false, true>(a, acc, lds, tile, n, cs, oz0, oy0, ox0, lz, ly0, tid);
    else conv_epilogue<1, 2, OUT, false>(a, acc, lds, tile, n, cs, oz0, oy0, ox0, lz, ly0, tid);
}

// pairs of a weight stage: seven, or three where that lets two workgroups share a CU (80 KB: e4m3, e2m1 in chunks of one or two blocks) and more tiles than CUs want it
static inline int conv3_pipe_pps(int fmt, int CB, size_t tiles) { return tiles > 256 && (fmt == 8 || CB <= 2) ? 3 : 7; }
static inline size_t conv3_pipe_lds(int fmt, int CB, int pps) {
    if (pps == 3) return fmt == 8 ? pipe_t<8, 1, 3>::LDS : CB == 1 ? pipe_t<4, 1, 3>::LDS : pipe_t<4, 2, 3>::LDS;
    return fmt == 8 ? pipe_t<8, 1, 7>::LDS : CB == 1 ? pipe_t<4, 1, 7>::LDS : CB == 2 ? pipe_t<4, 2, 7>::LDS : CB == 3 ? pipe_t<4, 3, 7>::LDS : pipe_t<4, 4, 7>::LDS;
}
static_assert(pipe_t<8, 1, 3>::LDS + 3 * 128 + 1024 <= 80 * 1024 && pipe_t<4, 2, 3>::LDS + 3 * 128 + 1024 <= 80 * 1024 && pipe_t<4, 4, 7>::LDS + 3 * 128 + 1024 <= 160 * 1024, "two workgroups per CU; one");
template <int FMT, int OUT, int CB, int PPS>
static void launch_pipe_t(const conv_args &a, size_t smem) {
    static bool attr[8];
    int d = 0; MIRT(hipGetDevice(&d)); d &= 7;
    if (!attr[d]) { MIRT(hipFuncSetAttribute((const void *)conv3_pipe_k<FMT, OUT, CB, PPS>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024)); attr[d] = true; }
    const unsigned per = (a.ntiles + 7u) / 8u;
    conv3_pipe_k<FMT, OUT, CB, PPS><<<per * 8u, 256, smem>>>(a);
    MICK();
    snprintf(g_last_kernel, sizeof g_last_kernel, "conv3_pipe_k for conv3_mx_k<fmt %d, stride 1, MT 1, NT 2, out %d, epi 0> stage %d CB %d tiles %u", FMT, OUT, PPS, CB, a.ntiles);
}
template <int FMT, int OUT>
static void launch_pipe(const conv_args &a, size_t smem) {
    const bool three = conv3_pipe_pps(FMT, a.CB, a.ntiles) == 3;
    if constexpr (FMT == 8) { if (three) launch_pipe_t<8, OUT, 1, 3>(a, smem); else launch_pipe_t<8, OUT, 1, 7>(a, smem); }
    else switch (a.CB) {
        case 1: if (three) launch_pipe_t<4, OUT, 1, 3>(a, smem); else launch_pipe_t<4, OUT, 1, 7>(a, smem); break;
        case 2: if (three) launch_pipe_t<4, OUT, 2, 3>(a, smem); else launch_pipe_t<4, OUT, 2, 7>(a, smem); break;
        case 3: launch_pipe_t<4, OUT, 3, 7>(a, smem); break;
        default: launch_pipe_t<4, OUT, 4, 7>(a, smem);
    }
}
