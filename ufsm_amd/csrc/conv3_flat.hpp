// conv3_mx_k's form for launches with about one small tile per CU (the coarse levels of a window of 64 .. 128 voxels): flat runs of output voxels, the taps
// split over the wavefronts of a workgroup, the input two pairs of blocks ahead in LDS. Included by conv3_kernel.hpp.
//
// What bounds such a launch on the staged kernels is a chain of latencies, not a rate: 256 -> 256 at 2 x 16^3 is 256 workgroups whose matrix work is 6 us and
// whose eight halo chunks are staged, waited for and multiplied one after the other, 37 us. Here
//   * a workgroup's tile is 128 consecutive output voxels (four runs of 32; no voxel is lost to tile edges of a ragged volume) x 64 channels, so that a launch
//     of the coarse levels fills the CUs once, and every input fragment feeds two products and every weight fragment four;
//   * the eight wavefronts split the 27 taps (waves 0 - 2 take four, the others three: seven per SIMD) and each keeps all eight accumulators; the tile's input
//     is walked in pairs of 32-channel blocks, one tap of a pair being one K step of the matrix instruction. A wavefront's taps are the same for every pair;
//   * because a tile's voxels are consecutive, what the nine taps of a plane kz can reach is one range of 128 + 2 W + 2 consecutive voxels of each stored block: three ranges
//     are copied to LDS as they are, without coordinates, into a ring of three slots (five in e2m1), two pairs ahead. A lane whose tap lies outside the volume reads
//     a row of zeros instead, chosen once per tap and run (ten bits in a register);
//   * the weights come from the caches into registers one or two taps ahead; the five wavefronts with three taps do the copies. One barrier per pair, before a
//     wavefront's last tap: behind it the next pair's first rows are fetched under the last products;
//   * the eight partial accumulators of a tile meet in LDS and are added in wavefront order (the same bits on every run), each wavefront then runs the shared
//     epilogue on one of the eight 32 x 32 tiles. Statistics records are the K-split kernel's: one per run of 32 voxels, none across a multiple of four planes.
// Measured, kernel time: 256 -> 256 at 2 x 16^3 37.2 -> 22.2 us, 384 -> 128 at 22 x 26^2 62.9 -> 26.5; in e2m1 192 -> 192 at 2 x 16^3 36.7 -> 15.4. A tile of 12
// blocks takes 43 000 cycles: 2 600 to the first copy, 3 000 until it has landed, 4 600 per pair (3 584 of products on three of the SIMDs), 4 500 for the exchange of 256 KB
// through LDS (4 096 at its rate), 2 100 for the epilogue. The two rings deeper or the rows fetched a tap ahead changed nothing beyond 2 %.
#pragma once

// FMT 8: three slots of two input blocks in LDS, FMT 4: five (rows and scale words are half as long)
template <int FMT> struct flat_t {
    static constexpr int TT = 640, TTS = TT + 4;              // staged positions, ten copy groups of 64; the row of zeros for taps outside the volume is position TT
    static constexpr int NH = fmt_t<FMT>::NH, ROWS = 2 * NH * TTS * 16, SLOT = ROWS + 2 * TTS * 4, NS = FMT == 8 ? 3 : 5;
    static constexpr int WMAX = (TT - 3 * 130) / 6;           // three slabs of 128 + 2 W + 2 positions
    static constexpr int EXCH = 8 * 8 * 2 * 64 * 16;          // the exchange of the partial accumulators, half of their registers at a time
    static constexpr int LDS = NS * SLOT > EXCH ? NS * SLOT : EXCH;
};
template <int FMT, int OUT>
__global__ void __launch_bounds__(512, 1) conv3_flat_k(const conv_args a) {
    using F = flat_t<FMT>;
    constexpr int RB = fmt_t<FMT>::RB, WTILE = fmt_t<FMT>::WTILE, NH = F::NH, TTS = F::TTS, MT = 2, NT = 4;
    extern __shared__ __align__(16) unsigned char lds[];
    const unsigned lds0 = (unsigned)(size_t)lds;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 31, h = lane >> 5;
    // consecutive workgroup ids land on different XCDs (gridDim.x is a multiple of 8): each XCD takes a contiguous range of tiles, with all their channel slices
    const unsigned per = gridDim.x >> 3;
    const int g = (int)((blockIdx.x & 7u) * per + (blockIdx.x >> 3)), cs2 = (int)blockIdx.y, n = (int)blockIdx.z;
    if (4 * g >= a.ntz) return;
    const int HW = a.H * a.W, Scol = a.Do * HW, off = a.zc & 31;
    const size_t Sin = (size_t)a.D * HW;
    const int f0 = g * 128 - off;                             // first output voxel of the tile (negative: a z-range whose first run starts before it)
    // ---- weights ----
    const unsigned wq_ps = (unsigned)a.nmt_all * WTILE, wsc_ps = (unsigned)a.nmt_all * 256;
    auto wrsrc = [](const uint8_t *p) { return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, 0x7fffffff, 0x00027000); };
    const auto wrs = wrsrc(a.wq + (size_t)cs2 * MT * WTILE), srs = wrsrc(a.wsc + (size_t)cs2 * MT * 256);
    struct wf { v4i lo[MT], hi[MT]; int s[MT]; };
    auto wload = [&](int s, int k, wf &w) {               // (one lane offset and a uniform one per tap: no 64-bit lane addresses)
                const unsigned gp = (unsigned)(s * 27 + wave + 8 * k);
                const int oq = (int)(gp * wq_ps), os = (int)(gp * wsc_ps);
    #pragma unroll
                for (int m = 0; m < MT; m++) {
                    w.lo[m] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wrs, lane * 16, oq + m * WTILE, 0));
                    if constexpr (NH == 2) w.hi[m] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wrs, lane * 16 + 1024, oq + m * WTILE, 0)); else w.hi[m] = (v4i){0, 0, 0, 0};
                    w.s[m] = __builtin_amdgcn_raw_buffer_load_b32(srs, lane * 4, os + m * 256, 0);
                }
            };
    const int PL = 130 + 2 * a.W;                             // positions of a staged slab: those a plane of taps can reach from the tile's voxels
    // ---- copies: waves 3 .. 7 (those with three taps) own the (block of the pair, group of 64 positions) items wave - 3 + 5 k ----
    constexpr int NI = 4;
    auto copy = [&](int s, unsigned so, auto K) {             // item K of block pair s into the slot at so
        constexpr int k = decltype(K)::value;
        const int i = wave - 3 + 5 * k, sel = i & 1, rd = i >> 1, b = 2 * s + sel, seg = b >= a.nb0p, blk = seg ? b - a.nb0p : b;
        const size_t pl = ((size_t)n * a.nbs[seg] + blk) * Sin;
        const uint8_t *q = a.xq[seg] + pl * RB, *sc = a.xsc[seg] + pl;
        // the lane's position and the voxel it stages (what lies outside the tensor is never read: its taps read the row of zeros); formed per request, no register held for it
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int pos = rd * 64 + ln, dz = HW - PL;
        const int vi = f0 + (a.zi0 - 1) * HW - a.W - 1 + pos + (pos >= PL ? dz : 0) + (pos >= 2 * PL ? dz : 0);
        const unsigned v = (unsigned)min(max(vi, 0), (int)Sin - 1);
        const unsigned ro = lds0 + so + (unsigned)(sel * (NH * TTS * 16) + rd * 1024);
        dma16s(v * RB, q, ro);
        if constexpr (NH == 2) dma16s(v * RB + 16, q, ro + TTS * 16);
        dma1s(v, sc, lds0 + so + (unsigned)(F::ROWS + sel * (TTS * 4) + rd * 256));
    };
    const int ns = a.nbt >> 1;
    if (wave >= 3) {
        static_for<NI>([&](auto K) { copy(0, 0u, K); });
        static_for<NI - 1>([&](auto K) { copy(min(1, ns - 1), (unsigned)F::SLOT, K); });      // (its last item goes out in the first step)
    } else if (wave == 0) {                                   // the rows of zeros of every slot (and their scale words)
        for (int i = lane; i < F::NS * 2 * NH; i += 64) *(v4i *)(lds + (i / (2 * NH)) * F::SLOT + (i % (2 * NH)) * (TTS * 16) + F::TT * 16) = (v4i){0, 0, 0, 0};
        for (int i = lane; i < F::NS * 2; i += 64) *(int *)(lds + (i >> 1) * F::SLOT + F::ROWS + ((i & 1) * TTS + F::TT) * 4) = 0;
    }
    conv_epi_consts<MT, false>(a, lds, cs2, tid);
    // ---- the lane's voxel of each run: which of the offsets -1, 0, +1 stay inside the volume, per dimension ----
    const float rW = 1.f / (float)a.W, rH = 1.f / (float)a.H;
    auto udiv = [](int v, int d, float rd) {                  // v / d by the reciprocal (fewer than 2^24 voxels: off by one at most)
        int q = (int)((float)v * rd);
        const int e = v - q * d;
        return e < 0 ? q - 1 : e >= d ? q + 1 : q;
    };
    unsigned vm[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const int col = f0 + j * 32 + r;
        const bool ok = (unsigned)col < (unsigned)Scol;
        const unsigned cc = ok ? (unsigned)col : 0u;
        const int row = udiv((int)cc, a.W, rW), x = (int)cc - row * a.W, zo = udiv(row, a.H, rH), y = row - zo * a.H, z = zo + a.zi0;
        unsigned m = 0;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            m |= ((unsigned)(z + d - 1) < (unsigned)a.D ? 1u : 0u) << d;
            m |= ((unsigned)(y + d - 1) < (unsigned)a.H ? 1u : 0u) << (3 + d);
            m |= ((unsigned)(x + d - 1) < (unsigned)a.W ? 1u : 0u) << (6 + d);
        }
        vm[j] = ok ? m : 0u;
    }
    v16f acc[MT][NT], sum[1][1];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[m][j][i] = 0.f;
    // ---- K loop of a wavefront: NK taps of every pair of blocks, the weights PD taps ahead in registers ----
    auto kloop = [&](auto NKc, auto PDc) {
        constexpr int NK = decltype(NKc)::value, PD = decltype(PDc)::value, RS = PD + 1, WL = MT * (NH + 1);      // (WL: loads of a tap's weights)
        static_assert(NK % RS == 0 || RS == 2, "the ring's sets follow the tap");
        constexpr bool COPY = NK == 3;
        // the staged position a run's lane reads for each tap, ten bits apiece
        unsigned ad[(NK + 2) / 3][NT];
#pragma unroll
        for (int j = 0; j < NT; j++) {
            static_for<(NK + 2) / 3>([&](auto I) { ad[decltype(I)::value][j] = 0u; });
            static_for<NK>([&](auto K) {
                constexpr int k = decltype(K)::value;
                const int t = wave + 8 * k, kz = t / 9, ky = t / 3 - 3 * kz, kx = t % 3;
                const unsigned bit = (1u << kz) | (8u << ky) | (64u << kx);
                ad[k / 3][j] |= (unsigned)((vm[j] & bit) == bit ? kz * PL + ky * a.W + kx + r + 32 * j : F::TT) << (10 * (k % 3));
            });
        }
        wf fa[RS];
        static_for<PD>([&](auto K) { wload(0, decltype(K)::value, fa[decltype(K)::value]); });
        if constexpr (COPY) wait_vm<(NI - 1) * (NH + 1) + PD * WL>();      // block pair 0 has landed (what was requested after it has not)
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        v8i B[NT]; int sb[NT];
        // lane half h reads half h of a row (e4m3) or the row of block h (e2m1), and block h's scale word
        const unsigned hr = (unsigned)(h * TTS * 16), hs = (unsigned)(F::ROWS + h * TTS * 4);
        auto fetch = [&](int j, unsigned so, auto K) {
            constexpr int k = decltype(K)::value;
            const unsigned pos = (ad[k / 3][j] >> (10 * (k % 3))) & 1023u;
            const unsigned char *p = lds + (so + hr + pos * 16u);
            const v4i lo = *(const v4i *)p;
            if constexpr (NH == 2) {
                const v4i hi = *(const v4i *)(p + 2 * TTS * 16);
                B[j] = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            } else B[j] = (v8i){lo[0], lo[1], lo[2], lo[3], 0, 0, 0, 0};
            sb[j] = *(const int *)(lds + (so + hs + pos * 4u));
        };
        static_for<NT>([&](auto J) { fetch(decltype(J)::value, 0u, std::integral_constant<int, 0>{}); });
        auto next = [&](unsigned o) { return o + F::SLOT == (unsigned)(F::NS * F::SLOT) ? 0u : o + F::SLOT; };
        unsigned so = 0;                                      // slot of this step's pair
        int s = 0;
        do {                                                  // (at least one pair)
            const int s1 = min(s + 1, ns - 1), s2 = min(s + 2, ns - 1);      // (past the end: copied and loaded again, into slots and registers that nothing reads)
            const unsigned so1 = next(so), so2 = next(so1);
#pragma unroll
            for (int j = 0; j < NT; j++)                      // (opaque: the addresses are formed per tap, not kept in registers over the loop)
                for (int i = 0; i < (NK + 2) / 3; i++) asm volatile("" : "+v"(ad[i][j]));
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int j = 0; j < NT; j++) asm volatile("" : "+a"(acc[m][j]));      // (the accumulators keep the accumulation registers: the rest fits the other half)
            static_for<NK>([&](auto K) {
                constexpr int k = decltype(K)::value;
                if constexpr (k + PD < NK) wload(s, k + PD, fa[(k + PD) % RS]); else wload(s1, k + PD - NK, fa[(k + PD) % RS]);
                if constexpr (k == NK - 1) {
                    // the next pair is complete - its last copy went out two taps ago, all but the weights of two taps before that - and nobody reads the pair before this one
                    if constexpr (COPY) wait_vm<2 * WL>();
                    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                    if constexpr (COPY) static_for<NI - 1>([&](auto I) { copy(s2, so2, I); });
                } else if constexpr (COPY && k == 0) copy(s1, so1, std::integral_constant<int, NI - 1>{});
                const wf &w = fa[k % RS];
                // a run's two products, then its row for the next tap into the registers they leave: the reads of one run wait behind the products of the other three
                static_for<NT>([&](auto J) {
                    constexpr int j = decltype(J)::value;
#pragma unroll
                    for (int m = 0; m < MT; m++) {
                        const v8i A = {w.lo[m][0], w.lo[m][1], w.lo[m][2], w.lo[m][3], w.hi[m][0], w.hi[m][1], w.hi[m][2], w.hi[m][3]};
                        acc[m][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A, B[j], acc[m][j], FMT == 8 ? 0 : 4, FMT == 8 ? 0 : 4, 0, w.s[m], 0, sb[j]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    fetch(j, k + 1 < NK ? so : so1, std::integral_constant<int, (k + 1) % NK>{});
                    __builtin_amdgcn_sched_barrier(0);
                });
            });
            so = so1;
        } while (++s < ns);
        if constexpr (COPY) wait_vm<0>();                     // (no copy lands in what the exchange writes)
        asm volatile("s_barrier" ::: "memory");
        // ---- the eight partial accumulators of tile (m, j) meet at wavefront 4 m + j, which adds them in wavefront order, eight registers at a time ----
        float4 *part = (float4 *)lds;
        static_for<2>([&](auto P) {
            constexpr int p = decltype(P)::value;
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int j = 0; j < NT; j++)
#pragma unroll
                    for (int k = 0; k < 2; k++)
                        part[((wave * 8 + m * 4 + j) * 2 + k) * 64 + lane] = make_float4(acc[m][j][8 * p + 4 * k], acc[m][j][8 * p + 4 * k + 1], acc[m][j][8 * p + 4 * k + 2], acc[m][j][8 * p + 4 * k + 3]);
            __syncthreads();
#pragma unroll
            for (int k = 0; k < 2; k++) {
                float4 t = part[(wave * 2 + k) * 64 + lane];
#pragma unroll
                for (int w = 1; w < 8; w++) { const float4 u = part[((w * 8 + wave) * 2 + k) * 64 + lane]; t.x += u.x; t.y += u.y; t.z += u.z; t.w += u.w; }
                sum[0][0][8 * p + 4 * k] = t.x; sum[0][0][8 * p + 4 * k + 1] = t.y; sum[0][0][8 * p + 4 * k + 2] = t.z; sum[0][0][8 * p + 4 * k + 3] = t.w;
            }
            if (p == 0) __syncthreads();
        });
    };
    if (wave < 3) __builtin_amdgcn_s_setprio(1);              // (four taps to the others' three)
    if (wave < 3) kloop(std::integral_constant<int, 4>{}, std::integral_constant<int, 1>{});
    else kloop(std::integral_constant<int, 3>{}, std::integral_constant<int, 2>{});
    const int m = wave >> 2, j = wave & 3, run = g * 4 + j, cs = cs2 * MT + m;
    if (run >= a.ntz || cs >= a.nmt_all) return;              // (no barrier follows)
    // the run's statistics records, as the K-split kernel's: a run that meets a multiple of four planes of the whole tensor leaves one per side
    int rec = n * a.nty + g * 4, seg = 33; const int step = a.ntx;
    if (step) {
        const int f = run * 32 - off, zg = f < 0 ? -1 : f / step;
        seg = (zg + 1) * step - f;
        rec += zg + (off > 0);
    }
    const int col = f0 + j * 32 + r;
    const long long ovx[1] = {(unsigned)col < (unsigned)Scol ? (long long)col + (long long)a.yzo * HW : -1};
    conv_epilogue<1, 1, OUT, false, false, true, false, true, 1, true, true, true>(a, sum, lds + m * 128, (unsigned)rec, n, cs, 0, 0, 0, 0, 0, j * 64 + lane, ovx, seg, step, a.zc > 31, f0 + j * 32);
}
template <int FMT, int OUT>
static void launch_flat(const conv_args &a, size_t smem) {
    static bool attr[8];
    int d = 0; MIRT(hipGetDevice(&d)); d &= 7;
    if (!attr[d]) { MIRT(hipFuncSetAttribute((const void *)conv3_flat_k<FMT, OUT>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024)); attr[d] = true; }
    conv3_flat_k<FMT, OUT><<<dim3((a.ngrp + 7u) / 8u * 8u, (unsigned)(a.nmt_all + 1) / 2, (unsigned)a.N), 512, smem>>>(a);
    MICK();
    snprintf(g_last_kernel, sizeof g_last_kernel, "conv3_flat_k<fmt %d, out %d> blocks %d tiles %u", FMT, OUT, a.nbt, a.ngrp * (unsigned)((a.nmt_all + 1) / 2 * a.N));
}
