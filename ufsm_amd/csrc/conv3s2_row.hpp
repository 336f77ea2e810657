// The 3x3x3 stride-2 conv of one input block into one channel tile (the level-0 down conv of a U-Net), on rows of more than 16 output voxels. Included by
// conv2_kernel.hpp.
//
// Bound by memory: 32 -> 32 from 2 x 128^3 reads 138 MB and writes 17, 31 us at the 5 TB/s a large copy reaches; its products are 7 us. The direct kernel (conv2_kernel.hpp) reads
// every tap's rows from memory, 27 loads of rows 64 bytes apart per voxel, and the vector cache's queue of pending lines is what it waits for (59 us, the input read 1.9 times
// from HBM); the general kernel stages 5 x 17 x 33 positions through registers for 2 x 8 x 16 outputs. Here a workgroup of four wavefronts takes 4 rows of 32 output voxels of a plane:
// 27 input rows of 65 voxels, copied to LDS asynchronously as they lie in memory (64 KB, so that two workgroups share a CU and one's copies run under the
// other's products). The fourteen weight pairs stay in registers over the workgroup's walk, so the K loop is LDS reads at constant offsets and products; the next
// tile's copies go out before the epilogue. A tap's 32 lanes read every second voxel of a row; the 16-byte pieces of a row lie permuted (swz) so that they meet all
// banks. The walk runs down the planes: the plane two tiles share is in the L2 the second time. 2 x 128^3 59.0 -> 43.6 us (3.6 TB/s), nine windows 278 -> 170 (4.1 TB/s) for the conv
// by itself; inside a forward, whose last kernel has just written the input, 47.5 and 185.
#pragma once

template <int FMT> struct s2row_t {
    static constexpr int TY = 4, TX = 32;                       // a workgroup's tile: 4 rows of 32 output voxels of one plane
    static constexpr int HY = 2 * TY + 1, HX = 2 * TX + 1, ROWS = 3 * HY;      // staged input rows of 65 voxels
    static constexpr int NH = fmt_t<FMT>::NH, GC = HX * NH, PC = (GC + 3) & ~3;      // 16-byte pieces of a row, and its pitch in pieces
    static constexpr int NG = (ROWS * PC + 63) / 64;            // copy groups of 64 pieces
    static constexpr int PS = HX + 1, NGS = (ROWS * PS + 63) / 64;      // scale words: pitch of a row, copy groups
    static constexpr int SC = NG * 1024, LDS = SC + NGS * 256;
    // piece g of a row lies at place g ^ swz(g): 32 lanes read every second voxel's piece, and without the exchange half of the LDS banks
    __host__ __device__ static constexpr int swz(int g) { return FMT == 8 ? (g >> 4) & 3 : (g >> 4) & 1; }
};
template <int FMT, int OUT>
__global__ void __launch_bounds__(256, 2) conv3s2_row_k(const conv_args a) {
    using T = s2row_t<FMT>;
    constexpr int NH = T::NH, RB = fmt_t<FMT>::RB, WTILE = fmt_t<FMT>::WTILE, NP = 14, HY = T::HY, PB = T::PC * 16, SB = T::PS * 4;
    extern __shared__ __align__(16) unsigned char lds[];
    const unsigned lds0 = (unsigned)(size_t)lds;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 31, h = lane >> 5;
    const size_t Sin = (size_t)a.D * a.H * a.W;
    // XCD-aware persistent walk, planes fastest: the workgroups of an XCD run down neighbouring columns, so a plane's second reader finds it in the L2
    const unsigned per = (a.ntiles + 7u) / 8u, wg_per_xcd = gridDim.x >> 3, xcd = blockIdx.x & 7u, wix = blockIdx.x >> 3;
    struct tile_t { int n, oz, oy, ox; bool ok; };
    auto decode = [&](unsigned it) {
        tile_t t; const unsigned k = wix + it * wg_per_xcd;
        t.ok = k < per && xcd * per + k < a.ntiles;
        unsigned tt = t.ok ? xcd * per + k : 0u;
        t.oz = (int)(tt % (unsigned)a.ntz); tt /= (unsigned)a.ntz;
        t.ox = (int)(tt % (unsigned)a.ntx) * T::TX; tt /= (unsigned)a.ntx;
        t.oy = (int)(tt % (unsigned)a.nty) * T::TY; t.n = (int)(tt / (unsigned)a.nty);
        return t;
    };
    tile_t cur = decode(0);
    if (!cur.ok) return;
    // what a lane copies: group g = wave + 4 k of the rows' pieces, and of the scale words: voxel and row packed, bit 31 for a place that holds nothing
    constexpr int NK = (T::NG + 3) / 4, NKS = (T::NGS + 3) / 4;
    unsigned pk[NK], pks[NKS];
#pragma unroll
    for (int k = 0; k < NK; k++) {
        const int L = (wave + 4 * k) * 64 + lane, row = L / T::PC, c = L - row * T::PC, g = c ^ T::swz(c);
        pk[k] = (unsigned)(g / NH) | (unsigned)(g % NH) << 8 | (unsigned)(row % HY) << 12 | (unsigned)(row / HY) << 20 | (row < T::ROWS && g < T::GC ? 0u : 1u << 31);
    }
#pragma unroll
    for (int k = 0; k < NKS; k++) {
        const int L = (wave + 4 * k) * 64 + lane, row = L / T::PS, px = L - row * T::PS;
        pks[k] = (unsigned)px | (unsigned)(row % HY) << 12 | (unsigned)(row / HY) << 20 | (row < T::ROWS && px < T::HX ? 0u : 1u << 31);
    }
    // the tile's rows and scale bytes into LDS; positions outside the volume read the constant page (zero rows, scale byte 1)
    auto request = [&](const tile_t &t) {
        const int z0 = 2 * t.oz - 1, y0 = 2 * t.oy - 1, x0 = 2 * t.ox - 1;
        const uint8_t *xq = a.xq[0] + (size_t)t.n * a.nbs[0] * Sin * RB, *xs = a.xsc[0] + (size_t)t.n * a.nbs[0] * Sin;
        auto vox = [&](unsigned &p, int &v) {
            asm volatile("" : "+v"(p));                         // (opaque: unpacked per request, not kept unpacked in registers)
            const int gz = z0 + (int)((p >> 20) & 3u), gy = y0 + (int)((p >> 12) & 15u), gx = x0 + (int)(p & 255u);
            v = (gz * a.H + gy) * a.W + gx;
            return (p >> 31) == 0u && (unsigned)gz < (unsigned)a.D && (unsigned)gy < (unsigned)a.H && (unsigned)gx < (unsigned)a.W;
        };
        static_for<NK>([&](auto K) {
            constexpr int k = decltype(K)::value;
            if (T::NG % 4 == 0 || wave + 4 * k < T::NG) {
                int v; unsigned q = pk[k]; const bool in = vox(q, v);
                dma16(in ? xq + (size_t)v * RB + ((q >> 8) & 15u) * 16u : a.zpage, lds0 + (unsigned)(wave + 4 * k) * 1024u);
            }
        });
        static_for<NKS>([&](auto K) {
            constexpr int k = decltype(K)::value;
            if (T::NGS % 4 == 0 || wave + 4 * k < T::NGS) {
                int v; unsigned q = pks[k]; const bool in = vox(q, v);
                dma1(in ? xs + v : a.zpage + 64, lds0 + T::SC + (unsigned)(wave + 4 * k) * 256u);
            }
        });
    };
    conv_epi_consts<1, false>(a, lds, 0, tid);
    request(cur);
    // the weights stay in registers: fourteen pairs in the order of the direct kernel (mi_s2_unit), four pairs' scale bytes in a word
    v8i wf[NP]; int ws[(NP + 3) / 4];
#pragma unroll
    for (int i = 0; i < (NP + 3) / 4; i++) ws[i] = 0;
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const v4i lo = *(const v4i *)(a.wq + (size_t)p * WTILE + lane * 16);
        const v4i hi = FMT == 8 ? *(const v4i *)(a.wq + (size_t)p * WTILE + 1024 + lane * 16) : (v4i){0, 0, 0, 0};
        wf[p] = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        ws[p >> 2] |= (*(const int *)(a.wsc + ((size_t)p * 64 + lane) * 4) & 255) << (8 * (p & 3));
    }
    // per kx the lane's piece of row (kz 0, ky 0) of its run: voxel 2 r + kx, half h (e4m3); e2m1: the lane half's own unit. Scale words: the half's unit
    auto place = [&](int g) { return (unsigned)((g ^ T::swz(g)) * 16 + 2 * wave * PB); };
    unsigned b0, b1 = 0, b2, b2s = 0;
    if constexpr (FMT == 8) { b0 = place(4 * r + h); b1 = place(4 * r + 2 + h); b2 = place(4 * r + 4 + h); }
    else { b0 = place(2 * r + h); b2 = place(2 * r + 2) + h * PB; b2s = b2 + h * (HY - 3) * PB; }      // (units in rows ky, ky + 1; in rows ky 2 and ky 0 of the next plane)
    const unsigned s0 = T::SC + (2 * r + h) * 4 + 2 * wave * SB, s2 = T::SC + (2 * r + 2) * 4 + 2 * wave * SB + h * SB, s2s = s2 + h * (HY - 3) * SB;
    for (unsigned it = 0;; it++) {
        const tile_t nxt = decode(it + 1);
        wait_vm<0>();
        __syncthreads();
        v16f acc[1][1];
#pragma unroll
        for (int i = 0; i < 16; i++) acc[0][0][i] = 0.f;
        static_for<NP>([&](auto P) {
            // pair p: rows (kz, ky) = R of the taps kx 0 and 1; or the taps kx 2 of rows R and R + 1 (one of them alone at the end)
            constexpr int p = decltype(P)::value, G = p < 12 ? p / 3 : 4, q = p - 3 * G, nrow = G < 4 ? 2 : 1;
            constexpr bool two = q < nrow;
            constexpr int R = two ? 2 * G + q : 2 * G, ro = R / 3 * HY + R % 3;
            constexpr bool last = !two && nrow == 1, cross = !two && R % 3 == 2;
            v4i lo, hi = {0, 0, 0, 0}; int sb;
            if constexpr (FMT == 8) {
                constexpr int ro1 = (R + 1) / 3 * HY + (R + 1) % 3;
                lo = *(const v4i *)(lds + (two ? b0 : b2) + ro * PB);
                if constexpr (two) hi = *(const v4i *)(lds + b1 + ro * PB); else if constexpr (!last) hi = *(const v4i *)(lds + b2 + ro1 * PB);
            } else {
                lo = *(const v4i *)(lds + (two ? b0 : last ? b2 - h * PB : cross ? b2s : b2) + ro * PB);
                if constexpr (last) lo = h ? (v4i){0, 0, 0, 0} : lo;
            }
            sb = *(const int *)(lds + (two ? s0 : last ? s2 - h * SB : cross ? s2s : s2) + ro * SB);
            if constexpr (last) sb = h ? 127 : sb;              // (the unit past the last: zero codes on both sides)
            const v8i B = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            acc[0][0] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wf[p], B, acc[0][0], FMT == 8 ? 0 : 4, FMT == 8 ? 0 : 4, p & 3, ws[p >> 2], 0, sb);
            if constexpr (p % 4 == 3 || p == NP - 1) row_pin(acc[0][0]);      // (the products stay here: left alone they sink to the epilogue, with all fourteen pairs' rows in registers)
        });
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // everyone has read the tile's rows
        if (nxt.ok) request(nxt);                               // they land while the epilogue, and the other workgroup of the CU, run
        conv_epilogue<1, 1, OUT, false, false, true, false, true, 4, true>(a, acc, lds, 0u, cur.n, 0, cur.oz, cur.oy, cur.ox, 0, wave, tid);
        if (!nxt.ok) break;
        cur = nxt;
    }
}
template <int FMT, int OUT>
static void launch_s2row(const conv_args &a, size_t smem) {
    static bool attr[8]; static int ncu[8];
    int d = 0; MIRT(hipGetDevice(&d)); d &= 7;
    if (!attr[d]) {
        MIRT(hipFuncSetAttribute((const void *)conv3s2_row_k<FMT, OUT>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        hipDeviceProp_t pr; MIRT(hipGetDeviceProperties(&pr, d));
        ncu[d] = pr.multiProcessorCount > 8 ? pr.multiProcessorCount & ~7 : 8;
        attr[d] = true;
    }
    const unsigned per = (a.ntiles + 7u) / 8u, nwg = per * 8u < 2u * (unsigned)ncu[d] ? per * 8u : 2u * (unsigned)ncu[d];
    conv3s2_row_k<FMT, OUT><<<nwg, 256, smem>>>(a);
    MICK();
    snprintf(g_last_kernel, sizeof g_last_kernel, "conv3s2_row_k<fmt %d, out %d> tiles %u wgs %u", FMT, OUT, a.ntiles, nwg);
}
