// 2x2x2 stride-2 conv into MX rows (17 and more output channels): the general kernel's products (conv2_mx_k) with what its wavefronts wait for requested earlier.
//
// The launch is one tile per wavefront deep: its length is a chain of latencies and of its wavefronts' instructions. The general kernel keeps two wavefronts per SIMD (two column tiles x four channel
// tiles, 224 registers), each with the next pair's weights in flight from the L2 and three pairs of rows, and forms its voxel with 64-bit divisions first.
// Here a wavefront owns ONE tile of 32 columns x MT channel tiles (64 accumulator registers with four: e2m1 takes 123 registers, four wavefronts per SIMD; e4m3 145, so that its workgroups of eight
// run one per CU, two wavefronts per SIMD), the weights of a stage (two K pairs, four with fewer than four channel tiles) come by LDS-DMA two stages ahead, shared by the workgroup's eight
// wavefronts, and the rows of the next AR - 1 pairs are in flight in registers. Counted waits: a wavefront issues the same memory operations in every stage, so that the copies of stage s + 1 have
// landed when at most the CW operations younger than them are outstanding. One barrier per stage.
// Three things keep the rows in flight: a unit is read from a lane table (a walk's scalar branches and multiplies were half of a pair's instructions, and a basic block each), the scale bytes stay
// bytes until they are used (widened at once, the compiler gathers the widening of all sets at the loop's head, behind a wait for every load), and the accumulators are pinned after a pair
// (products are free to sink below the barrier else, with their fragments kept, or spilled, until then).
// Measured, passes back to back, us, the general kernel / without those three / this: e2m1 128 -> 256 from 2 x 64^3 (44.6 MB) 21.6 / 20.1 / 16.7, 256 -> 256 from 2 x 48^3 25.8 / 20.1 / 16.8,
// 256 -> 32 from 32^3 13.1 / 15.8 / 7.8, 64 -> 160 from 2 x 64^3 14.0 / 19.3 / 12.2; e4m3 128 -> 256 from 2 x 64^3 33.8 / 32.1 / 31.2, from 1 x 32^3 14.6 / 12.6 / 10.2, 256 -> 64 from 32^3
// 17.1 / 17.5 / 13.7. Seven pairs in flight instead of three: slower (256 -> 32 from 16^3 15.6 against 14.5, before the table). Eight channel tiles per wavefront at two wavefronts per SIMD, the rows read
// once instead of once per slice of 128: no difference.
#pragma once
#include "conv2_up.hpp"

template <int FMT, int OUT, int MT>
__global__ void __launch_bounds__(512, FMT == 4 ? 4 : 2) conv2_down_k(const conv_args a) {
    constexpr int RB = fmt_t<FMT>::RB, WTILE = fmt_t<FMT>::WTILE, KT = WTILE / 1024, YB = OUT * 4;
    constexpr int SP = MT == 4 ? 2 : 4, nti = SP * MT, NPC = nti * KT + (nti + 3) / 4, PC = (NPC + 7) / 8;      // pairs of a stage; its weight tiles; 1 KiB pieces (scale words: four tiles each); pieces per wavefront
    constexpr unsigned SLOT = (unsigned)NPC * 1024u;
    constexpr int AR = 4;                        // pairs of rows in flight
    constexpr int RL = FMT == 4 ? 2 : 3;                        // memory operations of a pair's rows
    extern __shared__ __align__(16) unsigned char lds[];
    const unsigned lds0 = (unsigned)(size_t)lds;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 31, h = lane >> 5;
    const int n = blockIdx.z, cs = blockIdx.y, nb = a.nbs[0], np = 4 * nb, ns = np / SP;      // (np is a multiple of AR)
    const size_t Sin = (size_t)a.D * a.H * a.W, So = (size_t)a.Do * a.Ho * a.Wo;
    const unsigned ring0 = MT * 128u;
    // (stages past the last: the last one's pieces again; pieces past a stage's last: that one again)
    auto copy = [&](int s, unsigned so) {
        const int sc_ = min(s, ns - 1);
#pragma unroll
        for (int k = 0; k < PC; k++) {
            const int i = min(wave + 8 * k, NPC - 1);
            const bool sc = i >= nti * KT;
            const int ti = sc ? min((i - nti * KT) * 4 + (lane >> 4), nti - 1) : i / KT;          // (scale words past the last tile: copied, not read)
            const size_t t = (size_t)(sc_ * SP + ti / MT) * a.nmt_all + cs * MT + ti % MT;
            const uint8_t *src = sc ? a.wsc + t * 256 + (lane & 15) * 16 : a.wq + t * WTILE + (i % KT) * 1024 + lane * 16;
            dma16(src, lds0 + so + (unsigned)i * 1024u);
        }
    };
    copy(0, ring0);
    copy(1, ring0 + SLOT);
    if (tid < MT * 32) { const int co = cs * MT * 32 + tid; ((float *)lds)[tid] = a.bias && co < a.Co ? a.bias[co] : 0.f; }
    // the lane's output voxel and the input voxel of its tap (0, 0, 0) (32-bit: the dispatch keeps tensors of 2^27 voxels and more away)
    const unsigned c0 = (blockIdx.x * 8u + (unsigned)wave) * 32u, Wo = (unsigned)a.Wo, Ho = (unsigned)a.Ho;
    const bool cok = c0 + (unsigned)r < (unsigned)So;
    const unsigned cv = cok ? c0 + (unsigned)r : 0u, yz = cv / Wo, x = cv - yz * Wo, z = yz / Ho, y = yz - z * Ho;
    const unsigned iv0 = (2u * z * (unsigned)a.H + 2u * y) * (unsigned)a.W + 2u * x;
    const uint8_t *xq = a.xq[0] + (size_t)n * nb * Sin * RB, *xsc = a.xsc[0] + (size_t)n * nb * Sin;
    struct bfrag { v4i lo, hi; uint8_t sb; };
    bfrag fb[AR];
    // the rows of the next K pair, units 2 p and 2 p + 1 of the (tap, block) order (pairs past the last: the last unit's rows again). Lane l holds the voxel offset of unit ubase + l, formed once
    // for 64 units by all lanes together
    const int nu = 8 * nb;
    unsigned long long uoff = 0;
    auto fill = [&](int ubase) {
        const unsigned u = (unsigned)min(ubase + lane, nu - 1), t = u / (unsigned)nb, b = u - t * (unsigned)nb;
        uoff = (unsigned long long)b * Sin + ((size_t)(t >> 2) * a.H + ((t >> 1) & 1)) * a.W + (t & 1);
    };
    fill(0);
    int ui = 0, ub = 0;                                         // (uniform) the next unit's lane; the table's first unit
    auto unit = [&](int i) { return (size_t)((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(unsigned)uoff, i) | (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(unsigned)(uoff >> 32), i) << 32); };
    auto rows = [&](auto SET) {
        constexpr int set = decltype(SET)::value;
        const size_t o0 = unit(ui), o1 = unit(ui + 1);
        ui += 2;
        if constexpr (FMT == 8) {
            fb[set].lo = *(const v4i *)(xq + o0 * RB + (size_t)iv0 * RB + 16 * h);
            fb[set].hi = *(const v4i *)(xq + o1 * RB + (size_t)iv0 * RB + 16 * h);
        } else { fb[set].lo = *(const v4i *)(xq + ((h ? o1 : o0) + iv0) * RB); fb[set].hi = (v4i){0, 0, 0, 0}; }
        fb[set].sb = xsc[(h ? o1 : o0) + iv0];
    };
    static_for<AR - 1>([&](auto I) { rows(I); });
    v16f acc[MT];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[m][i] = 0.f;
    wait_vm<PC + (AR - 1) * RL>();                              // stage 0's pieces
    __syncthreads();
    // Operations younger than the copies of stage s + 1 at the end of stage s: the rows requested in stages s - 1 and s and the copies of stage s + 2 between them
    constexpr int CW = (SP + (SP < AR - 1 ? SP : AR - 1)) * RL + PC;
    unsigned slot = ring0;
    for (int p0 = 0; p0 < np; p0 += AR) {
        if (ui + 2 * AR > 64) { ub += ui; fill(ub); ui = 0; }      // (uniform)
        static_for<AR / SP>([&](auto Q) {
            constexpr int q = decltype(Q)::value;
            const int s = p0 / SP + q;
            copy(s + 2, slot + 2 * SLOT >= ring0 + 3 * SLOT ? slot - SLOT : slot + 2 * SLOT);      // (the slot that stage s - 1 has left)
            static_for<SP>([&](auto I) {
                constexpr int i = q * SP + decltype(I)::value;
                rows(std::integral_constant<int, (i + AR - 1) % AR>{});
                const v8i B = {fb[i].lo[0], fb[i].lo[1], fb[i].lo[2], fb[i].lo[3], fb[i].hi[0], fb[i].hi[1], fb[i].hi[2], fb[i].hi[3]};
#pragma unroll
                for (int m = 0; m < MT; m++) {
                    const unsigned ti = (unsigned)(decltype(I)::value * MT + m), o = slot + lane * 16 + ti * WTILE;
                    const v4i lo = *(const v4i *)(lds + o);
                    v8i A;
                    if constexpr (FMT == 8) { const v4i hi = *(const v4i *)(lds + o + 1024); A = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}; }
                    else A = (v8i){lo[0], lo[1], lo[2], lo[3], 0, 0, 0, 0};
                    const int sw = *(const int *)(lds + slot + lane * 4 + nti * WTILE + ti * 256);
                    acc[m] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A, B, acc[m], FMT == 8 ? 0 : 4, FMT == 8 ? 0 : 4, 0, sw, 0, (int)fb[i].sb);
                }
#pragma unroll
                for (int m = 0; m < MT; m++) asm volatile("" : "+v"(acc[m]) : : "memory");
                __builtin_amdgcn_sched_barrier(0);              // (one pair's weight fragments at a time in registers)
            });
            wait_vm<CW>();
            __syncthreads();
            slot = slot + SLOT >= ring0 + 3 * SLOT ? ring0 : slot + SLOT;
        });
    }
    const int nbo = (a.Co + 31) >> 5;
    uint8_t *yq = (uint8_t *)a.y, *ysc = yq + (size_t)a.N * nbo * So * YB;
    static_for<MT>([&](auto M) {
        constexpr int m = decltype(M)::value;
        float bias[16];
#pragma unroll
        for (int i = 0; i < 4; i++) { const float4 b = *(const float4 *)(lds + (m * 32 + 16 * h + 4 * i) * 4); bias[4 * i] = b.x; bias[4 * i + 1] = b.y; bias[4 * i + 2] = b.z; bias[4 * i + 3] = b.w; }
        unsigned d[OUT / 2];
        const unsigned e = c2_codes<OUT>(acc[m], bias, d);
        const size_t row = ((size_t)n * nbo + cs * MT + m) * So + cv;
        if (cok) {
            if constexpr (OUT == 8) *(uint4 *)(yq + row * 32 + 16 * h) = make_uint4(d[0], d[1], d[2], d[3]);
            else *(uint2 *)(yq + row * 16 + 8 * h) = make_uint2(d[0], d[1]);
            if (!h) ysc[row] = (uint8_t)e;
        }
    });
    wait_vm<0>();                                               // (the copies of stages past the last)
}
template <int FMT> constexpr size_t conv2_down_lds(int MT) { const int nti = (MT == 4 ? 2 : 4) * MT; return (size_t)MT * 128 + 3 * (size_t)(nti * (FMT == 8 ? 2 : 1) + (nti + 3) / 4) * 1024; }
template <int FMT, int OUT>
static void launch_conv2_down_t(const conv_args &a, int MT) {
    const dim3 grid((unsigned)(((size_t)a.Do * a.Ho * a.Wo + 255) / 256), (unsigned)(a.nmt_all / MT), (unsigned)a.N);
    const size_t smem = conv2_down_lds<FMT>(MT);
    if (MT == 4) conv2_down_k<FMT, OUT, 4><<<grid, 512, smem>>>(a);
    else if (MT == 2) conv2_down_k<FMT, OUT, 2><<<grid, 512, smem>>>(a);
    else conv2_down_k<FMT, OUT, 1><<<grid, 512, smem>>>(a);
    MICK();
    snprintf(g_last_kernel, sizeof g_last_kernel, "conv2_down_k<fmt %d, out %d, MT %d> (conv2_mx_k's products) blocks %d grid %u x %u x %u", FMT, OUT, MT, a.nbs[0], grid.x, grid.y, grid.z);
}
