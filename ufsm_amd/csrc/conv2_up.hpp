// 2x2x2 transposed conv into MX rows (17 and more output channels, up to CU2_NP K pairs = 256 input channels): the eight taps of 32 input voxels by one
// wavefront, from rows it reads once.
//
// What bounds it is the epilogue: an accumulator tile is as little as two products (64 input channels) and always about 100 vector instructions of bias, block
// scale, codes and stores. The general kernel (conv2_mx_k) takes a tap per workgroup with eight accumulator tiles per wavefront: 240 registers, two wavefronts per
// SIMD, each of which spends a third of its life in front of its first product (64-bit divisions for the lane's voxel, then the rows, then the weights) and
// writes every second 16-byte row of its output lines. Here
//   * a wavefront owns 32 consecutive input voxels whose fragments of all K pairs stay in registers; a workgroup of eight walks CHUNKS: chunk (dz, dy, m) is the
//     two dx taps into channel tile m, two accumulator tiles, 32 registers. Four wavefronts per SIMD fit (e4m3 with four K pairs by five spilled registers into
//     e4m3 rows and three into e2m1 ones, stored once and read back once a chunk), and one's epilogue runs beside another's products;
//   * a chunk's weights (2 taps x K pairs) come by LDS-DMA into the second of two slots while the chunk before is multiplied: the workgroup's 256 voxels share
//     them. One barrier per chunk, in front of its stores, so that waiting for the copies waits for stores a chunk old;
//   * the two voxels of a chunk are neighbours in memory: e2m1 rows change halves between the lanes of a voxel (one lane gets a whole row of each), so that a
//     wavefront's store covers 1 KiB without holes, and the two scale bytes leave as one 16-bit store.
// The launch splits the chunks over blockIdx.y until two workgroups per CU are there (the rows are then read once per split, from the L2).
// The products and their order are those of conv2_mx_k: the same bytes. Measured, passes back to back, us, conv2_mx_k / this: e2m1 256 -> 128 from 2 x 32^3 (44.6 MB, 8.6 GFLOP) 27.8 / 20.9
// (2.1 TB/s); e4m3 the same 104.3 / 32.2, 224 -> 128 there 103.2 / 31.7, 128 -> 128 from 2 x 38 x 50 x 20 90.9 / 28.9. With the down conv in front of it (conv2_down.hpp), e2m1 128 -> 256 -> 128 at
// 2 x 64^3: 48.8 -> 35.5.
// What is left is the start (rows and the first weights, about 3 us, which every workgroup of the single round waits for) and the epilogues.
#pragma once
#include "conv3_kernel.hpp"

constexpr int CU2_NP = 4, CU2_MT = 32;                          // K pairs of 64 input channels held in registers; channel tiles (their biases lie in LDS)

// a tile of 32 voxels x 32 channels: bias, block scale, codes (4 words of e4m3 or 2 of e2m1: the lane's 16 channels); returns the scale byte
template <int OUT>
__device__ __forceinline__ unsigned c2_codes(const v16f &acc, const float *bias, unsigned (&d)[OUT / 2]) {
    float v[16], am = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) { v[i] = acc[i] + bias[i]; am = fmaxf(am, fabsf(v[i])); }
    am = lane_pair_max(am);
    const int e = d_mx_exp(am, OUT == 8 ? MI_INVQ8 : MI_INVQ4);
    const float p2e = d_exp2i(e);
    if constexpr (OUT == 8) {
#pragma unroll
        for (int q = 0; q < 4; q++) d[q] = d_enc_e4m3x4_hw(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3], p2e);
    } else { d[0] = d_enc_e2m1x8_hw(v, p2e); d[1] = d_enc_e2m1x8_hw(v + 8, p2e); }
    if (d_any_nf(e)) {
        const unsigned z = d_opaque_zero();
        if (e == 128) {
            if constexpr (OUT == 8) {
#pragma unroll
                for (int q = 0; q < 4; q++) d[q] = d_enc4_e4m3_nf(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3], z);
            } else { d[0] = d_enc8_e2m1_nf(v, z); d[1] = d_enc8_e2m1_nf(v + 8, z); }
        }
    }
    return (unsigned)(e + 127);
}

template <int FMT, int OUT, int NP>
__global__ void __launch_bounds__(512, 4) conv2_up_k(const conv_args a, int cpw) {
    constexpr int RB = fmt_t<FMT>::RB, WTILE = fmt_t<FMT>::WTILE, KT = WTILE / 1024, YB = OUT * 4;
    constexpr int nti = 2 * NP, npc = nti * KT + (nti + 3) / 4; // a slot: 2 NP weight tiles (tap dx, pair p), then their scale words (whole KiB: four tiles' worth each); 1 KiB pieces of it
    constexpr unsigned sslot = (unsigned)npc * 1024u;
    extern __shared__ __align__(16) unsigned char lds[];
    const unsigned lds0 = (unsigned)(size_t)lds;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 31, h = lane >> 5;
    const int n = blockIdx.z, nb = a.nbs[0], nmt = a.nmt_all;
    const int q0 = (int)blockIdx.y * cpw, q1 = min(q0 + cpw, 4 * nmt);
    const size_t Sin = (size_t)a.D * a.H * a.W, So = 8 * Sin;
    const unsigned slot0 = (unsigned)nmt * 128u;
    auto copy = [&](int dzy, int m, unsigned so) {              // the wavefronts take the pieces in turn
        for (int i = wave; i < npc; i += 8) {
            const bool sc = i >= nti * KT;
            const int k = sc ? min((i - nti * KT) * 4 + (lane >> 4), nti - 1) : i / KT;      // (scale words past the last tile: copied, not read)
            const size_t t = ((size_t)(2 * dzy) * NP + k) * nmt + m;                       // (tap 2 dzy + dx, pair p) = row 2 dzy NP + k of the prepared weights
            const uint8_t *src = sc ? a.wsc + t * 256 + (lane & 15) * 16 : a.wq + t * WTILE + (i % KT) * 1024 + lane * 16;
            dma16(src, lds0 + so + (unsigned)i * 1024u);
        }
    };
    struct chunk_t { int dzy, m; };
    auto next = [&](chunk_t c) { c.m++; if (c.m == nmt) { c.m = 0; c.dzy++; } return c; };
    chunk_t ch = {q0 / nmt, q0 % nmt}, c2 = next(ch);           // this chunk; the one whose weights are requested next
    copy(ch.dzy, ch.m, slot0);
    if (q0 + 1 < q1) copy(c2.dzy, c2.m, slot0 + sslot);
    for (int i = tid; i < nmt * 32; i += 512) ((float *)lds)[i] = a.bias && i < a.Co ? a.bias[i] : 0.f;
    // the lane's input voxel (32-bit: the dispatch keeps tensors of 2^27 voxels and more away)
    const unsigned c0 = (blockIdx.x * 8u + (unsigned)wave) * 32u, S32 = (unsigned)Sin, W = (unsigned)a.W, H = (unsigned)a.H;
    const bool cok = c0 + (unsigned)r < S32;
    const unsigned iv = cok ? c0 + (unsigned)r : 0u;
    const unsigned yz = iv / W, x = iv - yz * W, z = yz / H, y = yz - z * H;
    const uint8_t *xq = a.xq[0] + (size_t)n * nb * Sin * RB, *xsc = a.xsc[0] + (size_t)n * nb * Sin;
    v8i fb[NP]; int sb[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const bool ok1 = p < NP - 1 || 2 * p + 1 < nb;          // (no second block: zero codes beside scale 1)
        const size_t v0 = (size_t)(2 * p) * Sin + iv, v1 = (size_t)(ok1 ? 2 * p + 1 : 2 * p) * Sin + iv;
        if constexpr (FMT == 8) {
            const v4i lo = *(const v4i *)(xq + v0 * RB + 16 * h), hi = *(const v4i *)(xq + v1 * RB + 16 * h);
            fb[p] = (v8i){lo[0], lo[1], lo[2], lo[3], ok1 ? hi[0] : 0, ok1 ? hi[1] : 0, ok1 ? hi[2] : 0, ok1 ? hi[3] : 0};
        } else {
            const v4i lo = *(const v4i *)(xq + (h ? v1 : v0) * RB);
            const bool k = !h || ok1;
            fb[p] = (v8i){k ? lo[0] : 0, k ? lo[1] : 0, k ? lo[2] : 0, k ? lo[3] : 0, 0, 0, 0, 0};
        }
        sb[p] = h ? (ok1 ? (int)xsc[v1] : 127) : (int)xsc[v0];
    }
    wait_vm<0>();
    __syncthreads();
    const int nbo = (a.Co + 31) >> 5;
    uint8_t *yq = (uint8_t *)a.y, *ysc = yq + (size_t)a.N * nbo * So * YB;
    const size_t ov = ((size_t)(2 * z) * (2 * H) + 2 * y) * (2 * W) + 2 * x;
    for (int q = q0; q < q1; q++) {
        const unsigned so = slot0 + ((q - q0) & 1 ? sslot : 0u);
        v16f acc[2];
        static_for<NP>([&](auto P) {
            constexpr int p = decltype(P)::value;
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const unsigned o = so + lane * 16;
                constexpr unsigned tb = p * WTILE;
                const v4i lo = *(const v4i *)(lds + o + t * NP * WTILE + tb);
                v8i A;
                if constexpr (FMT == 8) { const v4i hi = *(const v4i *)(lds + o + t * NP * WTILE + tb + 1024); A = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}; }
                else A = (v8i){lo[0], lo[1], lo[2], lo[3], 0, 0, 0, 0};
                const int s = *(const int *)(lds + so + lane * 4 + nti * WTILE + (t * NP + p) * 256);
                acc[t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A, fb[p], p == 0 ? (v16f){} : acc[t], FMT == 8 ? 0 : 4, FMT == 8 ? 0 : 4, 0, s, 0, sb[p]);      // (the first pair adds to a literal zero)
            }
        });
        float bias[16];
#pragma unroll
        for (int i = 0; i < 4; i++) { const float4 b = *(const float4 *)(lds + (ch.m * 32 + 16 * h + 4 * i) * 4); bias[4 * i] = b.x; bias[4 * i + 1] = b.y; bias[4 * i + 2] = b.z; bias[4 * i + 3] = b.w; }
        unsigned d0[OUT / 2], d1[OUT / 2];
        const unsigned e0 = c2_codes<OUT>(acc[0], bias, d0), e1 = c2_codes<OUT>(acc[1], bias, d1);
        wait_vm<0>();                                           // this wavefront's pieces of the next chunk (and the stores of the last one)
        __syncthreads();                                        // every piece has landed, and everyone is done with this chunk's slot
        const chunk_t c = ch; ch = c2; c2 = next(c2);
        if (q + 2 < q1) copy(c2.dzy, c2.m, so);
        const size_t row = ((size_t)n * nbo + c.m) * So + ov + ((size_t)(c.dzy >> 1) * (2 * H) + (c.dzy & 1)) * (2 * W);
        if constexpr (OUT == 8) {
            if (cok) {
                *(uint4 *)(yq + row * 32 + 16 * h) = make_uint4(d0[0], d0[1], d0[2], d0[3]);
                *(uint4 *)(yq + row * 32 + 32 + 16 * h) = make_uint4(d1[0], d1[1], d1[2], d1[3]);
            }
        } else {
            // lane (r, 0) has bytes 0 .. 7 of both voxels' rows, lane (r, 1) bytes 8 .. 15: after the exchange lane (r, t) has the whole row of voxel t
            const auto s0 = __builtin_amdgcn_permlane32_swap(d0[0], d1[0], false, false), s1 = __builtin_amdgcn_permlane32_swap(d0[1], d1[1], false, false);
            if (cok) *(uint4 *)(yq + (row + h) * 16) = make_uint4(s0[0], s1[0], s0[1], s1[1]);
        }
        if (cok && !h) *(unsigned short *)(ysc + row) = (unsigned short)(e0 | e1 << 8);
    }
}
// chunks per workgroup: the fewest splits that give two workgroups per CU (512); LDS bytes
static inline int conv2_up_cpw(const conv_args &a, unsigned gx) {
    const int C = 4 * a.nmt_all;
    const long long wg = (long long)gx * a.N;
    long long sp = (512 + wg - 1) / wg;
    if (sp > C) sp = C;
    return (int)((C + sp - 1) / sp);
}
static inline size_t conv2_up_lds(const conv_args &a, int fmt) {
    const int nti = 2 * ((a.nbs[0] + 1) / 2);
    return (size_t)a.nmt_all * 128 + 2 * (size_t)(nti * (fmt == 8 ? 2 : 1) + (nti + 3) / 4) * 1024;
}
template <int FMT, int OUT>
static void launch_conv2_up_t(const conv_args &a, size_t smem) {
    const unsigned gx = (unsigned)(((size_t)a.D * a.H * a.W + 255) / 256);
    const int cpw = conv2_up_cpw(a, gx), np = (a.nbs[0] + 1) / 2;
    const dim3 grid(gx, (unsigned)((4 * a.nmt_all + cpw - 1) / cpw), (unsigned)a.N);
    if (np == 4) conv2_up_k<FMT, OUT, 4><<<grid, 512, smem>>>(a, cpw);
    else if (np == 3) conv2_up_k<FMT, OUT, 3><<<grid, 512, smem>>>(a, cpw);
    else if (np == 2) conv2_up_k<FMT, OUT, 2><<<grid, 512, smem>>>(a, cpw);
    else conv2_up_k<FMT, OUT, 1><<<grid, 512, smem>>>(a, cpw);
    MICK();
    snprintf(g_last_kernel, sizeof g_last_kernel, "conv2_up_k<fmt %d, out %d, pairs %d> (conv2_mx_k's products) chunks %d grid %u x %u x %u", FMT, OUT, np, cpw, grid.x, grid.y, grid.z);
}
