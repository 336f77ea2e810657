// MX-fp8 attention forward core: softmax(Q K^T / sqrt(48)) V per sequence and head on block-scaled e4m3 MFMA (32x32x64).
// Interface and arithmetic: src/lp_attn8.cu:1-13 (definition), :29-76 (conversions), :124-180 (forward), :319-328 (entry) of the reference.
//
// The products are formed transposed, S^T = K Q^T and O^T = V^T P^T, so a query is a column of every accumulator: a lane (r, h) holds,
// for query r of its wavefront, 16 of the 32 keys of each key block and its partner lane (r, h ^ 1) the other 16. All row statistics
// of the softmax (maximum, sum, the rescale factor, the MX scale of P) are then per lane plus one exchange with the partner.
// An 8-bit operand fragment of the 32x32x64 MFMA holds, in lane (r, h), bytes 16 h ... 16 h + 15 of both 32-K blocks of row r (and
// that lane's scale operand is block h's): exactly the 16 + 16 keys whose P the lane has in its accumulators, so P goes from
// accumulators to the B fragment of the second product in registers with no data exchange at all. The transposed V stores the tokens
// of a block in the matching order.
#include <hip/hip_fp16.h>
#include <type_traits>
#include "mx_dev.hpp"
#include "attn_rope.hpp"
#include "../../include/mi_attn.h"

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
#define HD AT_HD
#define FT 64            // keys per tile; sequences are padded to a multiple of it in the quantised tensors (rows past S are zero)

// Slot k of a 32-token block of the transposed V holds token a8_slot_token(k) of the block: slots 16 h + 4 q + c are lane half h's
// accumulator elements 4 q + c, which are the block's keys 8 q + 4 h + c.
__host__ __device__ __forceinline__ int a8_slot_token(int k) { return 8 * ((k >> 2) & 3) + 4 * (k >> 4) + (k & 3); }

// ---- operand quantisation (src/lp_attn8.cu:29-76): the fp16 head-major pack [3][H][Tp][48] -> e4m3 blocks of 32 with one E8M0 scale each ----
// q and k rows: dst [H][R][64] e4m3 + scales [H][R][2], R = nseq Sp rows (token i of sequence s in row s Sp + i, rows past S zero). A row's 64
// output bytes are four 16-byte quarters: dims 0-15 and 16-31 (block 0), 32-47 and sixteen zeros (block 1). Four neighbouring lanes own a row,
// each one quarter: 32 bytes of halves in (two 16-byte loads), 16 bytes of codes out, the block's amax through one exchange with the
// partner quarter. blockIdx.y: 0 the queries, 1 the keys.
__global__ void __launch_bounds__(256) a8_rows_k(const __half *__restrict__ src_q, uint8_t *__restrict__ dst_q, uint8_t *__restrict__ sc_q, int H, int nseq, int S, int Sp, long long Tp, size_t part_src, size_t part_dst, size_t part_sc) {
    const long long R = (long long)nseq * Sp, i = blockIdx.x * 256ll + threadIdx.x, hr = i >> 2;
    if (hr >= (long long)H * R) return;
    const int qt = (int)(i & 3), h = (int)(hr / R); const long long row = hr - (long long)h * R;
    const int seq = (int)(row / Sp), ii = (int)(row - (long long)seq * Sp);
    const __half *src = src_q + blockIdx.y * part_src; uint8_t *dst = dst_q + blockIdx.y * part_dst, *sc = sc_q + blockIdx.y * part_sc;
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; k++) v[k] = 0.f;
    if (ii < S && qt < 3) {
        const uint4 *p = (const uint4 *)(src + ((size_t)h * Tp + (size_t)seq * S + ii) * HD + 16 * qt);
        const uint4 a = p[0], b = p[1];
        const unsigned w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int k = 0; k < 8; k++) { const __half2 hh = *(const __half2 *)&w[k]; v[2 * k] = __low2float(hh); v[2 * k + 1] = __high2float(hh); }
    }
    float am = 0.f;
#pragma unroll
    for (int k = 0; k < 16; k++) am = fmaxf(am, fabsf(v[k]));
    am = __uint_as_float(max(__float_as_uint(am), d_quad_xor_u<1>(__float_as_uint(am))));       // quarters (0, 1) and (2, 3) are the two blocks (am >= 0, never NaN: it orders as its bits; the four lanes of a row leave together)
    const int e = d_mx_exp(am, MI_INVQ8);
    *(uint4 *)(dst + (size_t)hr * 64 + 16 * qt) = make_uint4(d_enc4_e4m3(v[0], v[1], v[2], v[3], e), d_enc4_e4m3(v[4], v[5], v[6], v[7], e), d_enc4_e4m3(v[8], v[9], v[10], v[11], e), d_enc4_e4m3(v[12], v[13], v[14], v[15], e));
    if (!(qt & 1)) sc[(size_t)hr * 2 + (qt >> 1)] = (uint8_t)(e + 127);
}
// transposed v: dst [H][R / 64][48][64], the 64 tokens of a key tile in slot order (two blocks of 32) per dim, + scales [H][R / 64][48][2]: what the
// core reads of a key tile is 3 KB in a row. One wavefront per (head, 32-token block), lane d < 48 owns dim d: it gathers the block's 32 values of its
// dim (each gather reads one token's 96 contiguous bytes across the lanes), quantises them as one block and writes 32 contiguous bytes.
__global__ void __launch_bounds__(256) a8_vt_k(const __half *__restrict__ src, uint8_t *__restrict__ dst, uint8_t *__restrict__ sc, int H, int nseq, int S, int Sp, long long Tp) {
    const long long R = (long long)nseq * Sp, nb = R / 32, wb = blockIdx.x * 4ll + (threadIdx.x >> 6);
    const int d = threadIdx.x & 63;
    if (wb >= (long long)H * nb || d >= HD) return;
    const int h = (int)(wb / nb); const long long b = wb - (long long)h * nb, r0 = b * 32;
    const int seq = (int)(r0 / Sp), i0 = (int)(r0 - (long long)seq * Sp);       // (Sp is a multiple of 64: a block never straddles two sequences)
    const __half *base = src + ((size_t)h * Tp + (size_t)seq * S) * HD + d;
    float v[32];
#pragma unroll
    for (int k = 0; k < 32; k++) { const int ii = i0 + a8_slot_token(k); v[k] = ii < S ? __half2float(base[(size_t)ii * HD]) : 0.f; }
    unsigned codes[8];
    const unsigned sb = d_quant_row<8, false>(v, 32, codes);
    const size_t td = ((size_t)h * (R / 64) + (b >> 1)) * HD + d;               // (head, key tile, dim)
    uint4 *o = (uint4 *)(dst + td * 64 + (b & 1) * 32);
    o[0] = make_uint4(codes[0], codes[1], codes[2], codes[3]); o[1] = make_uint4(codes[4], codes[5], codes[6], codes[7]);
    sc[td * 2 + (b & 1)] = (uint8_t)sb;
}

// The block forward's way to the same operands: qkv_pack_k's arithmetic (attn_block.hip: QK-norm, gains, rotary embedding, rounding to binary16), a8_rows_k's and
// a8_vt_k's quantisation in one pass over the projection's rows, without the binary16 tensor between them (three launches of 20 + 5 + 12 us for
// two 16^3 windows in 4 heads, 11 us as this one: a workgroup forms the rotary angles once for 64 rows). Bound by its vector instructions and the chain of one row, not by
// the 192 bytes in and 62 out of a row and part. A workgroup takes one part (queries, keys, values) of the 64 tokens of a key tile of one head, thread (row, quarter)
// 16 dims: the row's sum of squares meets over the quarters in the order of qkv_pack_k's eight lanes; the V tile turns in LDS.
template <int MODE>
__global__ void __launch_bounds__(256) a8_pack_k(const float *__restrict__ qkv, const float *__restrict__ qg, const float *__restrict__ kg, uint8_t *__restrict__ q8, uint8_t *__restrict__ q8s,
                                                 size_t part, size_t part_sc, uint8_t *__restrict__ vt, uint8_t *__restrict__ vts, float *__restrict__ rq, float *__restrict__ rk, float *__restrict__ amx,
                                                 int H, int S, unsigned tiles, long long R, rope_t rp) {
    __shared__ float2 rtab[ROPE_TAB * 8];
    __shared__ float vl[64][HD + 1];
    __shared__ unsigned bmax;
    // eight tiles at a time, their 3 H workgroups each on one XCD (workgroups go to the XCDs in turn): the parts' 192-byte pieces of a token's row share cache lines
    const unsigned u = blockIdx.x >> 3, g = u / (3u * H), hp = u - g * (3u * H), tile = g * 8 + (blockIdx.x & 7);
    if (tile >= (unsigned)(R >> 6)) return;
    const int p = (int)(hp / (unsigned)H), h = (int)hp - p * H, C = H * HD, row = threadIdx.x >> 2, qt = threadIdx.x & 3;
    const unsigned seq = tile / tiles;                                           // (whole tiles of 64 tokens per sequence)
    const int ii = (int)(tile - seq * tiles) * 64 + row;
    const long long t = (long long)seq * S + ii;
    const bool live = ii < S && qt < 3;
    float v[16];
    {
        const float4 *x = (const float4 *)(qkv + t * 3 * C + p * C + h * HD + 16 * qt);
#pragma unroll
        for (int k = 0; k < 4; k++) { const float4 a = live ? x[k] : make_float4(0.f, 0.f, 0.f, 0.f); v[4 * k] = a.x; v[4 * k + 1] = a.y; v[4 * k + 2] = a.z; v[4 * k + 3] = a.w; }
    }
    if (p < 2) {
        const float *gs = (p ? kg : qg) + h * HD + 16 * qt;                      // (the gains sit at an arbitrary offset of the flat parameter vector: dword loads)
        float gn[16];
#pragma unroll
        for (int k = 0; k < 16; k++) gn[k] = qt < 3 ? gs[k] : 0.f;
        const int ts = ii - rp.nreg;
        const bool turn = rp.on && live && ts >= 0;
        const float pos = turn ? rope_pos<MODE>(rp, t, ts, qt) : 0.f;
        if (MODE == ROPE_TABLE && rp.on) { rope_fill(rtab, rope_positions(rp), rp.lbase); __syncthreads(); }
        float s0 = 0.f, s1 = 0.f;
#pragma unroll
        for (int k = 0; k < 8; k++) { s0 = fmaf(v[k], v[k], s0); s1 = fmaf(v[8 + k], v[8 + k], s1); }
        float ss = s0 + s1;
        ss += d_quad_xor_f<1>(ss); ss += d_quad_xor_f<2>(ss);
        const float r = 1.f / sqrtf(ss / HD + 1e-6f);
        if (!qt && live) (p ? rk : rq)[t * H + h] = r;
#pragma unroll
        for (int k = 0; k < 16; k++) v[k] *= r * gn[k];
        if (turn) {
#pragma unroll
            for (int f = 0; f < 8; f++) rope_turn<MODE>(rp, rtab, pos, f, v[2 * f], v[2 * f + 1]);
        }
        float am = 0.f;
#pragma unroll
        for (int k = 0; k < 16; k++) { v[k] = __half2float(__float2half_rn(v[k])); am = fmaxf(am, fabsf(v[k])); }
        am = __uint_as_float(max(__float_as_uint(am), d_quad_xor_u<1>(__float_as_uint(am))));      // (quarters (0, 1) and (2, 3) are the two blocks)
        const int e = d_mx_exp(am, MI_INVQ8);
        const size_t hr = (size_t)h * R + tile * 64ll + row;
        *(uint4 *)(q8 + p * part + hr * 64 + 16 * qt) = make_uint4(d_enc4_e4m3(v[0], v[1], v[2], v[3], e), d_enc4_e4m3(v[4], v[5], v[6], v[7], e), d_enc4_e4m3(v[8], v[9], v[10], v[11], e), d_enc4_e4m3(v[12], v[13], v[14], v[15], e));
        if (!(qt & 1)) q8s[p * part_sc + hr * 2 + (qt >> 1)] = (uint8_t)(e + 127);
        return;
    }
    if (threadIdx.x == 0) bmax = 0u;
    __syncthreads();
    float m = 0.f;
#pragma unroll
    for (int k = 0; k < 16; k++) { m = fmaxf(m, fabsf(v[k])); if (qt < 3) vl[row][16 * qt + k] = __half2float(__float2half_rn(v[k])); }
    m = fmaxf(m, d_quad_xor_f<1>(m)); m = fmaxf(m, d_quad_xor_f<2>(m));
    if (!qt) atomicMax(&bmax, __float_as_uint(m));                               // (non-negative floats order as their bit patterns)
    __syncthreads();
    // (the running maximum only grows: a workgroup that does not exceed the value it reads has nothing to add)
    if (threadIdx.x == 0 && bmax > *(volatile unsigned *)((unsigned *)amx + 1)) atomicMax((unsigned *)amx + 1, bmax);
    if (threadIdx.x >= HD * 4) return;
    const int d = threadIdx.x >> 2, b = (threadIdx.x >> 1) & 1, hh = threadIdx.x & 1;      // dim, block of 32 tokens, half of its slots
    float am = 0.f;
#pragma unroll
    for (int k = 0; k < 16; k++) { v[k] = vl[32 * b + a8_slot_token(16 * hh + k)][d]; am = fmaxf(am, fabsf(v[k])); }
    am = __uint_as_float(max(__float_as_uint(am), d_quad_xor_u<1>(__float_as_uint(am))));
    const int e = d_mx_exp(am, MI_INVQ8);
    const size_t td = ((size_t)h * (R / 64) + tile) * HD + d;
    *(uint4 *)(vt + td * 64 + b * 32 + hh * 16) = make_uint4(d_enc4_e4m3(v[0], v[1], v[2], v[3], e), d_enc4_e4m3(v[4], v[5], v[6], v[7], e), d_enc4_e4m3(v[8], v[9], v[10], v[11], e), d_enc4_e4m3(v[12], v[13], v[14], v[15], e));
    if (!hh) vts[td * 2 + b] = (uint8_t)(e + 127);
}

__device__ __forceinline__ float a8_xor32f(float x, int h) {
    const unsigned u = __float_as_uint(x);
    const auto r2 = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __uint_as_float(h ? r2[0] : r2[1]);
}
// the larger of the lane's and its partner's value
__device__ __forceinline__ float a8_max32f(float x) {
    const unsigned u = __float_as_uint(x);
    const auto r2 = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaxf(__uint_as_float(r2[0]), __uint_as_float(r2[1]));
}
// 2^(s sl2 - m): the scaled logit is rounded before the maximum is taken off, as where the maximum was formed
__device__ __forceinline__ float a8_prob(float s, float sl2, float m) {
#pragma clang fp contract(off)
    return __builtin_amdgcn_exp2f(s * sl2 - m);
}
// the lane's fragment of a 64-byte row of two 32-K blocks: bytes 16 h ... of each (p already points at byte 16 h)
__device__ __forceinline__ v8i a8_frag(const uint8_t *p) {
    const v4i lo = *(const v4i *)p, hi = *(const v4i *)(p + 32);
    return (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

// the same through a pointer whose uniform part is in scalar registers (opaque: the address is not folded into the lane's offset) and a 32-bit lane offset
typedef const __attribute__((address_space(1))) uint8_t *a8_gp;
__device__ __forceinline__ a8_gp a8_uniform(const uint8_t *p) { a8_gp g = (a8_gp)p; asm("" : "+s"(g)); return g; }
__device__ __forceinline__ v8i a8_frag(a8_gp p, unsigned o) {
    typedef const __attribute__((address_space(1))) v4i *g4;
    const v4i lo = *(g4)(p + o), hi = *(g4)(p + o + 32);
    return (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

// grid: H nseq (sequence, head) pairs, the pairs fastest, times the query tiles of 32. Consecutive workgroups go to the XCDs in turn, so with 8 pairs (or
// a divisor or multiple) each XCD's L2 holds one pair's K and V (120 bytes per key, 0.5 MB at 4 100) instead of all of them. Fragments are the quantised
// tensors' rows as they lie in memory (32 contiguous bytes per lane), loaded from global memory directly.
// A key tile of 64 keys is four matrix products (256 cycles) and about 210 vector instructions, 34 of them exponentials. Many query tiles (several wavefronts per
// SIMD): bound by those, 1 300 cycles per tile at 16 x 4 heads of 4 100 tokens (513 -> 340 us; block maxima, masks and rescalings that change nothing left out, 268 + 57
// instructions before). One wavefront per SIMD (129 x 4 tiles): its own chain, hence the products of the next tile beside the softmax of this one (66 -> 55 us; 202 registers
// and two wavefronts per SIMD, which costs the many-tile launches 1 %) and loads whose addresses and waits are the hardware's, not the compiler's.
// A workgroup of four wavefronts whose first alone has queries (the sequence's last query tile: the few tokens past a multiple of 128) shares that
// tile's keys among its wavefronts, a range of the key tiles each, and merges the four partial softmaxes. Each wavefront starts from the running maximum of the
// tiles before its range, so the probabilities and their e4m3 codes are those of the one-wavefront pass; only the order in which the partial sums are
// added differs. The maxima come from a first walk of the wavefronts over their own ranges (the K Q^T products and a maximum per logit), exchanged through LDS.
__global__ void __launch_bounds__(256, 2) a8_fwd_k(const uint8_t *__restrict__ Q8, const uint8_t *__restrict__ Q8s, const uint8_t *__restrict__ K8, const uint8_t *__restrict__ K8s,
                                                const uint8_t *__restrict__ Vt, const uint8_t *__restrict__ Vts, float *__restrict__ o, float *__restrict__ lse,
                                                int S, int Sp, int H, int C, long long R, float sl2, unsigned pairs) {
    const unsigned bq = blockIdx.x / pairs, bp = blockIdx.x - bq * pairs;
    const int seq = (int)(bp / (unsigned)H), hd = (int)(bp - (unsigned)seq * (unsigned)H), tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nwv = blockDim.x >> 6, tq = (int)bq * nwv;
    const bool split = nwv == 4 && (tq + 1) * 32 >= S;
    const int q0 = (split ? tq : tq + wave) * 32;
    if (q0 >= S) return;                                   // (no barriers outside a split workgroup: a wavefront without queries leaves)
    const long long rb = (long long)hd * R + (long long)seq * Sp;          // the sequence's first row in the row-quantised tensors
    const long long tb = rb / FT;                                          // ... and its first key tile in the transposed one
    const v8i qf = a8_frag(Q8 + (rb + q0 + r) * 64 + 16 * h);
    const int qs = Q8s[(rb + q0 + r) * 2 + h];
    // (uniform bases and small lane offsets: one address instruction per load or none)
    const uint8_t *kp = K8 + rb * 64, *ksp = K8s + rb * 2;
    const unsigned ko = (unsigned)(r * 64 + 16 * h), kso = (unsigned)(r * 2 + h);
    // V^T rows: dims r and 32 + r (of the second the first 16 are real; the others repeat the last one into accumulator rows that are never read)
    const int d1 = min(32 + r, HD - 1);
    const uint8_t *vp = Vt + tb * (HD * 64), *vsp = Vts + tb * (HD * 2);
    const unsigned vo0 = (unsigned)(r * 64 + 16 * h), vo1 = (unsigned)(d1 * 64 + 16 * h), vso0 = (unsigned)(r * 2 + h), vso1 = (unsigned)(d1 * 2 + h);
    const int nt = (S + FT - 1) / FT;
    // the K fragments of a tile are requested behind the products of the one before it, into the registers those products have read, and so are the V
    // fragments: K then has the softmax and the second products of a tile to arrive, V the next tile's first products and softmax
    v8i kf[2], vf0, vf1; int ks[2], e0v, e1v;
    auto request_k = [&](int it) {
        const a8_gp k = a8_uniform(kp + (size_t)it * (FT * 64)), s = a8_uniform(ksp + (size_t)it * (FT * 2));
#pragma unroll
        for (int b = 0; b < 2; b++) { kf[b] = a8_frag(k, ko + 2048u * b); ks[b] = s[kso + 64u * b]; }
    };
    auto request_v = [&](int it) {
        const a8_gp v = a8_uniform(vp + (size_t)it * (HD * 64)), vs = a8_uniform(vsp + (size_t)it * (HD * 2));
        vf0 = a8_frag(v, vo0); vf1 = a8_frag(v, vo1); e0v = vs[vso0]; e1v = vs[vso1];
    };
    // S^T = K Q^T for the two blocks of 32 keys of tile it, the next tile's K requested behind it (the last tile re-requests itself)
    auto logits = [&](int it, v16f (&s)[2]) {
#pragma unroll
        for (int b = 0; b < 2; b++) {
            v16f z;
#pragma unroll
            for (int i = 0; i < 16; i++) z[i] = 0.f;
            s[b] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(kf[b], qf, z, 0, 0, 0, ks[b], 0, qs);
        }
        __builtin_amdgcn_sched_barrier(0);
        request_k(min(it + 1, nt - 1));
        __builtin_amdgcn_sched_barrier(0);
    };
    extern __shared__ float4 cmb4[];                       // split: [range][6][lane] float4 of O^T, then [range][2][lane] floats: m, l; the exchanged maxima before that
    float m = -INFINITY;
    int it0 = 0, it1 = nt;
    if (split) {
        const int cut[5] = {0, nt * 34 / 100, nt * 61 / 100, nt * 83 / 100, nt};
        it0 = cut[wave]; it1 = cut[wave + 1];
        float mx = -INFINITY;
        if (wave < 3) {                                    // (keys past S count for nothing here: a range that holds the last tile has none behind it)
            request_k(min(it0, nt - 1));
            // (the loads of tile it + 1 are requested behind the products of tile it, into the registers these have read)
            for (int it = it0; it < it1; it++) {
                v16f s[2];
                logits(it, s);
#pragma unroll
                for (int b = 0; b < 2; b++)
#pragma unroll
                    for (int i = 0; i < 16; i++) mx = fmaxf(mx, s[b][i]);
            }
            mx = a8_max32f(mx) * sl2;        // (sl2 > 0 and rounding is monotone: the largest scaled logit)
        }
        float *pm = (float *)cmb4;
        pm[wave * 64 + lane] = mx;
        __syncthreads();
        if (it0 < it1) for (int w = 0; w < wave; w++) m = fmaxf(m, pm[w * 64 + lane]);      // (a range without tiles keeps -inf)
        __syncthreads();
    }
    float l = 0.f;
    v16f oa0, oa1;                                         // O^T: dims 4 h + 8 g + c in element 4 g + c; of the second tile elements 0 .. 7 are dims below 48
#pragma unroll
    for (int i = 0; i < 16; i++) { oa0[i] = 0.f; oa1[i] = 0.f; }
    auto softmax_pv = [&](int it, v16f (&s)[2], auto last) {
        if constexpr (decltype(last)::value) {             // keys past S masked (only the last tile can hold them)
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int i = 0; i < 16; i++) { const int key = it * FT + 32 * b + (i & 3) + 4 * h + 8 * (i >> 2); if (key >= S) s[b][i] = -INFINITY; }
        }
        // ---- the largest logit of each block of 32 keys, in the products' own units (the scaling to base 2 is monotone): it gives the running maximum and, as
        // the exponential of its scaled value, the largest probability of the block, which fixes the block's scale ----
        float bm[2] = {s[0][0], s[1][0]};
#pragma unroll
        for (int i = 1; i < 16; i++) { bm[0] = fmaxf(bm[0], s[0][i]); bm[1] = fmaxf(bm[1], s[1][i]); }
        bm[0] = a8_max32f(bm[0]); bm[1] = a8_max32f(bm[1]);
        const float mn = fmaxf(m, fmaxf(bm[0], bm[1]) * sl2), corr = __builtin_amdgcn_exp2f(m - mn);
        m = mn;
        if (__builtin_amdgcn_ballot_w64(corr != 1.f) != 0ull) {      // (uniform: most tiles late in a row raise no query's maximum)
#pragma unroll
            for (int i = 0; i < 16; i++) oa0[i] *= corr;
#pragma unroll
            for (int i = 0; i < 16; i++) oa1[i] *= corr;
        }
        // ---- P = 2^(logit - m) -> e4m3 with one scale per query per 32 keys; the lane's codes are its B fragment, its scale operand is block h's ----
        unsigned cw[2][4]; int ep[2];
#pragma unroll
        for (int b = 0; b < 2; b++) {
            ep[b] = d_mx_expb_fin(a8_prob(bm[b], sl2, m), MI_INVQ8);
            const float p2e = __uint_as_float((unsigned)ep[b] << 23);
#pragma unroll
            for (int i = 0; i < 16; i++) { s[b][i] = a8_prob(s[b][i], sl2, m); l = b || i ? l + s[b][i] : fmaf(l, corr, s[b][i]); }
#pragma unroll
            for (int q = 0; q < 4; q++) cw[b][q] = d_enc_e4m3x4_hw(s[b][4 * q], s[b][4 * q + 1], s[b][4 * q + 2], s[b][4 * q + 3], p2e);
        }
        const v8i pf = {(int)cw[0][0], (int)cw[0][1], (int)cw[0][2], (int)cw[0][3], (int)cw[1][0], (int)cw[1][1], (int)cw[1][2], (int)cw[1][3]};
        const int ps = h ? ep[1] : ep[0];
        // ---- O^T += V^T P^T ----
        oa0 = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(vf0, pf, oa0, 0, 0, 0, e0v, 0, ps);
        oa1 = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(vf1, pf, oa1, 0, 0, 0, e1v, 0, ps);
        if constexpr (!decltype(last)::value) { __builtin_amdgcn_sched_barrier(0); request_v(it + 1); __builtin_amdgcn_sched_barrier(0); }
    };
    if (it0 < it1) {
        // the products of tile it + 1 are issued before the softmax of tile it, whose vector instructions run beside them
        request_k(it0); request_v(it0);
        v16f sa[2], sb[2];
        logits(it0, sa);
        int it = it0;
        for (; it + 2 < it1; it += 2) {
            logits(it + 1, sb); softmax_pv(it, sa, std::false_type{});
            logits(it + 2, sa); softmax_pv(it + 1, sb, std::false_type{});
        }
        if (it + 1 < it1) { logits(it + 1, sb); softmax_pv(it, sa, std::false_type{}); softmax_pv(it + 1, sb, std::true_type{}); }
        else softmax_pv(it, sa, std::true_type{});
    }
    l += a8_xor32f(l, h);
    const int i = q0 + r;
    float *orow = o + ((size_t)seq * S + (i < S ? i : S - 1)) * C + hd * HD + 4 * h;
    if (!split) {
        if (i >= S) return;
        const float il = 1.f / l;
#pragma unroll
        for (int g = 0; g < 4; g++) *(float4 *)(orow + 8 * g) = make_float4(oa0[4 * g] * il, oa0[4 * g + 1] * il, oa0[4 * g + 2] * il, oa0[4 * g + 3] * il);
#pragma unroll
        for (int g = 0; g < 2; g++) *(float4 *)(orow + 32 + 8 * g) = make_float4(oa1[4 * g] * il, oa1[4 * g + 1] * il, oa1[4 * g + 2] * il, oa1[4 * g + 3] * il);
        if (!h) lse[((size_t)seq * H + hd) * S + i] = m + __log2f(l);
        return;
    }
    // partial (m, l, O^T) of the key ranges -> LDS; every wavefront adds its share of the dims in range order at the common maximum (a wavefront without
    // keys holds l = 0, O = 0; its factor, of a maximum at most the common one, is finite)
    float *ml = (float *)(cmb4 + 4 * 6 * 64);
#pragma unroll
    for (int g = 0; g < 4; g++) cmb4[(wave * 6 + g) * 64 + lane] = make_float4(oa0[4 * g], oa0[4 * g + 1], oa0[4 * g + 2], oa0[4 * g + 3]);
#pragma unroll
    for (int g = 0; g < 2; g++) cmb4[(wave * 6 + 4 + g) * 64 + lane] = make_float4(oa1[4 * g], oa1[4 * g + 1], oa1[4 * g + 2], oa1[4 * g + 3]);
    ml[(wave * 2) * 64 + lane] = m; ml[(wave * 2 + 1) * 64 + lane] = l;
    __syncthreads();
    float mw[4], mm = -INFINITY, ls = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) { mw[w] = ml[(w * 2) * 64 + lane]; mm = fmaxf(mm, mw[w]); }
#pragma unroll
    for (int w = 0; w < 4; w++) { mw[w] = __builtin_amdgcn_exp2f(mw[w] - mm); ls = fmaf(ml[(w * 2 + 1) * 64 + lane], mw[w], ls); }
    if (i >= S) return;
    const float il = 1.f / ls;
    for (int g = wave; g < 6; g += 4) {                    // (float4 group g: dims 8 g + 4 h ...)
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const float4 p = cmb4[(w * 6 + g) * 64 + lane];
            a.x = fmaf(p.x, mw[w], a.x); a.y = fmaf(p.y, mw[w], a.y); a.z = fmaf(p.z, mw[w], a.z); a.w = fmaf(p.w, mw[w], a.w);
        }
        *(float4 *)(orow + 8 * g) = make_float4(a.x * il, a.y * il, a.z * il, a.w * il);
    }
    if (wave == 3 && !h) lse[((size_t)seq * H + hd) * S + i] = mm + __log2f(ls);
}

static int g_a8_waves = 0;
extern "C" void at_fa8_waves(int nw) { g_a8_waves = nw == 1 || nw == 4 ? nw : 0; }
namespace {
// the quantised operands of one call in the library's scratch, and the core on them
struct a8_ops { uint8_t *q8, *k8, *qs, *ks, *vt, *vts; int Sp; long long R; };
bool a8_carve(a8_ops *w, const at_geom *g, int H) {
    w->Sp = (g->S + FT - 1) / FT * FT; w->R = (long long)g->nseq * w->Sp;
    const size_t rq = (size_t)H * w->R * 64, rqs = (size_t)H * w->R * 2, tq = (size_t)H * HD * w->R, tqs = (size_t)H * HD * (w->R / 32);
    auto al = [](size_t n) { return (n + 255) & ~(size_t)255; };
    uint8_t *base = (uint8_t *)mi_ws(MI_WS_ATTN, 2 * (al(rq) + al(rqs)) + al(tq) + al(tqs));
    if (!base) return false;
    w->q8 = base; w->k8 = w->q8 + al(rq); w->qs = w->k8 + al(rq); w->ks = w->qs + al(rqs); w->vt = w->ks + al(rqs); w->vts = w->vt + al(tq);
    return true;
}
void a8_core(const a8_ops &w, float *o, float *lse, const at_geom *g, int H, int C) {
    // four wavefronts share a workgroup's reads of K and V, and its last query tile when that is alone (8 stragglers of 1 032 tiles on 1 024 SIMDs otherwise: 90 against 65 us);
    // sequences of at most 256 tokens have too few key tiles to share (5 tokens: 9.8 against 10.3 us)
    const size_t pairs = (size_t)H * g->nseq, qt = (size_t)(g->S + 31) / 32;
    const int nw = g_a8_waves ? g_a8_waves : g->S <= 256 ? 1 : 4;
    const size_t nblk = pairs * ((qt + nw - 1) / nw);
    if (nblk * (size_t)(64 * nw) >= (size_t)1 << 32) mi_die("at_fa8_fwd: %zu workgroups exceed the launch grid", nblk);
    a8_fwd_k<<<(unsigned)nblk, 64 * nw, nw == 4 ? 4 * 26 * 64 * sizeof(float) : 0>>>(w.q8, w.qs, w.k8, w.ks, w.vt, w.vts, o, lse, g->S, w.Sp, H, C, w.R, 1.4426950408889634f / sqrtf((float)HD), (unsigned)pairs);
    MICK();
}
}
extern "C" int at_fa8_fwd(const void *qkvh, float *o, float *lse, const at_geom *g, int H, int C) {
    if (!g || g->nseq <= 0 || g->S <= 0 || H <= 0) return 0;
    if (C != H * HD) mi_die("at_fa8_fwd: C %d is not %d heads of %d", C, H, HD);
    if (g->lens || g->rays) mi_die("at_fa8_fwd: per-sequence lengths and ray geometry are not supported");
    a8_ops w;
    if (!a8_carve(&w, g, H)) return -1;
    const long long Tp = (long long)g->nseq * g->S + FT;
    const __half *Qh = (const __half *)qkvh, *Kh = Qh + (size_t)H * Tp * HD, *Vh = Kh + (size_t)H * Tp * HD;
    // (queries and keys in one launch: their sources, code planes and scale planes each lie one fixed stride apart)
    a8_rows_k<<<dim3(nblk_((size_t)H * w.R * 4, 256), 2), 256>>>(Qh, w.q8, w.qs, H, g->nseq, g->S, w.Sp, Tp, (size_t)(Kh - Qh), (size_t)(w.k8 - w.q8), (size_t)(w.ks - w.qs));
    a8_vt_k<<<nblk_((size_t)H * (w.R / 32), 4), 256>>>(Vh, w.vt, w.vts, H, g->nseq, g->S, w.Sp, Tp);
    a8_core(w, o, lse, g, H, C);
    return 0;
}
// workgroups of a8_pack_k: the three parts of every 64-token tile (sequences padded to whole tiles) and head, tiles rounded up to eight
static unsigned long long a8_pack_blocks(int nseq, int S, int H) { return ((unsigned long long)nseq * (((unsigned)S + FT - 1) / FT) + 7) / 8 * 8 * 3 * (unsigned)H; }
// a launch has fewer than 2^32 threads. Short sequences reach that first, every one of them being a tile (5.6 million sequence x head pairs of up to 64 tokens); the separate passes'
// launches have a third of the threads at most
extern "C" int at_fa8_one_pass(int nseq, int S, int H) { return nseq > 0 && S > 0 && H > 0 && a8_pack_blocks(nseq, S, H) < (1ull << 32) / 256; }
// (internal) at_fa_pack and at_fa8_fwd from the projection's rows qkv [T][3 C], 16-byte aligned, without the binary16 tensor between them: the same operands, the same
// outputs, rq / rk / amx included (amx: four floats that are zero when this runs). at_fa8_one_pass(g->nseq, g->S, H) must hold
int mi_fa8_from_qkv(const float *qkv, const float *qg, const float *kg, float *rq, float *rk, float *amx, float *o, float *lse, const at_geom *g, int nreg, int H, int rope, float base) {
    a8_ops w;
    if (!a8_carve(&w, g, H)) return -1;
    const rope_t rp = {rope, g->S, g->Hh, g->W, nreg, log2f(base), rope ? g->pos : nullptr};
#define A8P(MODE) a8_pack_k<MODE><<<(unsigned)a8_pack_blocks(g->nseq, g->S, H), 256>>>(qkv, qg, kg, w.q8, w.qs, (size_t)(w.k8 - w.q8), (size_t)(w.ks - w.qs), w.vt, w.vts, rq, rk, amx, H, g->S, (unsigned)(w.Sp / 64), w.R, rp)
    switch (rope_mode(rp)) { case ROPE_TABLE: A8P(ROPE_TABLE); break; case ROPE_REAL: A8P(ROPE_REAL); break; default: A8P(ROPE_EACH); }
#undef A8P
    a8_core(w, o, lse, g, H, H * HD);
    return 0;
}
