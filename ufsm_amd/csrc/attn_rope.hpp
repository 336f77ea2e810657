// The rotary embedding of the QKV packs (attn_block.hip, attn8.hip): 16 dims per coordinate, pair f of a coordinate turns by position x base^(-f / 8)
// (src/nn_attn_tc.cu:99-136, src/nn_attn.cu:272-289 of the reference). Angles of whole positions take few values, and a sine / cosine pair costs far more than the rest
// of a row: a workgroup forms them once, a table [position][8] in LDS, positions below ROPE_TAB per axis.
#pragma once
#include "mx_dev.hpp"

constexpr int ROPE_TAB = 64;
struct rope_t { int on, S, Hh, W, nreg; float lbase; const float *gpos; };      // lbase: log2 of the base; gpos: per-token coordinates [T][3] (null: the grid indices)
// positions along an axis: < this (registers included in S: an upper bound); the table serves when it is at most ROPE_TAB (gpos: real numbers, every angle is evaluated)
__device__ __forceinline__ int rope_positions(const rope_t &R) { return max(max(R.S / (R.Hh * R.W), R.Hh), R.W); }
__device__ __forceinline__ void rope_fill(float2 *tab, int pmax, float lbase) {
    for (int i = threadIdx.x; i < pmax * 8; i += blockDim.x) { float sn, cs; sincosf((float)(i >> 3) * exp2f(-lbase * (float)(i & 7) / 8.f), &sn, &cs); tab[i] = make_float2(sn, cs); }
}
// how a launch evaluates its angles, known to the host (a template argument of the packs: sixteen inlined sines that a launch never runs are 30 KB of code that it
// still fetches): from the table, the hardware sine / cosine of real coordinates (as the reference's fast-math build), or one by one
enum { ROPE_TABLE = 0, ROPE_REAL = 1, ROPE_EACH = 2 };
// coordinate ax of grid token ts >= 0 of token row t (two unsigned divisions whatever the axis: the lanes of a wavefront hold all three)
template <int MODE> __device__ __forceinline__ float rope_pos(const rope_t &R, long long t, int ts, int ax) {
    if (MODE == ROPE_REAL) return R.gpos[3 * t + ax];
    const unsigned row = (unsigned)ts / (unsigned)R.W, z = row / (unsigned)R.Hh;
    return (float)(ax == 0 ? z : ax == 1 ? row - z * (unsigned)R.Hh : (unsigned)ts - row * (unsigned)R.W);
}
inline int rope_mode(const rope_t &R) {
    if (!R.on) return ROPE_TABLE;                              // (nothing turns: no table is formed either)
    if (R.gpos) return ROPE_REAL;
    if (R.Hh <= 0 || R.W <= 0) return ROPE_EACH;               // (no grid: an empty call's geometry; nothing here may divide by it)
    const int a = R.S / (R.Hh * R.W), b = R.Hh > R.W ? R.Hh : R.W;
    return (a > b ? a : b) <= ROPE_TAB ? ROPE_TABLE : ROPE_EACH;
}
// pair (a, b) of frequency fi turned
template <int MODE> __device__ __forceinline__ void rope_turn(const rope_t &R, const float2 *tab, float pos, int fi, float &a, float &b) {
    float sn, cs;
    if (MODE == ROPE_TABLE) { const float2 sc2 = tab[(int)pos * 8 + fi]; sn = sc2.x; cs = sc2.y; }
    else if (MODE == ROPE_REAL) { const float ang = pos * exp2f(-R.lbase * (float)fi / 8.f); sn = __sinf(ang); cs = __cosf(ang); }
    else sincosf(pos * exp2f(-R.lbase * (float)fi / 8.f), &sn, &cs);
    const float x = a, y = b;
    a = x * cs - y * sn; b = x * sn + y * cs;
}
