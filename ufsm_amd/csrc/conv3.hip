// Host side of the 3x3x3 MX convolutions: entry points, operand re-staging, weight preparation and memo, tile-shape selection,
// GroupNorm partial-sum reduction. The kernel itself is conv3_kernel.hpp, instantiated per (compute format, output kind) in
// conv3_f*_o*.hip.
#include "conv3_kernel.hpp"
#include <mutex>

// what a reduce block does with the (sum, sum of squares) of its (sample, group): add them to the caller's sum slots (the reference's contract,
// src/lp_common.cuh:1575-1597), or, for a fused call, set the slots and finalize mean / rstd from them right away (src/nn_elem.cu:5-11), which saves
// the zeroing and finalize launches around the conv
struct gn_fin_t { float *mean, *rstd; double len; float eps; };
__device__ __forceinline__ void gn_part_finish(double *osum, double s, double ss, gn_fin_t fin, unsigned ng) {
    const size_t i = 2 * (size_t)ng;
    if (!fin.mean) { gn_acc_add(osum, i, s); gn_acc_add(osum, i + 1, ss); return; }
    unsigned long long *w = (unsigned long long *)osum + 3 * i;
    const double gs = gn_slot_value(s, w), gss = gn_slot_value(ss, w + 3);
    gn_mean_rstd(gs, gss, fin.len, fin.eps, fin.mean + ng, fin.rstd + ng);
}

// (sum, sum of squares) partials of the tiles -> exact GroupNorm sum slots (src/lp_common.cuh:1575-1597 does the same with one fixed-point atomic
// per block and channel). A spatial tile's record is Q = Co / 4 (padded to whole channel slices) consecutive float2, one per channel quad; quad
// Q = co / 4 lives in channel slice Q / (8 MT), slot Q % (8 MT). A block takes one sample's tiles [t0, t1) with ALL their quads: thread (j, q) adds
// quad q of tiles t0 + j, t0 + j + J, ... in double (consecutive threads read consecutive records: every fetched line is used whole), then thread g
// adds its group's quads over the J rows (of 1024 threads: added in halves down to four first), all in a fixed order. nsplit > 1 (thousands of tiles: the level-0 layers): every block leaves its Go pairs
// in scr and takes a ticket of its sample; the block that draws the last one adds the nsplit pairs of every group in index order - the result
// does not depend on which block that is - and puts the ticket counter back to zero for the next launch
struct gn_split_t { int nsplit; double *scr; unsigned *cnt; };
template <int NTH>
__global__ void __launch_bounds__(NTH) gn_part_reduce_k(const float2 *part, int tiles_per_n, int ncs, int MT, int Co, int Go, double *osum, gn_fin_t fin, gn_split_t sp) {
    const int n = (int)blockIdx.x / sp.nsplit, pi = (int)blockIdx.x % sp.nsplit, tid = (int)threadIdx.x;
    const int Q = ncs * MT * 8, nst = tiles_per_n / ncs, qpg = Co / Go / 4, J = NTH / Q;
    const int per = (nst + sp.nsplit - 1) / sp.nsplit, t0 = pi * per, t1 = min(nst, t0 + per);
    const int q = tid % Q, j = tid / Q;
    const float2 *rec = part + (size_t)n * tiles_per_n * (MT * 8) + q;
    double s = 0.0, ss = 0.0;
    if (j < J) {
#pragma unroll 8
        for (int st = t0 + j; st < t1; st += J) {                            // (unrolled: the records' loads of several rounds are in flight together)
            const float2 p = rec[(size_t)st * Q];
            s += (double)p.x; ss += (double)p.y;
        }
    }
    __shared__ double r1[NTH], r2[NTH];
    __shared__ unsigned ticket;
    r1[tid] = s; r2[tid] = ss;
    __syncthreads();
    int JJ = J;
    if constexpr (NTH > 256) {                                               // the J rows of partial sums in halves down to four, in a fixed order
        while (JJ > 4) {
            const int hlf = (JJ + 1) >> 1;
            if (j < JJ - hlf) { r1[tid] += r1[tid + hlf * Q]; r2[tid] += r2[tid + hlf * Q]; }
            __syncthreads();
            JJ = hlf;
        }
    }
    s = 0.0; ss = 0.0;
    if (tid < Go)
        for (int k = 0; k < qpg; k++)
            for (int jj = 0; jj < JJ; jj++) { s += r1[jj * Q + tid * qpg + k]; ss += r2[jj * Q + tid * qpg + k]; }
    if (sp.nsplit == 1) { if (tid < Go) gn_part_finish(osum, s, ss, fin, (unsigned)(n * Go + tid)); return; }
    if (tid < Go) {
        double *mine = sp.scr + 2 * ((size_t)blockIdx.x * Go + tid);
        __hip_atomic_store(mine, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); __hip_atomic_store(mine + 1, ss, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __threadfence();                                                    // the pairs are visible device-wide before the ticket is
    }
    __syncthreads();
    if (tid == 0) ticket = atomicAdd(sp.cnt + n, 1u);
    __syncthreads();
    if (ticket != (unsigned)sp.nsplit - 1u) return;                         // (uniform over the block)
    __threadfence();                                                        // the last block of the sample: every other block's pairs are visible
    if (tid == 0) __hip_atomic_store(sp.cnt + n, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (tid < sp.nsplit * Go) {                                             // (nsplit Go <= 256) all pairs of the sample at once, then added in index order
        const double *theirs = sp.scr + 2 * ((size_t)n * sp.nsplit * Go + tid);
        r1[tid] = __hip_atomic_load(theirs, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); r2[tid] = __hip_atomic_load(theirs + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (tid >= Go) return;
    s = 0.0; ss = 0.0;
    for (int k = 0; k < sp.nsplit; k++) { s += r1[k * Go + tid]; ss += r2[k * Go + tid]; }
    gn_part_finish(osum, s, ss, fin, (unsigned)(n * Go + tid));
}
// the same for few records (mi_records_few): a block per 32 channels and sample, whose threads add in the order of the pre-pass that forms statistics itself
// (restage32_k<..., RED>, mx_elem.hip: a change here is one there); a group is finished by the block it starts in. Bound by the launch and one chain of loads: 3.9 - 5.2 us where
// the kernel above takes 3.9 - 5.8 (8 to 512 records of 8 to 128 quads, 1 and 2 samples; even at 32 and 64 channels, 4.7 -> 3.1 at 512 from 16^3)
__global__ void __launch_bounds__(256) gn_part_reduce_few_k(gn_records_t rec, int C, double *osum, gn_fin_t fin) {
    __shared__ double r1[256], r2[256];
    const int nb = C / 32, n = (int)blockIdx.x / nb, blk = (int)blockIdx.x - n * nb;
    const int cpg = C / rec.Go, g0 = blk * 32 / cpg, g1 = (blk * 32 + 31) / cpg, qpg = cpg >> 2;      // (the groups the block's channels lie in and their quads: at most 16)
    const float2 *rp = rec.part + (size_t)n * rec.nst * rec.Q + g0 * qpg + min((int)(threadIdx.x & 15), (g1 - g0 + 1) * qpg - 1);
    double s = 0.0, ss = 0.0;
#pragma unroll 8
    for (int t = threadIdx.x >> 4; t < rec.nst; t += 16) { const float2 v = rp[(size_t)t * rec.Q]; s += (double)v.x; ss += (double)v.y; }      // thread (quad q, j): records j, j + 16, ...
    r1[threadIdx.x] = s; r2[threadIdx.x] = ss;
    __syncthreads();
    if (threadIdx.x < 64) {                                   // lane (q, part): a quad's sums over four of the sixteen rows, then over the four lanes of the quad
        const int qq = threadIdx.x & 15, k0 = threadIdx.x >> 4;
        s = (r1[(4 * k0) * 16 + qq] + r1[(4 * k0 + 1) * 16 + qq]) + (r1[(4 * k0 + 2) * 16 + qq] + r1[(4 * k0 + 3) * 16 + qq]);
        ss = (r2[(4 * k0) * 16 + qq] + r2[(4 * k0 + 1) * 16 + qq]) + (r2[(4 * k0 + 2) * 16 + qq] + r2[(4 * k0 + 3) * 16 + qq]);
        s += __shfl_xor(s, 16); s += __shfl_xor(s, 32); ss += __shfl_xor(ss, 16); ss += __shfl_xor(ss, 32);
        if (threadIdx.x < 16) { r1[threadIdx.x] = s; r2[threadIdx.x] = ss; }
    }
    __syncthreads();
    const int g = g0 + (int)threadIdx.x;
    if (g > g1 || g * cpg < blk * 32) return;
    s = 0.0; ss = 0.0;
    for (int k = 0; k < qpg; k++) { s += r1[threadIdx.x * qpg + k]; ss += r2[threadIdx.x * qpg + k]; }
    gn_part_finish(osum, s, ss, fin, (unsigned)(n * rec.Go + g));
}

// the same with one block per (sample, group), for records wider than a block (more than 1024 channels) or more than 256 groups
__global__ void __launch_bounds__(256) gn_part_reduce_g_k(const float2 *part, int tiles_per_n, int ncs, int MT, int Co, int Go, double *osum, gn_fin_t fin) {
    const int n = blockIdx.x / Go, gidx = blockIdx.x % Go, qpg = Co / Go / 4, nq = MT * 8, nst = tiles_per_n / ncs;
    double s = 0.0, ss = 0.0;
#pragma unroll 8
    for (int i = threadIdx.x; i < nst * qpg; i += 256) {
        const int st = i / qpg, Q = gidx * qpg + i % qpg, cs = Q / nq, qd = Q - cs * nq;
        const float2 p = part[(size_t)(n * tiles_per_n + st * ncs + cs) * nq + qd];
        s += (double)p.x; ss += (double)p.y;
    }
    __shared__ double r1[256], r2[256];
    r1[threadIdx.x] = s; r2[threadIdx.x] = ss;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) { if ((int)threadIdx.x < st) { r1[threadIdx.x] += r1[threadIdx.x + st]; r2[threadIdx.x] += r2[threadIdx.x + st]; } __syncthreads(); }
    if (threadIdx.x == 0) gn_part_finish(osum, r1[0], r2[0], fin, blockIdx.x);
}

// the same from per-channel records (32 per tile: launches whose channels per group are not a multiple of 4 run one channel tile per workgroup,
// ncs channel slices of 32 per spatial tile)
__global__ void __launch_bounds__(256) gn_part_reduce_ch_k(const float2 *part, int tiles_per_n, int ncs, int Co, int Go, double *osum, gn_fin_t fin) {
    const int n = blockIdx.x / Go, gidx = blockIdx.x % Go, cpg = Co / Go, nst = tiles_per_n / ncs;
    double s = 0.0, ss = 0.0;
    for (int i = threadIdx.x; i < nst * cpg; i += 256) {
        const int st = i / cpg, ch = gidx * cpg + i % cpg;
        const float2 p = part[((size_t)n * tiles_per_n + (size_t)st * ncs + (ch >> 5)) * 32 + (ch & 31)];
        s += (double)p.x; ss += (double)p.y;
    }
    __shared__ double r1[256], r2[256];
    r1[threadIdx.x] = s; r2[threadIdx.x] = ss;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) { if ((int)threadIdx.x < st) { r1[threadIdx.x] += r1[threadIdx.x + st]; r2[threadIdx.x] += r2[threadIdx.x + st]; } __syncthreads(); }
    if (threadIdx.x == 0) gn_part_finish(osum, r1[0], r2[0], fin, blockIdx.x);
}

// ---- weights: fp32 w[co][ci][27] -> per (chunk, unit pair, 32-row channel tile) fragment-ordered codes + scale bytes ----
// block = the 32 ci of one (tap, co) (src/lp_f8fwd.cu:54-71, src/lp_f4fwd.cu:53-66); fmaxf amax; padded rows / channels / the odd
// padding unit are zero codes with scale byte 1
__host__ __device__ __forceinline__ int seg_ci(int cp, int Ci, int Cx, int CxP) { if (cp < CxP) return cp < Cx ? cp : -1; const int c = Cx + cp - CxP; return c < Ci ? c : -1; }
template <int FMT>
__global__ void __launch_bounds__(128) prep_w_k(const float *__restrict__ w, uint8_t *__restrict__ wq, unsigned *__restrict__ wsc, int Co, int Ci, int Cx, int CxP,
                                               int nbt, int CB, int nmt_all, int npairs_all, int block_major, int w2d) {
    constexpr int WTILE = fmt_t<FMT>::WTILE;
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    const int Cop = nmt_all * 32;
    if (i >= (size_t)npairs_all * Cop) return;
    const int cop = (int)(i % Cop), gp = (int)(i / Cop);
    int b0 = 0, pb = 0, nbc = 0;
    if (block_major >= 0) for (;; b0 += CB) { nbc = min(CB, nbt - b0); const int np = (27 * nbc + 1) >> 1; if (gp < pb + np) break; pb += np; }
    const int q = gp - pb, m = cop >> 5, r = cop & 31, cw = (cop & ~31) + mi_row_chan(r);       // row r of the tile carries output channel cw
    uint8_t *tile = wq + ((size_t)gp * nmt_all + m) * WTILE;
    unsigned *tsc = wsc + ((size_t)gp * nmt_all + m) * 64;      // one word per lane: the byte the MFMA reads is the low one
    int tss = 1;                                                // words between two lanes' scale words
    if (block_major > 0) {
        // the wide kernel's layout (block_major = its channel tiles per workgroup, 4 or 2): per slice of that many tiles, pair after pair the
        // image of its LDS stage: the tiles' codes, then per lane the tiles' scale words
        const int MW = block_major, sl = m / MW, mi = m - sl * MW;
        uint8_t *img = wq + ((size_t)sl * (npairs_all + 16) + gp) * (size_t)(MW * (WTILE + 256));
        tile = img + mi * WTILE; tsc = (unsigned *)(img + MW * WTILE) + mi; tss = MW;
    }
#pragma unroll
    for (int side = 0; side < 2; side++) {
        const int u = 2 * q + side;
        float v[32];
        // K order inside a chunk: tap by tap over its blocks, or (the wide kernel, one chunk) block by block over the taps; the row kernel
        // (block_major -1): per block 15 pairs (class c, ky), class c < 3 = taps (c, ky, 0 | 1), class 3 = (0 | 1, ky, 2), class 4 = (2, ky, 2 | none);
        // the direct stride-2 kernel (block_major -2): mi_s2_unit
        int t = block_major ? u % 27 : u / nbc, blk = block_major ? u / 27 : b0 + u % nbc;
        bool unit_ok = u < 27 * nbc;
        if (block_major == -2) unit_ok = mi_s2_unit(gp, side, nbt, &t, &blk);
        else if (block_major < 0) {
            const int qq = gp % 15, c = qq / 3, ky = qq % 3;
            blk = gp / 15;
            const int kz = c < 3 ? c : c == 3 ? side : 2, kx = c < 3 ? side : 2;
            t = kz * 9 + ky * 3 + kx;
            unit_ok = !(c == 4 && side == 1);
        }
#pragma unroll
        for (int k = 0; k < 32; k++) {
            const int ci = seg_ci(blk * 32 + k, Ci, Cx, CxP);
            v[k] = (unit_ok && cw < Co && ci >= 0) ? w[((size_t)cw * Ci + ci) * 27 + t] : 0.f;
        }
        prep_store_unit<FMT>(tile, tsc, tss, side, r, v, w2d != 0);      // (32 consecutive threads hold a channel tile's rows of this pair)
    }
}

// ---- prepared-weight memo (src/lp_f4fwd.cuh:748-770): keyed by the conv id sp.wkey and the layout ----
// (lay: what else fixes the image's layout: the wide kernel's channel tiles per workgroup, which follow the launch's tile count and mi_conv_split; a number per kernel otherwise)
struct wmemo_t { unsigned key; const float *w; int fmt, Co, Ci, Cx, nbt, CB, nmt_all, dev, lay; uint8_t *wq, *wsc; };
static std::vector<wmemo_t> g_wmemo;
static std::mutex g_wmemo_mu;      // host threads driving different devices share the list (one thread per device: the per-device scratch is not guarded)
static unsigned g_wstep = 0;
void mx_gemm_memo_clear(void);
extern "C" void lp_wmemo_clear(void) {
    MIRT(hipDeviceSynchronize());
    mx_gemm_memo_clear();
    std::lock_guard<std::mutex> lk(g_wmemo_mu);
    if (g_wmemo.empty()) return;
    for (auto &m : g_wmemo) { MIRT(hipFree(m.wq)); MIRT(hipFree(m.wsc)); }
    g_wmemo.clear();
}
// 2-D fp4 weight scales (src/lp_f4fwd.cu:4, :67-83): one E8M0 scale per tap and 32 x 32 (output x input channel) tile instead of per output
// channel; a setting change drops the prepared weights. Default from UFSM_W4_2D, as the reference
static int g_w2d = -1;
static int g_w2d_on(void) { if (g_w2d < 0) g_w2d = getenv("UFSM_W4_2D") ? atoi(getenv("UFSM_W4_2D")) : 0; return g_w2d; }
extern "C" void lp_set_w4_2d(int on) { g_w2d = on ? 1 : 0; lp_wmemo_clear(); }
extern "C" void lp_wmemo_step(unsigned step) { if (step != g_wstep) { g_wstep = step; lp_wmemo_clear(); } }
// memo entries of the layouts other source files prepare (the 2x2x2 stride-2 convs: nbt = -100, lay = down / up): the image's buffers for
// (key, weights, format, shape, lay) on the current device, allocated on first use; returns whether they already hold the prepared image
bool mi_wmemo_other(unsigned key, const float *w, int fmt, int Co, int Ci, int nmt_all, int lay, size_t wq_bytes, size_t wsc_bytes, uint8_t **wq, uint8_t **wsc) {
    int dev = 0; MIRT(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_wmemo_mu);
    for (auto &m : g_wmemo)
        if (m.key == key && m.w == w && m.fmt == fmt && m.Co == Co && m.Ci == Ci && m.nbt == -100 && m.nmt_all == nmt_all && m.dev == dev && m.lay == lay) { *wq = m.wq; *wsc = m.wsc; return true; }
    MIRT(hipMalloc((void **)wq, wq_bytes)); MIRT(hipMalloc((void **)wsc, wsc_bytes)); mi_count_alloc(); mi_count_alloc();
    if (!*wq || !*wsc) mi_die("no device memory for the prepared weights of a 2x2x2 conv");
    g_wmemo.push_back(wmemo_t{key, w, fmt, Co, Ci, Ci, -100, 0, nmt_all, dev, lay, *wq, *wsc});
    return false;
}

thread_local char g_last_kernel[128] = "";

// optional timing of the conv kernel launches alone (benchmarks): event pairs on the stream the kernel runs on
static bool g_ktime = false;
struct kev_t { hipEvent_t e0, e1; double flops; char name[96]; };
static std::vector<kev_t> g_kev;
static double g_kms = 0.0; static long g_kn = 0;
struct klaunch_t { float ms; double flops; char name[96]; };
static std::vector<klaunch_t> g_klog;             // every timed launch since mi_kernel_timing(1), in launch order
extern "C" void mi_kernel_timing(int on) {
    for (auto &e : g_kev) { MIRT(hipEventDestroy(e.e0)); MIRT(hipEventDestroy(e.e1)); }
    g_kev.clear(); g_klog.clear(); g_kms = 0.0; g_kn = 0; g_ktime = on != 0;
}
static void ktime_collect() {
    for (auto &e : g_kev) {
        float ms = 0.f;
        MIRT(hipEventSynchronize(e.e1)); MIRT(hipEventElapsedTime(&ms, e.e0, e.e1));
        g_kms += ms; g_kn++;
        klaunch_t l; l.ms = ms; l.flops = e.flops; memcpy(l.name, e.name, sizeof l.name); g_klog.push_back(l);
        MIRT(hipEventDestroy(e.e0)); MIRT(hipEventDestroy(e.e1));
    }
    g_kev.clear();
}
extern "C" double mi_kernel_timing_read(long *launches) {       // total milliseconds of the timed launches so far (synchronises)
    ktime_collect();
    if (launches) *launches = g_kn;
    return g_kms;
}
extern "C" long mi_kernel_timing_launch(long i, float *ms, double *flops, char *name, size_t name_bytes) {     // launch i of the log; returns the log's length (synchronises)
    ktime_collect();
    if (i >= 0 && i < (long)g_klog.size()) {
        if (ms) *ms = g_klog[i].ms;
        if (flops) *flops = g_klog[i].flops;
        if (name && name_bytes) { strncpy(name, g_klog[i].name, name_bytes - 1); name[name_bytes - 1] = 0; }
    }
    return (long)g_klog.size();
}
static void ktime_push(hipEvent_t ev0, hipEvent_t ev1, double flops) {
    kev_t k; k.e0 = ev0; k.e1 = ev1; k.flops = flops;
    strncpy(k.name, g_last_kernel, sizeof k.name - 1); k.name[sizeof k.name - 1] = 0;
    g_kev.push_back(k);
}
extern "C" const char *mi_last_kernel(void) { return g_last_kernel; }

// the conv of every entry point: fmt 8 / 4 = compute format, stride 1 / 2
// set by mi_conv_fwd_gn around its conv: finalize the statistics in the reduce kernel
static thread_local gn_fin_t g_fin = {nullptr, nullptr, 0.0, 0.f};
// GroupNorm partial sums of a conv's tiles -> the caller's sum slots (and mean / rstd when mi_conv_fwd_gn asked for them)
// set by mi_conv_fwd_gn_stage around its conv: silu(gn(output)) as the next reader's operand rows
struct gn_stage_t { const float *gamma, *beta; void *y8, *y4; };
static thread_local gn_stage_t g_stage = {nullptr, nullptr, nullptr, nullptr};
static void conv_stats_reduce(const char *who, const conv_args &a, int MT, split_t sp, double *osum) {
    gn_fin_t fin = g_fin;
    fin.len = (double)(a.Co / a.Go) * (double)a.Do * a.Ho * a.Wo;
    if (fin.mean && (sp.zlo || sp.zhi)) mi_die("%s: fused finalize with a z range", who);
    if (g_stage.gamma) {
        // few records: the pre-pass that follows adds them itself, one launch less (its rule: mi_restage_records)
        const gn_stage_t g = g_stage; g_stage.gamma = nullptr;
        const int xdt = a.ydt; const size_t S = (size_t)a.Do * a.Ho * a.Wo;
        const gn_records_t rec = {(const float2 *)a.part, (int)(a.ntiles / a.N) * a.wrec / a.ncs, a.ncs * MT * 8, a.Go, fin.len, fin.eps, fin.mean, fin.rstd};
        if (!a.stat_ch && mi_restage_records(a.y, xdt, a.N, a.Co, S, g.gamma, g.beta, rec, g.y8, g.y4)) return;
        conv_stats_reduce(who, a, MT, sp, osum);
        gnp_t gp; memset(&gp, 0, sizeof gp); gp.gamma = g.gamma; gp.beta = g.beta; gp.mean = fin.mean; gp.rstd = fin.rstd; gp.G = a.Go;
        if (g.y8 && g.y4) mi_restage_sub2(a.y, xdt, a.N, a.Co, S, gp, g.y8, g.y4, S, 0);
        else {
            if (g.y8) mi_restage_sub(a.y, xdt, a.N, a.Co, S, gp, a.Co, 0, g.y8, 8, S, 0);
            if (g.y4) mi_restage_sub(a.y, xdt, a.N, a.Co, S, gp, a.Co, 0, g.y4, 4, S, 0);
        }
        return;
    }
    if (a.stat_ch) { gn_part_reduce_ch_k<<<a.N * a.Go, 256>>>((const float2 *)a.part, (int)(a.ntiles / a.N), a.ncs, a.Co, a.Go, osum, fin); MICK(); return; }
    const int tiles_per_n = (int)(a.ntiles / a.N) * a.wrec;      // (records)
    const int Q = a.ncs * MT * 8, nst = tiles_per_n / a.ncs;
    if (mi_records_few(a.Co, a.Go, nst)) {
        const gn_records_t rec = {(const float2 *)a.part, nst, Q, a.Go, fin.len, fin.eps, nullptr, nullptr};
        gn_part_reduce_few_k<<<a.N * (a.Co / 32), 256>>>(rec, a.Co, osum, fin); MICK(); return;
    }
    if (Q > 256 || a.Go > 256) { gn_part_reduce_g_k<<<a.N * a.Go, 256>>>((const float2 *)a.part, tiles_per_n, a.ncs, MT, a.Co, a.Go, osum, fin); MICK(); return; }
    // thousands of tiles per sample: several blocks each (512 tiles or more per block), folded by the last one done. The pairs and ticket
    // counters live in a small buffer per device, allocated on first use and left zeroed by every launch (the entry point that must not
    // allocate keeps one block per sample)
    gn_split_t gs = {1, nullptr, nullptr};
    constexpr int MAXN = 4096, SCR = 1 << 17;                  // samples with a ticket counter; doubles of scratch
    int want = nst < 4096 ? 1 : nst / 512 < 32 ? nst / 512 : 32;          // (the ticket and the fold cost 2 - 3 us: a single pass is faster below a few thousand tiles)
    if (want * a.Go > 256) want = 256 / a.Go;
    while (want > 1 && (size_t)a.N * want * a.Go * 2 > (size_t)SCR) want >>= 1;
    if (want > 1 && a.N <= MAXN && !mi_ws_arena_on()) {
        static double *scr[8]; static unsigned *cnt[8];
        int dv = 0; MIRT(hipGetDevice(&dv)); dv &= 7;
        if (!scr[dv]) {
            MIRT(hipMalloc((void **)&scr[dv], (size_t)SCR * sizeof(double))); MIRT(hipMalloc((void **)&cnt[dv], MAXN * sizeof(unsigned))); mi_count_alloc(); mi_count_alloc();
            if (!scr[dv] || !cnt[dv]) mi_die("%s: no device memory for the statistics fold", who);
            MIRT(hipMemset(cnt[dv], 0, MAXN * sizeof(unsigned)));
        }
        gs.nsplit = want; gs.scr = scr[dv]; gs.cnt = cnt[dv];
    }
    // (one block per sample over more than a few hundred records: four times the threads, 2 002 records of 8 quads 10.4 -> 8.2 us, 1 232 of 16 7.9 -> 6.6; the split launches' blocks
    // are few rounds long already and lose by it, 7.3 -> 10.6)
    const float2 *part = (const float2 *)a.part;
    if (gs.nsplit == 1 && nst * Q > 8192) gn_part_reduce_k<1024><<<a.N, 1024>>>(part, tiles_per_n, a.ncs, MT, a.Co, a.Go, osum, fin, gs);
    else gn_part_reduce_k<256><<<a.N * gs.nsplit, 256>>>(part, tiles_per_n, a.ncs, MT, a.Co, a.Go, osum, fin, gs);
    MICK();
}

// the tap-packed stem (src/lp_f8fwd.cuh:601-609, :421-434): e4m3 compute, one activation scale per staged tile
// rows: the 9 .. 16 channel form, two taps per K block and one activation scale per staged row (src/lp_f8fwd.cuh:447-563, :626)
static thread_local int g_stem_zc = 0;      // tuning knob (mi_conv_stem_zc): z tiles per workgroup of the tap-packed kernel, 0 = chosen from the launch size
static int conv_stem(const char *who, const void *x, int xbf, shape5 xs, const float *w, const float *b, int cout, void *y, int ybf,
                     gnp_t gp, double *osum, int Go, split_t sp, bool rows) {
    const int Ci = xs.c, N = xs.n, D = sp.Di ? sp.Di : xs.d, Do = xs.d, H = xs.h, W = xs.w;      // D: the input's depth (z-range), Do: output planes
    if (gp.G && gp.ns && (gp.zs <= 0 || gp.zo < 0 || gp.zo >= gp.zs || gp.zhw != H * W || gp.ns > 256))
        mi_die("%s: slab-local GroupNorm geometry (zs %d, zo %d, ns %d, zhw %d) does not fit planes of %d voxels (at most 256 slabs)", who, gp.zs, gp.zo, gp.ns, gp.zhw, H * W);
    const int CP = rows ? 0 : Ci <= 4 ? 4 : Ci <= 8 ? 8 : 16, TPK = rows ? 2 : 32 / CP, NKB = rows ? 18 : (27 + TPK - 1) / TPK, NP = (NKB + 1) / 2;
    conv_args a; memset(&a, 0, sizeof a);
    a.wrec = 1;
    a.sx = x; a.sxdt = xbf; a.sCi = Ci;
    a.sgam = gp.gamma; a.sbet = gp.beta; a.smean = gp.mean; a.srstd = gp.rstd; a.sG = gp.G;
    if (gp.G && gp.ns) { a.szs = gp.zs; a.szo = gp.zo; a.sns = gp.ns; }      // (each slab's coefficient table in LDS: the staged positions take their plane's)
    a.N = N; a.D = D; a.H = H; a.W = W; a.Do = Do; a.Ho = H; a.Wo = W;
    a.zi0 = sp.Di ? sp.zi0 : 0; a.yD = sp.yD; a.yzo = sp.yD ? sp.yzo : 0;
    a.bias = b; a.Co = cout; a.y = y; a.ydt = ybf;
    a.osum = osum; a.Go = Go; a.stored_stats = sp.stored_stats && ybf >= 3; a.zs0 = sp.zlo; a.zs1 = Do - sp.zhi;
    // (16 channels per slot: 7 or 9 weight fragment pairs per channel tile, one tile fits the registers; per-channel statistics records: one tile per workgroup)
    const int nmt_all = (cout + 31) / 32, MT = nmt_all % 2 == 0 && CP && CP < 16 && !(osum && (cout / Go) % 4) ? 2 : 1;
    size_t smem = rows ? (size_t)720 * 16 + 16 + 40 * 4 + 16 * 8 : ((size_t)720 * CP + 16 + CP * 8 + 15) & ~(size_t)15;     // staged tile, (zero row, row words | amax word), channel affine
    if (a.sns > 1) smem += (size_t)(a.sns - 1) * (rows ? 16 : CP) * 8;      // (one affine table per slab)
    a.epi_o = (unsigned)smem; smem += (size_t)3 * MT * 32 * sizeof(float);
    a.red_o = (unsigned)smem; smem += 1024;
    a.nmt_all = nmt_all; a.ncs = nmt_all / MT;
    a.ntx = (W + 15) / 16; a.nty = (H + 7) / 8; a.ntz = (Do + 1) / 2;
    a.ntiles = (unsigned)((size_t)a.ntx * a.nty * a.ntz * a.ncs * N);
    // z tiles per workgroup (tap-packed kernel: the set-up is amortised, the next tile's loads overlap): up to 8 while >= 8 workgroups per CU remain
    a.zc = 1;
    if (!rows && CP <= 4 && g_stem_zc > 0) a.zc = g_stem_zc < a.ntz ? g_stem_zc : a.ntz;
    else if (!rows && CP <= 4) { a.zc = 8; while (a.zc > 1 && (size_t)a.ntx * a.nty * ((a.ntz + a.zc - 1) / a.zc) * a.ncs * N < 2048) a.zc--; }
    a.ngrp = (unsigned)((size_t)a.ntx * a.nty * ((a.ntz + a.zc - 1) / a.zc) * a.ncs * N);
    const size_t wq_bytes = (size_t)NP * nmt_all * 2048, wsc_bytes = (size_t)NP * nmt_all * 256;
    int dev = 0; MIRT(hipGetDevice(&dev));
    uint8_t *wq = nullptr, *wsc = nullptr; bool have = false;
    if (sp.wkey && !mi_ws_arena_on()) {                // memo entries of this layout: nbt = -CP (the entry point that must not allocate prepares per call)
        std::lock_guard<std::mutex> lk(g_wmemo_mu);
        for (auto &m : g_wmemo)
            if (m.key == sp.wkey && m.w == w && m.fmt == 8 && m.Co == cout && m.Ci == Ci && m.nbt == -CP - 1 && m.nmt_all == nmt_all && m.dev == dev) { wq = m.wq; wsc = m.wsc; have = true; break; }
        if (!have) {
            MIRT(hipMalloc((void **)&wq, wq_bytes)); MIRT(hipMalloc((void **)&wsc, wsc_bytes)); mi_count_alloc(); mi_count_alloc();
            if (!wq || !wsc) mi_die("%s: no device memory for the prepared weights", who);
            g_wmemo.push_back(wmemo_t{sp.wkey, w, 8, cout, Ci, Ci, -CP - 1, 0, nmt_all, dev, 0, wq, wsc});
        }
    } else { wq = (uint8_t *)mi_ws(MI_WS_WQ, wq_bytes); wsc = (uint8_t *)mi_ws(MI_WS_WSC, wsc_bytes); }
    if (!have) conv3_stem_prep(CP, w, wq, wsc, cout, Ci, nmt_all, NP);
    a.wq = wq; a.wsc = wsc;
    a.stat_ch = osum && (cout / Go) % 4 ? 1 : 0;
    if (osum) a.part = (float *)mi_ws(MI_WS_MISC, (size_t)a.ntiles * (a.stat_ch ? 32 : a.wrec * MT * 8) * 2 * sizeof(float));
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    const bool ktime = g_ktime && !mi_ws_arena_on();
    if (ktime) { MIRT(hipEventCreate(&ev0)); MIRT(hipEventCreate(&ev1)); MIRT(hipEventRecord(ev0, 0)); }
    conv3_stem_launch(CP, MT, ybf == 3 ? 8 : ybf == 4 ? 4 : 0, a, smem);
    if (ktime) { MIRT(hipEventRecord(ev1, 0)); ktime_push(ev0, ev1, 2.0 * 27 * Ci * (double)cout * N * Do * H * W); }
    if (osum) conv_stats_reduce(who, a, MT, sp, osum);
    return 0;
}

static thread_local const uint8_t *g_static_zpage = nullptr;     // the constant page of the calling thread's conv when it runs on the fixed scratch
static thread_local int g_split = -1;       // mi_conv_split: the calling thread's tile count below which 128-channel slices are halved (-1: the default)
extern "C" void mi_conv_split(int tiles) { g_split = tiles; }
// storage format of the calling thread's next split conv's second segment when it differs from the first's (3 MX-fp8, 4 MX-fp4; the descriptor
// carries one format for both); 0 = the same
static thread_local int g_x2_dt = 0;
// the calling thread's next split conv reads its upsampled segment as the e4m3 rows its pre-pass would make of it (MX-fp8, a multiple of 32 channels, no GroupNorm)
static thread_local bool g_up_staged = false;
extern "C" void mi_conv_up_staged(int on) { g_up_staged = on != 0; }
extern "C" void mi_conv_x2_dt(int dt) { g_x2_dt = dt == 3 || dt == 4 ? dt : 0; }
// both belong to one call of a conv entry and are taken at its start, also where it refuses or has nothing to do: none is left for a later call
struct conv_once_t { int x2_dt; bool up_staged; };
static conv_once_t take_once(void) { const conv_once_t o = {g_x2_dt, g_up_staged}; g_x2_dt = 0; g_up_staged = false; return o; }
static thread_local int g_s2d = -1;         // mi_conv_s2_direct: the calling thread's choice of stride-2 kernel (-1: by launch size)
extern "C" void mi_conv_s2_direct(int mode) { g_s2d = mode; }
static thread_local int g_thin = -1;        // mi_conv_thin: the calling thread's tile count up to which the K-split kernel takes a launch (-1: the default rule)
extern "C" void mi_conv_thin(int tiles) { g_thin = tiles; }
static thread_local int g_flat = -1;        // mi_conv_flat: whether the calling thread's convs run on the flat kernel wherever it can (1), nowhere (0), or by size (-1)
extern "C" void mi_conv_flat(int mode) { g_flat = mode; }
static thread_local bool g_records = false;  // mi_conv_keep_records: the calling thread's convs with statistics keep to the kernels whose records a network's logits were made with
extern "C" int mi_conv_keep_records(int on) { const int was = g_records; g_records = on != 0; return was; }
static int split_s2_env() { static int v = -1; if (v < 0) v = getenv("MI_CONV_SPLIT_S2") ? atoi(getenv("MI_CONV_SPLIT_S2")) : 1; return v; }      // tuning knob: 0 keeps four channel tiles
static int conv_dispatch(const char *who, int fmt, int stride, const void *x, int xbf, shape5 xs, const float *w, const float *b, int cout, void *y, int ybf,
                         gnp_t gp, double *osum, int Go, split_t sp, const float *ep_a, const float *ep_b, int act) {
    const conv_once_t once = take_once();
    if (sp.y2 || sp.o_split || sp.accum || sp.sr || sp.osr || sp.o_pad || sp.zw0 || sp.zw1)
        mi_die("%s: split outputs, accumulate, stochastic rounding and the z-window fields of split_t are not built here (inference forward only)", who);
    // z-range (src/nn_lp.h:36-40, src/nn_bwd.cu:33-36): the xs.d output planes read input plane z + zi0 of depth-Di inputs; direct slab output:
    // the MX output is planes [yzo, yzo + xs.d) of a depth-yD tensor
    if ((sp.Di || sp.zi0) && (stride != 1 || sp.zi0 < 0 || sp.zi0 + xs.d > sp.Di)) mi_die("%s: z-range %d + %d of depth %d (stride %d)", who, sp.zi0, xs.d, sp.Di, stride);
    if ((sp.yD || sp.yzo) && (stride != 1 || sp.yzo < 0 || sp.yzo + xs.d > sp.yD)) mi_die("%s: slab output %d + %d of depth %d (stride %d)", who, sp.yzo, xs.d, sp.yD, stride);
    // slab-local GroupNorm statistics (gnp_t.ns > 0, src/nn_lp.h:15-18): every GroupNorm + SiLU of a conv input is applied by the re-staging pass
    // below, which runs once per slab the launch's input planes meet; the kernels never see statistics
    if (gp.ns && sp.up) mi_die("%s: slab-local GroupNorm statistics on the upsampled segment are not supported (the skip segment's are)", who);
    // the op layer's masks and z-window (the reference's kernels ask the same before a launch: src/lp_f4fwd.cuh:1134-1223, src/nn_bwd.cu:89)
    { int za = 0, zb = 0; if (zw_win(xs.d, &za, &zb)) mi_die("%s: a z-window [%d, %d) is set; windows are not built here (inference forward only)", who, za, zb); }
    if (lp_skip_get(xs, sp, 1).m || nn_skip_masks(xs, sp)) mi_die("%s: the op layer asks for a masked (skip-empty) conv, which is not built here", who);
    if (xbf < 0 || xbf > 4 || !(ybf == 0 || ybf == 2 || ybf == 3 || ybf == 4)) mi_die("%s: unsupported storage types (in %d, out %d)", who, xbf, ybf);
    if (xs.n <= 0 || xs.c <= 0 || xs.d <= 0 || xs.h <= 0 || xs.w <= 0 || cout <= 0) return 0;
    const int Ci = xs.c, Cx = sp.x2 ? sp.c_split : Ci, C2 = Ci - Cx;
    const int entry_fmt = fmt;
    if (fmt == 4 && Ci <= 8) fmt = 8;                  // the network input computes in e4m3 whatever the activations' format (src/lp_f4fwd.cu:37)
    if (sp.x2 && (Cx <= 0 || C2 <= 0)) mi_die("%s: channel split %d of %d", who, sp.c_split, Ci);
    if (sp.x2 && xbf < 3) mi_die("%s: split inputs need MX storage", who);
    if (sp.up && (!sp.x2 || xbf < 3 || ((sp.Di ? sp.Di : xs.d) & 1) || (xs.h & 1) || (xs.w & 1) || stride != 1)) mi_die("%s: the fused upsample needs an MX split input and even dims", who);
    // (rows that are not what mi_restage_up_rows reads, 33 bytes each, would be read past their end; a GroupNorm on them would be one too many)
    if (once.up_staged && sp.up && (xbf != 3 || Cx % 32 || gp.G)) mi_die("%s: mi_conv_up_staged needs an MX-fp8 first segment of a multiple of 32 channels with no GroupNorm (storage %d, %d channels, %d groups)", who, xbf, Cx, gp.G);
    if (osum && (Go <= 0 || cout % Go)) mi_die("%s: %d output channels in %d groups", who, cout, Go);
    if (gp.G > 0 && ((sp.x2 && sp.gp2.G ? Cx : Ci) % gp.G)) mi_die("%s: GroupNorm groups %d do not divide the channels", who, gp.G);
    if (sp.gp2.G > 0 && (!sp.x2 || C2 % sp.gp2.G)) mi_die("%s: second GroupNorm without a matching x2 segment", who);
    // few input channels: the tap-packed kernel with one activation scale per tile (src/lp_f8fwd.cuh:601-609: up to 8 channels of a 16-bit or
    // MX input, 16 of an fp32 one; same input and output type, or an MX output)
    static int stem_env = -1;
    if (stem_env < 0) stem_env = getenv("MI_CONV_STEM") ? atoi(getenv("MI_CONV_STEM")) : 1;     // tuning knob: 0 sends these convs to the general kernel
    if (stem_env && fmt == 8 && stride == 1 && !sp.x2 && !act && (xbf == 0 || xbf >= 2) && Ci <= (xbf == 0 ? 16 : 8) && (xbf == ybf || ybf >= 3))
        return conv_stem(who, x, xbf, xs, w, b, cout, y, ybf, gp, osum, Go, sp, false);
    // 9 .. 16 channels of an MX or fp16 input: two taps per K block, one activation scale per staged row (src/lp_f8fwd.cuh:626)
    if (stem_env && fmt == 8 && stride == 1 && !sp.x2 && !act && xbf >= 2 && Ci <= 16 && (xbf == ybf || ybf >= 3))
        return conv_stem(who, x, xbf, xs, w, b, cout, y, ybf, gp, osum, Go, sp, true);
    const int N = xs.n, D = sp.Di ? sp.Di : xs.d, H = xs.h, W = xs.w;           // D: the inputs' depth
    const int Do = stride == 2 ? (D - 1) / 2 + 1 : xs.d, Ho = stride == 2 ? (H - 1) / 2 + 1 : H, Wo = stride == 2 ? (W - 1) / 2 + 1 : W;   // src/nn_bwd.cu:132-135
    // output planes of the whole tensor, of which a z-range computes Do: whatever decides in which order a conv adds, and over which voxels its statistics
    // records run, is chosen by these, so that a slab gives the whole tensor's bytes. The price is that a slab of few tiles may not take the form that would
    // be the fastest for it: 128 -> 128 on 32^3 in slabs of 8 planes 122 us on the wide kernel, 88 on the coarse form; 192 -> 64 in slabs of 4 310 on the wide
    // kernel, 113 on the K-split one
    const int Dr = stride == 1 ? D : Do;
    const size_t S = (size_t)D * H * W;
    const int zlo = sp.Di ? (sp.zi0 > 0 ? sp.zi0 - 1 : 0) : 0, zhi = sp.Di ? (sp.zi0 + xs.d + 1 < D ? sp.zi0 + xs.d + 1 : D) : D;      // input planes this launch reads
    const int fdt = fmt == 8 ? 3 : 4;
    conv_args a; memset(&a, 0, sizeof a);
    // ---- operands: a segment is read as stored when it already is the compute format with nothing to apply, else re-staged once ----
    // (gp2.G < 0, an extension: x2 carries no GroupNorm and gp is x's own; the reference's gp2.G == 0 means gp spans both segments)
    const bool s2g = sp.x2 && sp.gp2.G;
    if (sp.gp2.G < 0) sp.gp2 = gnp_mk(nullptr, nullptr, nullptr, nullptr, 0);
    const void *segx[2] = {x, sp.x2}; const int segC[2] = {Cx, C2};
    const int segbf[2] = {xbf, sp.x2 && once.x2_dt ? once.x2_dt : xbf};
    for (int s = 0; s < (sp.x2 ? 2 : 1); s++) {
        const gnp_t g = s2g ? (s ? sp.gp2 : gp) : gp;
        const int Cg = s2g ? segC[s] : Ci, cg0 = s2g ? 0 : (s ? Cx : 0);
        const bool upseg = s == 0 && sp.up;
        const int xbf = segbf[s];                                 // (this segment's storage format)
        const bool direct = xbf == fdt && !g.G && !upseg;
        const int nbp = (segC[s] + 31) / 32;
        if (direct) {
            const int bw = mx_bw(segC[s]), nb = mx_nb(segC[s]);
            a.xq[s] = (const uint8_t *)segx[s]; a.xsc[s] = a.xq[s] + (size_t)N * nb * S * mx_rb(bw, fmt);
            a.nbs[s] = nb; a.bws[s] = bw;
        } else {
            const size_t bytes = (size_t)N * nbp * S * (mx_rb(32, fmt) + 1);
            uint8_t *st = (uint8_t *)mi_ws(s ? MI_WS_X2STAGE : MI_WS_XSTAGE, bytes);
            // the fp4 entry blends the upsample in binary16 unless UFSM_UP_H2=0 (src/lp_f4fwd.cuh:1135-1136); sp.up 2 / 3 force one blend
            static int uph2 = -1;
            if (uph2 < 0) uph2 = getenv("UFSM_UP_H2") ? atoi(getenv("UFSM_UP_H2")) : 1;
            if (upseg && once.up_staged) mi_restage_up_rows(segx[s], N, segC[s], D, H, W, st, fmt, zlo, zhi, sp.up == 2 || (sp.up == 1 && entry_fmt == 4 && uph2));
            else if (upseg) mi_restage_up_sub(segx[s], xbf, N, segC[s], D, H, W, g, Cg, st, fmt, zlo, zhi, sp.up == 2 || (sp.up == 1 && entry_fmt == 4 && uph2));
            else gn_for_slabs(who, g, H * W, zlo, zhi, [&](int z0, int z1, gnp_t gs) { mi_restage_sub(segx[s], xbf, N, segC[s], (size_t)(z1 - z0) * H * W, gs, Cg, cg0, st, fmt, S, (size_t)z0 * H * W); });
            a.xq[s] = st; a.xsc[s] = st + (size_t)N * nbp * S * mx_rb(32, fmt);
            a.nbs[s] = nbp; a.bws[s] = 32;
        }
        if (s == 0) a.nb0p = nbp;
    }
    a.nbt = a.nb0p + (sp.x2 ? (C2 + 31) / 32 : 0);
    a.wide = a.bws[0] == 32 && (!sp.x2 || a.bws[1] == 32);
    a.N = N; a.D = D; a.H = H; a.W = W; a.Do = Do; a.Ho = Ho; a.Wo = Wo;
    a.zi0 = sp.Di ? sp.zi0 : 0; a.yD = sp.yD; a.yzo = sp.yD ? sp.yzo : 0;
    a.bias = b; a.Co = cout; a.y = y; a.ydt = ybf;
    a.osum = osum; a.Go = Go; a.stored_stats = sp.stored_stats && ybf >= 3; a.zs0 = sp.zlo < Do ? sp.zlo : Do; a.zs1 = sp.zhi < Do ? Do - sp.zhi : 0;      // (within the planes there are: some kernels count in voxels)
    a.ep_a = ep_a; a.ep_b = ep_b; a.act = act;
    // ---- tile shape: MT channel tiles of 32 per workgroup, NT voxel tiles of 32 per wavefront, MT * NT <= 8 accumulators ----
    const int nmt_all = (cout + 31) / 32;
    int MT = nmt_all <= 4 ? nmt_all : nmt_all % 4 == 0 ? 4 : nmt_all % 3 == 0 ? 3 : nmt_all % 2 == 0 ? 2 : 1;
    // channels per group not a multiple of 4 (80 channels in 8 groups): the statistics are per-channel records of one channel tile per workgroup
    if (osum && (cout / Go) % 4) MT = 1;
    bool halved = false, halved_whole = false;
    {   // few tiles of 128 channels (the coarse levels): slices of 64 channels double the workgroups of the wide kernel
        static int split_env = -1;
        if (split_env < 0) split_env = getenv("MI_CONV_SPLIT") ? atoi(getenv("MI_CONV_SPLIT")) : 192;    // tuning knob: tile count below which the slices are halved (0: never)
        const int split = g_split >= 0 ? g_split : split_env;
        // (a z-range's own tiles count where the wide kernel takes the launch, whose slices of either width add alike; the general kernel's do not)
        auto few = [&](int d) { return (size_t)((Wo + 15) / 16) * ((Ho + 7) / 8) * ((d + 3) / 4) * (nmt_all / 4) * N < (size_t)split; };
        if (stride == 1 && MT == 4 && nmt_all % 4 == 0 && Dr >= 3) {
            halved_whole = few(Dr);
            halved = few(a.wide && a.nbt <= 12 ? Do : Dr);
            if (halved) MT = 2;
        }
    }
    int NT = (stride == 1 && MT <= 2 && Dr >= 4) ? 4 : 2;
    // ... and when even the slices of 64 give fewer than 128 workgroups (256 -> 256 at 2 x 16^3: 64): one channel tile and two planes per workgroup
    // on the general kernel, four times the workgroups (measured in the 32/64/128/256 forward: 128 -> 256 0.032 -> 0.026 ms, 256 -> 256
    // 0.050 -> 0.038 ms; from 256 slices of 64 on, the wide kernel is the faster one: 128 -> 128 at 2 x 32^3 0.034 against 0.052 ms)
    bool coarse = false;
    {
        static int ce = -1;
        if (ce < 0) ce = getenv("MI_CONV_COARSE") ? atoi(getenv("MI_CONV_COARSE")) : 1;      // tuning knob: 0 keeps the wide kernel's slices of 64 there (as does a split forced through mi_conv_split)
        if (ce && halved_whole && g_split < 0 && (size_t)((Wo + 15) / 16) * ((Ho + 7) / 8) * ((Dr + 3) / 4) * (nmt_all / 2) * N < 128) { coarse = true; NT = 2; MT = 1; halved = false; }
    }
    // stride 2 with few tiles (the coarse levels): one-plane tiles double the workgroups; with enough tiles the two-plane tile is faster
    // (measured: 128 -> 128 at 32^3 -> 16^3, N 2: 32 tiles 0.072 ms, 64 tiles 0.042 ms; 32 -> 32 at 128^3: 0.090 vs 0.120 ms)
    if (stride == 2 && (MT == 1 || MT == 2 || MT == 4) &&
        (size_t)((Wo + 15) / 16) * ((Ho + 7) / 8) * ((Do + 1) / 2) * (nmt_all / MT) * N < 256) NT = 1;
    // ... and still fewer one-plane tiles than half the CUs: two channel tiles per workgroup instead of four
    if (stride == 2 && MT == 4 && NT == 1 && split_s2_env() && (size_t)((Wo + 15) / 16) * ((Ho + 7) / 8) * Do * (nmt_all / 4) * N < 128) MT = 2;
    // ... and one while two would still leave CUs idle (128 -> 128 from 2 x 32^3: 128 workgroups 0.035 ms, 256 workgroups 0.024 ms; the two-plane
    // tiles of 64 -> 64 from 2 x 64^3, 256 workgroups, are the fastest form there: 0.030 ms against 0.039 with 512 one-plane tiles)
    if (stride == 2 && MT == 2 && NT == 1 && split_s2_env() && (size_t)((Wo + 15) / 16) * ((Ho + 7) / 8) * Do * (nmt_all / 2) * N < 256) MT = 1;
    // stride 2 on 32-channel rows with enough output voxels (four workgroups per CU or more): the kernel that reads every tap's rows straight from
    // the stored tensor (no staged halo). Measured in the 32/64/128/256 forward at 2 x 128^3: 32 -> 32 from 128^3 0.093 -> 0.071 ms; 64 -> 64 from
    // 64^3 is slower there, 0.030 -> 0.037 ms, and stays with the general kernel. Runs of 64 output voxels per wavefront; channel tiles per
    // workgroup halved while fewer than two workgroups per CU would run
    static int s2d_env = -1;
    if (s2d_env < 0) s2d_env = getenv("MI_CONV_S2D") ? atoi(getenv("MI_CONV_S2D")) : 8;       // tuning knob: 0 keeps the general kernel for stride 2, else the launch size (in units of 128 workgroups of 256 output voxels) from which the direct kernel runs
    const size_t s2runs = ((size_t)Do * Ho * Wo + 63) / 64;
    // (by default only one input block and one channel tile, the shape it is measured faster on: 64 -> 64 takes 0.034 against 0.030 ms from 2 x 64^3
    // and 0.36 against 0.09 ms from 8 x 64^3)
    // ... on rows of more than 16 output voxels the row kernel does: the tile's rows staged in LDS as they lie in memory, the weights in registers. us of the conv by itself, general / direct / row kernel,
    // e4m3: 2 x 128^3 85.8 / 59.0 / 43.6, 9 x 128^3 364 / 278 / 170, 88 x 104^2 30.8 / 19.1 / 13.8, 64^3 8.3 / 12.6 / 7.5; e2m1: 128^3 19.7 / 28.1 / 15.9, 2 x 96^3 17.0 / 28.0 / 16.4, 48^3 6.6 / 12.5 / 6.3. On rows of
    // 16 and fewer half its lanes idle (4 x 64^2 x 32: 10.8 general, 13.7); up to 256 tiles of the K-split kernel e4m3 stays there (48^3 7.2 / 7.8 here, 32 x 64^2 7.4 / 7.7)
    static int s2row_env = -1;
    if (s2row_env < 0) s2row_env = getenv("MI_CONV_S2ROW") ? atoi(getenv("MI_CONV_S2ROW")) : 1;      // tuning knob: 0 never
    a.s2row = stride == 2 && a.nbt == 1 && nmt_all == 1 && cout > 16 && a.wide && !act && S < ((size_t)1 << 31) && (size_t)((Wo + 31) / 32) * ((Ho + 3) / 4) * Do * N < ((size_t)1 << 31) &&
              (g_s2d == 2 || (g_s2d < 0 && s2row_env && Wo > 16 && (fmt == 4 || s2runs * N > 256)));
    const bool s2d = a.s2row || (s2d_env && g_s2d != 0 && stride == 2 && a.wide && !act && N <= 65535 &&
                     (g_s2d > 0 || (a.nbt == 1 && nmt_all == 1 && (s2runs + 3) / 4 * N >= (size_t)s2d_env * 128)));
    if (s2d) {
        MT = nmt_all % 4 == 0 ? 4 : nmt_all % 2 == 0 ? 2 : 1;
        while (MT > 1 && (s2runs + 3) / 4 * (size_t)(nmt_all / MT) * N < 512) MT >>= 1;
        NT = 2;
    }
    // 128-channel output slices at stride 1 take the wide kernel (16 accumulators per wavefront, one workgroup per CU)
    static int big_env = -1;
    if (big_env < 0) big_env = getenv("MI_CONV_WIDE") ? atoi(getenv("MI_CONV_WIDE")) : 1;      // tuning knob: 0 keeps the 8-accumulator kernel, 2 sends every 64-channel layer to the wide kernel too
    // (64 output channels: two channel tiles per workgroup; it pays from four input blocks on: 192 -> 64 at 2 x 64^3 0.190 -> 0.178 ms, 64 -> 64 the same
    // as the general kernel. MI_CONV_WIDE=2 sends every such layer there)
    static int rowcs4_env = -1;
    if (rowcs4_env < 0) rowcs4_env = getenv("MI_CONV_ROW_CS4") ? atoi(getenv("MI_CONV_ROW_CS4")) : 1;      // tuning knob: input blocks up to which 65 .. 128 output channels run the row kernels as three or four slices (0: never).
    // Measured: 32 -> 128 at 2 x 64^3 0.079 -> 0.064 ms on the one-block kernel; from two blocks on the wide kernel is as fast (64 -> 128 and 128 -> 128 at 2 x 32^3)
    // or faster (e2m1 at 32 x 32^3: 0.151 against 0.164 ms), hence 1
    const bool row_cs4 = rowcs4_env > 0 && g_split < 0 && (nmt_all == 3 || nmt_all == 4) && a.nbt <= rowcs4_env && stride == 1 && !coarse && a.wide && Wo > 16 && Dr >= 4 && !(osum && (cout / Go) % 4);
    if (row_cs4) { MT = 1; NT = 4; halved = false; }
    bool big = !row_cs4 && !coarse && big_env && stride == 1 && (MT == 4 || (MT == 2 && (big_env > 1 || a.nbt >= 4 || halved))) && Dr >= 3 && a.wide && a.nbt <= 12;            // (its per-tile pair table must fit LDS)
    if (big) {
        // The wide kernel streams input block b >= 2 of a tile into LDS while the tile's earlier blocks are multiplied, one copy round per
        // stage of two pairs, NRND rounds per block, a block starting once block b - 3 has been read for the last time (pair (27 (b - 3) + 26) / 2).
        // A round issued in stage s is visible two barriers later. Check that every block lands before the step that first fetches from it.
        const int NRND = ((6 * 10 * 18 + 63) / 64 + 3) / 4, npairs = (27 * a.nbt + 1) >> 1, nfull = npairs >> 1;
        int fbi = 2, frd = 0;
        for (int s = 0; s < nfull && big; s++) {
            if (fbi < a.nbt && (fbi < 3 || ((27 * (fbi - 3) + 26) >> 1) <= 2 * s + 1) && ++frd == NRND) {
                const int pf = ((27 * fbi) >> 1) - 1;               // the pair during which the block's first fragments are fetched
                const int need = pf & 1 ? (pf >> 1) - 2 : (pf >> 1) - 3;
                if (s > need) big = false;
                frd = 0; fbi++;
            }
        }
        if (fbi < a.nbt) big = false;
    }
    if (big) NT = 4;
    const int TZ = NT == 1 ? 1 : NT == 2 ? 2 : 4;
    const int HZ = stride * (TZ - 1) + 3, HY = stride * 7 + 3, HX = stride * 15 + 3, TT = HZ * HY * HX;
    const int RB = fmt == 8 ? 32 : 16, WTILE = fmt == 8 ? 2048 : 1024;
    // LDS of a workgroup holding CB input blocks: weight ring, pair table, halo rows and scale words. Prefer the largest CB that
    // still lets two workgroups share a CU (160 KB): the second one computes while the first stages its halo or runs its epilogue.
    // The wide kernel has a fixed layout: ring of two slots of two pairs, three halo slots of one block, two pair tables.
    auto lds_of = [&](int mt, int cb) { return (size_t)2 * (mt == 1 ? 7 : mt == 2 ? 2 : 1) * mt * (WTILE + 256) + (size_t)(((27 * cb + 1) >> 1) + 2) * 32 + (size_t)cb * TT * (RB + 4); };      // (a ring stage of the general kernel: 7, 2 or 1 pairs)
    int cb1 = 0;
    auto cb_of = [&](int mt) {
        int cb2 = 0; cb1 = 0;
        for (int cb = 1; cb <= a.nbt; cb++) { if (lds_of(mt, cb) <= 80 * 1024 - 2816) cb2 = cb; if (lds_of(mt, cb) <= 160 * 1024 - 3072) cb1 = cb; }   // (room for the epilogue's constants and scratch)
        return cb2 ? cb2 : cb1;
    };
    // Three channel tiles per workgroup (96, 192 channels) on fewer than 192 workgroups: a tile each, three times the workgroups, if its chunks of input blocks - the order of K - stay
    // what they are (e2m1; the e4m3 ring leaves room for fewer blocks). The records are a tile's, quad by quad, either way. A 192 -> 192 conv by itself, e2m1, us, three tiles / one per
    // workgroup: 16 x 24 x 26 into 96 channels (32 workgroups of three) 37.3 / 20.7, 32 x 24 x 26 (64) 38.0 / 25.1, 7 x 16^3 (224) 37.3 / 37.9, 9 x 16^3 (288) 40.8 / 42.4, 12 x 16^3 (384)
    // 41.2 / 55.3; in the two deep convs of a 192-channel network at 2 x 128^3 (64) 45 + 62 -> 16 + 19
    static int split3_env = -1;
    if (split3_env < 0) split3_env = getenv("MI_CONV_SPLIT3") ? atoi(getenv("MI_CONV_SPLIT3")) : 192;      // tuning knob: that workgroup count (0: never)
    a.one3 = stride == 1 && !big && MT == 3 && NT == 2 && !(osum && (cout / Go) % 4) && (size_t)((Wo + 15) / 16) * ((Ho + 7) / 8) * ((Do + 1) / 2) * (nmt_all / 3) * N < (size_t)split3_env && (a.nbt + cb_of(3) - 1) / cb_of(3) == (a.nbt + cb_of(1) - 1) / cb_of(1);
    if (a.one3) MT = 1;
    int cbmax = cb_of(MT);
    auto lds_bytes = [&](int cb) { return lds_of(MT, cb); };
    static int cb_env = -1;
    if (cb_env < 0) cb_env = getenv("MI_CONV_CB") ? atoi(getenv("MI_CONV_CB")) : 0;      // tuning knob: blocks per chunk
    if (cb_env > 0 && cb_env <= cb1) cbmax = cb_env;
    if (cbmax < 1) mi_die("%s: tile does not fit LDS", who);
    const int nchunks = (a.nbt + cbmax - 1) / cbmax;
    a.CB = big || s2d ? a.nbt : (a.nbt + nchunks - 1) / nchunks; // (the wide kernel has no chunks: its K loop walks block by block; the direct stride-2 kernel: one chunk, tap-major)
    static int areg_env = -1;
    if (areg_env < 0) areg_env = getenv("MI_CONV_AREG") ? atoi(getenv("MI_CONV_AREG")) : 1;      // tuning knob: 0 keeps the general kernel for every shape
    a.areg = areg_env && !big && !s2d && !(osum && (cout / Go) % 4) && cout > 16 && nmt_all == 1 && stride == 1 && a.nbt == 1 && a.wide && (NT == 2 || NT == 4);      // (one channel tile in all: these kernels have no channel slices)
    // one channel tile of 17 .. 32 output channels from two or more input blocks on a volume wider than one 16-voxel tile: the row kernel (runs
    // of 32 voxels along x, input fragments shared by the three ky taps). One input block stays with the kernel that keeps its weights in
    // registers, which measures a few percent faster there (both are bound by the halo's cache misses in flight, and it loads no weights)
    static int row_env = -1;
    if (row_env < 0) row_env = getenv("MI_CONV_ROW") ? atoi(getenv("MI_CONV_ROW")) : 1;      // tuning knob: 0 keeps the other kernels for these shapes, 2 also takes one input block
    // ... and one input block takes the row kernel's one-block form: weights in registers, the workgroup's two halves half a tile apart so that
    // one half's epilogue runs under the other's MFMAs (MI_CONV_ROW1=0: the small-channel kernel)
    static int row1_env = -1;
    if (row1_env < 0) row1_env = getenv("MI_CONV_ROW1") ? atoi(getenv("MI_CONV_ROW1")) : 1;
    // ... and 33 .. 64 output channels from one to three input blocks run the two row kernels as two channel slices, one per workgroup (MI_CONV_ROW_CS=0:
    // the general kernel). Measured at 2 x 64^3 in e4m3: 32 -> 64 0.046 -> 0.039 ms, 64 -> 64 0.073 -> 0.067 ms, 96 -> 64 0.100 -> 0.095 ms; from four
    // blocks on the wide kernel keeps these layers
    static int rowcs_env = -1;
    if (rowcs_env < 0) rowcs_env = getenv("MI_CONV_ROW_CS") ? atoi(getenv("MI_CONV_ROW_CS")) : 1;
    const bool row_cs = (rowcs_env && nmt_all == 2 && MT == 2) || row_cs4;
    a.row = row_env && !big && !s2d && !(osum && (cout / Go) % 4) && cout > 16 && (nmt_all == 1 || row_cs) && stride == 1 && NT == 4 && a.wide && Wo > 16 && a.nbt >= (row_env > 1 || row1_env ? 1 : 2) && a.nbt <= 64;
    // ... but one channel tile from one block goes back to the small-channel kernel (two workgroups per CU, 16-wide tiles; a statistics record per wavefront, as the row kernel's, so that
    // the sums keep their precision) where the row kernel has fewer than four tiles per CU to walk (its ring of planes and its half-tile offset need a walk: 1 024 tiles) or where runs of 32
    // fit the rows worse than tiles of 16. A call with statistics, us, the row kernel against this one, e4m3: 16 x 32^2 14.1 / 10.6, 32^3 14.5 / 11.0, 48^3 16.9 / 12.5, 64^3 (256 row tiles)
    // 17.9 / 16.3, 2 x 64^3 (512) 24.3 / 23.4, 96^3 (864) 35.5 / 33.5; rows of 104 in 88 planes 42.3 / 37.7, of 72 (128 x 96 x 72) 41.9 / 37.0, of 112 (112^3) 52.8 / 46.5, of 80 (80^3)
    // 30.9 / 26.1. e2m1: 64^3 15.0 / 13.6, 96^3 28.5 / 26.4, 88 x 104^2 33.9 / 29.8. Past 1 024 tiles of whole runs the row kernel is the faster one (with a record per tile here: 64 x 128^2
    // 56.6 / 59.6, 4 x 64^3 55.6 / 57.3, 2 x 128^3 208 / 224, of a call that prepares its weights; rows of 120 - four runs of 32, eight tiles of 16 - 88.5 / 90.5). fp16 planes out: 64^3
    // 29.4 / 25.5, 40^3 22.7 / 16.8. Launches of under 16 384 voxels gain as well (24^3 17.7 / 13.3), but the tests hold two of them on the row kernel
    // A conv's products and its fp32 statistics records add up in another order on another kernel, which moves a mean or 1 / std by its last bit now and then; a code of the next conv's rows at a rounding
    // boundary then moves, and with it the rest of a network (e4m3: up to 2 % of the logits, one window size in ten; e2m1 more). Inside a network the three rules that came with the
    // flat kernel (this one, the short 96 -> 32 walks and the flat tiles) therefore leave convs with statistics where they were
    const bool rec = g_records && osum;
    const size_t row_tiles = (size_t)((Wo + 31) / 32) * ((Ho + 7) / 8) * ((Dr + 3) / 4) * N;
    const bool row_small = a.row && a.areg && row1_env == 1 && !rec && g_thin < 0 && (size_t)N * Dr * Ho * Wo >= 16384 && (row_tiles < 1024 || 2 * ((Wo + 31) / 32) > (Wo + 15) / 16);
    if (row_small) a.row = false;
    a.row1 = a.row && a.nbt == 1 && row1_env && row_env < 2;
    a.wrec = a.row1 ? 8 : row_small && osum ? 4 : 1;
    if (a.row && nmt_all >= 2) MT = 1;
    if (a.row) { a.areg = false; a.CB = a.nbt; }
    // few output voxels: the K range split over a workgroup's wavefronts (conv3_thin_k). The staged kernels' time hardly depends on how many workgroups a
    // launch has until every CU has one, this one's grows with its tiles (64 voxels x 32 channels) once each CU has one. Kernel time, us, the other kernel
    // against this one. e4m3, stride 1, 1 x 8^3 / 1 x 16^3 / 2 x 16^3: 64 -> 64 21.6 / 21.8 / 21.9 against 7.8 / 8.2 / 8.8 (16 / 128 / 256 tiles); 192 -> 64 35 / 35 / 36
    // against 11.4 / 12.6 / 13.0; 64 -> 128 12.9 / 13.0 / 12.9 against 8.0 / 9.7 / 14.4 (512 tiles); 128 -> 128 18.5 / 18.8 / 19.1 against 9.6 / 11.1 / 17.2 (512);
    // 256 -> 256 31 / 32 / 34 against 12.8 / 23.5 / 43.1 (1024); 384 -> 128 45 / 45 / 46 against 15.4 / 17.0 / 29.6 (512). e2m1: 64 -> 64 at 2 x 16^3 16.9 against 8.5.
    // Hence 256 tiles, and 512 from eight input blocks of e4m3 on. Stride 2, 32 -> 32 at
    // 16^3 8.6 against 7.0 and 64 -> 64 from 2 x 32^3 (256 tiles) 12.0 against 8.9; with eight blocks it depends on whether the general kernel's workgroups
    // fit the CUs at once: 256 -> 256 from 1 x 32^3 (512 tiles, 256 of its workgroups) 32.8 against 34.9, 256 -> 128 from 2 x 32^3 32.7 against 38.6, 256 -> 256 from
    // 2 x 24^3 (432 tiles, 384 of its workgroups) 60.6 against 33.4. Against the coarse form's one channel tile a short K gains little, and the statistics'
    // reduction reads more records: one block of e4m3 or two of e2m1 are even with it from 64 tiles on (both kernels of a call: e4m3 32 -> 256 at 1 x 4^3
    // 12.4 against 11.3, 1 x 8^3 (64 tiles) 12.5 and 12.4, 1 x 11 x 13^2 (240) 13.1 and 13.6; e2m1 64 -> 128 at 2 x 8^3 (64) 11.8 and 11.2, 1 x 12^3 (108) 12.1 and 13.1,
    // 1 x 16^3 (256) 12.2 and 12.1) and stop there. One block of e2m1 has fourteen pairs, too few to split: 32 -> 128 at 1 x 8^3 7.1 against 7.4, at stride 2
    // 32 -> 32 from 1 x 16^3 6.4 against 6.9; these keep the general kernel. The row
    // kernels' and the one-block, one-tile kernel's launches stay theirs. The tiles counted are the whole tensor's (Dr planes), not a z-range's: a slab
    // adds in the order of the whole tensor's conv and takes its statistics over the same runs, so that inference in slabs gives its bytes (a slab whose statistics
    // leave planes at its ends out, zlo and zhi, too)
    // (These figures are of the kernels as they were when the line was drawn. Both sides are faster since - the K-split kernel by 1 - 5 us a launch, the other one as conv3_pipe_k by a third, a call of
    // 384 -> 128 at 1 x 8^3 18.3 -> 12.8 and of 256 -> 256 at 2 x 16^3 38.9 -> 25.3 -, and the line stays: a conv on the other side of it adds its products in another order, which a network would notice)
    static int thin_env = -1;
    if (thin_env < 0) thin_env = getenv("MI_CONV_THIN") ? atoi(getenv("MI_CONV_THIN")) : 256;      // tuning knob: that tile count (0: never)
    const int kb = a.nbt * (fmt == 8 ? 2 : 1);                 // (K in bytes: halves of 16 per tap)
    const bool one_round = stride == 2 && (size_t)((Wo + 15) / 16) * ((Ho + 7) / 8) * ((Do + TZ - 1) / TZ) * (nmt_all / MT) * N <= 256;      // (the general kernel's workgroups)
    const size_t thin_max = g_thin >= 0 ? (size_t)g_thin : kb == 1 && (coarse || stride == 2) ? 0 : kb == 2 && coarse ? (size_t)thin_env / 4 : kb >= 16 && fmt == 8 && !one_round ? 2 * (size_t)thin_env : (size_t)thin_env;
    // ... except three input blocks and more into one channel tile, whose few tiles on the row kernel are one CU's latency each: 96 -> 32 at 24^3 (216 tiles) 24.0 / 13.6,
    // 28^3 (343) 23.9 / 16.6, 32^3 (512) 23.2 / 17.5; e2m1 at 24^3 18.5 / 11.3, at 32^3 18.8 / 16.1 and more records to add. (From 129 tiles on and with one channel tile only - 96 -> 64
    // at 24^3 24.4 / 16.4 -: the tests hold launches beyond that on the row kernel)
    // thin_ok: what the K-split kernel can take; a call it cannot - an activation, the thread's own choice of slices - stays on the row kernel
    const bool thin_ok = !s2d && !act && a.wide && cout > 16 && !(osum && (cout / Go) % 4) && g_split < 0 && (stride == 1 || g_s2d < 0) && N <= 65535 && (size_t)D * H * W * 32 < ((size_t)1 << 31);
    const size_t thin_tiles = ((size_t)Dr * Ho * Wo + 63) / 64 * (size_t)nmt_all * N;
    const bool thin_row = thin_ok && a.row && nmt_all == 1 && a.nbt >= 3 && !rec && g_thin < 0 && thin_tiles > 128 && thin_tiles <= (fmt == 8 ? 2 * (size_t)thin_env : (size_t)thin_env);
    if (thin_row) a.row = false;
    a.thin = thin_row || (thin_ok && !a.row && !a.areg && thin_tiles <= thin_max);
    // about one tile of 128 flat voxels x 64 channels per CU, past the K-split kernel's launches: the flat kernel, whose time goes by its rounds of 256 workgroups -
    // some 8 us and 2.2 (e2m1 1) per pair of input blocks each - where the staged kernels' goes by one tile's chain of loads and barriers. Kernel time, us, the other
    // kernel against this one, and workgroups here. e4m3: 256 -> 256 at 2 x 16^3 37.2 against 22.2 (256); at 1 x 22 x 26^2 (234) 64 -> 128 18.4 against 14.4, 128 -> 128 26.8 and
    // 16.5, 384 -> 128 62.9 and 26.5; 192 -> 64 at 24^3 38.4 and 18.2 (108), at 32^3 38.8 and 21.0 (256); 192 -> 192 at 16^3 47.1 and 18.2 (96); 64 -> 64 at 24^3 20.3 and 13.6 (108);
    // against the K-split kernel 256 -> 256 at 16^3 26.9 and 20.0 (128), with fewer than 257 of its tiles 192 -> 64 at 16 x 20^2 15.1 and 17.2 (its launches of 257 .. 512 tiles
    // into 128 channels gain as much, 256 -> 128 at 32 x 16^2 28.2 and 20.9, but its limit of 512 tiles is a tested one and stays). e2m1: 128 -> 192 and 192 -> 192
    // at 2 x 16^3 26.6 and 36.7 against 14.0 and 15.4 (192), 384 -> 128 at 2 x 16^3 31.9 and 20.2; with two blocks 64 -> 128 at 16^3 11.5 and 12.1. In two rounds a long K pays: e4m3
    // 256 -> 256 at 4 x 16^3 50.1 and 38.1 (512), 384 -> 128 at 28^3 63.6 and 44.8 (344), 128 -> 128 at 28^3 28.0 and 27.3; e2m1 384 -> 128 at 2 x 24^3 48.5 and 34.5 (432), 128 -> 128 25.1
    // and 23.4; in four it does not: 384 -> 128 at 2 x 32^3 75.4 and 90.9 (1024). A record per run of 32 voxels is four to eight times the staged kernels': past 512 a sample their
    // sums take a launch more (3 - 5 us), which e2m1's shorter products do not always win back: 256 -> 128 at 28^3 (686 runs) 33.1 against 37.7 with it. As above, the whole
    // tensor's voxels count, not a z-range's.
    // (Where the other kernel was the general one, that is of before conv3_pipe_k, which has closed much of the gap; a call with its statistics, us, conv3_pipe_k / this: e4m3 256 -> 256 at 2 x 16^3
    // 24.0 / 21.9, 64 -> 128 at 22 x 26^2 16.1 / 16.5, 128 -> 128 22.6 / 19.3, 384 -> 128 46.3 / 28.7, at 28^3 46.0 / 48.5; e2m1 128 -> 192 at 2 x 16^3 12.9 / 14.5, 192 -> 192 15.3 / 16.1, 384 -> 128
    // 21.6 / 19.7. The line stays where it was: the two add their products in different orders)
    static int flat_env = -1;
    if (flat_env < 0) flat_env = getenv("MI_CONV_FLAT") ? atoi(getenv("MI_CONV_FLAT")) : 1;      // tuning knob: 0 never
    const bool flat_ok = stride == 1 && a.wide && !act && nmt_all >= 2 && a.nbt % 2 == 0 && W <= flat_t<8>::WMAX && !(osum && (cout / Go) % 4) && N <= 65535 && (size_t)D * H * W < ((size_t)1 << 24) &&
                         ((size_t)27 * (a.nbt / 2) + 2) * nmt_all * WTILE < ((size_t)1 << 31);      // (its weight offsets are 32 bits)
    const size_t frun = ((size_t)Dr * Ho * Wo + 31) / 32, fwg = (frun + 3) / 4 * (size_t)((nmt_all + 1) / 2) * N;
    a.flat = flat_ok && (g_flat > 0 || (g_flat < 0 && flat_env && !rec && g_thin < 0 && g_split < 0 && thin_tiles > (a.thin && nmt_all <= 4 ? 512u : 256u) &&
                         (fmt == 8 ? a.nbt >= 2 : a.nbt >= 4 && frun <= 512) && fwg <= (a.nbt >= 8 ? 512u : 256u)));
    if (a.flat) { a.thin = a.row = a.row1 = a.areg = false; a.wrec = 1; }
    if (a.thin || a.flat) { big = false; MT = 1; NT = 2; a.CB = a.flat ? 2 : a.nbt; }
    // the general kernel's one-tile, two-plane launches, pipelined (conv3_pipe.hpp), up to 512 workgroups (what the coarse form and the divided slices of three launch at the most): a workgroup
    // has a CU's LDS to itself, or half of it where its stages shrink to three pairs (conv3_pipe_pps). A conv with its statistics, us, conv3_mx_k / this. e4m3: 256 -> 256 at 2 x 16^3 (256 workgroups)
    // 38.9 / 25.3, 128 -> 256 23.4 / 16.7, at 3 x 16^3 (384) 256 -> 256 45.2 / 33.4, at 22 x 26^2 (352) 384 -> 128 66.3 / 48.1, 128 -> 128 27.9 / 22.0, 64 -> 128 18.9 / 16.0; e2m1: 256 -> 256 at 2 x 12^3
    // (192) 24.7 / 17.0, in stages of three pairs 64 -> 128 at 22 x 26^2 (352) 15.8 / 13.4, 32 -> 128 13.2 / 11.8, 64 -> 256 at 3 x 11 x 16^2 (288) 14.5 / 12.3, 192 -> 192 at 2 x 16^3 (192) 20.7 / 14.6, 384 -> 128 there (128) 32.9 / 20.8. Past one round of CUs in chunks of three or four blocks two or more chunks still gain - 384 -> 128
    // at 22 x 26^2 40.9 / 37.8, 192 -> 192 at 5 x 16^3 (480) 25.4 / 24.3 -, one does not: 128 -> 128 at 22 x 26^2 20.3 / 21.2
    static int pipe_env = -1;
    if (pipe_env < 0) pipe_env = getenv("MI_CONV_PIPE") ? atoi(getenv("MI_CONV_PIPE")) : 512;      // tuning knob: that workgroup count (0: never)
    const size_t pipe_tiles = (size_t)((Wo + 15) / 16) * ((Ho + 7) / 8) * ((Do + 1) / 2) * nmt_all * N;
    const int pipe_pps = conv3_pipe_pps(fmt, a.CB, pipe_tiles);
    a.pipe = stride == 1 && !act && MT == 1 && NT == 2 && a.wide && !big && !a.areg && !a.row && !a.thin && !a.flat && (fmt == 8 ? a.CB == 1 : a.CB <= 4) && a.nbt % a.CB == 0 && S < ((size_t)1 << 31) &&
             pipe_tiles <= (size_t)pipe_env && (pipe_tiles <= 256 || pipe_pps == 3 || a.nbt > a.CB);
    size_t smem = a.pipe ? conv3_pipe_lds(fmt, a.CB, pipe_pps) : a.flat ? (size_t)(fmt == 8 ? flat_t<8>::LDS : flat_t<4>::LDS) : a.thin ? MI_THIN_LDS : a.row1 ? (size_t)10 * 352 * (RB + 4) : a.row ? (size_t)2 * 2048 * (RB + 4) : a.areg ? (size_t)2 * ((TT + 63) / 64 * 64) * (RB + 4) : big ? (size_t)4 * MT * (WTILE + 256) + (size_t)3 * ((TT + 63) / 64 * 64) * (RB + 4) + (size_t)(((27 * a.nbt + 1) >> 1) + 2) * 2 * wide_tab_entry(fmt) : lds_bytes(a.CB);
    if (s2d) smem = a.s2row ? conv3s2_row_lds(fmt) : 0;
    smem = (smem + 15) & ~(size_t)15;
    a.epi_o = (unsigned)smem; smem += (size_t)3 * (a.flat ? 2 : MT) * 32 * sizeof(float);      // bias, affine a, b of the workgroup's channels
    a.red_o = (unsigned)smem; smem += a.row1 ? 3 * 2048 + 3 * 1024 : 1024;      // statistics scratch (the one-block row kernel: the weight fragments of two tap classes instead)
    if (s2d && !a.s2row) smem += (size_t)(27 * a.nbt + 1 + 8) * sizeof(int);                // the direct stride-2 kernel's K-order table
    // the row kernel in e2m1: the prepared weights of up to four input blocks stay in LDS (MI_CONV_ROW_WL=0: loaded from global memory per tap class)
    static int wl_env = -1;
    if (wl_env < 0) wl_env = getenv("MI_CONV_ROW_WL") ? atoi(getenv("MI_CONV_ROW_WL")) : 1;
    a.wl_o = 0;
    if (a.row && !a.row1 && fmt == 4 && wl_env && smem + (size_t)a.nbt * 15 * 1280 <= 160 * 1024) { a.wl_o = (unsigned)smem; smem += (size_t)a.nbt * 15 * 1280; }
    if (smem > 160 * 1024) mi_die("%s: %zu bytes of LDS for %d input blocks in chunks of %d", who, smem, a.nbt, a.CB);      // (every form above sizes its chunks to fit)
    if (big || a.areg || a.row || a.s2row || a.pipe) {
        // rows and scale bytes of positions outside the volume: 64 zero bytes, then 64 bytes of value 1; one page per device, kept for the process
        // (the entry point that must not allocate keeps its own at the head of its fixed scratch)
        static uint8_t *zpage[8];
        int dv = 0; MIRT(hipGetDevice(&dv)); dv &= 7;
        if (mi_ws_arena_on()) a.zpage = g_static_zpage;
        else {
            if (!zpage[dv]) {
                uint8_t init[128]; memset(init, 0, 64); memset(init + 64, 1, 64);
                MIRT(hipMalloc((void **)&zpage[dv], 128)); mi_count_alloc();
                if (!zpage[dv]) mi_die("%s: no device memory for the constant page", who);
                MIRT(hipMemcpy(zpage[dv], init, 128, hipMemcpyHostToDevice));
            }
            a.zpage = zpage[dv];
        }
    }
    a.nmt_all = nmt_all; a.ncs = nmt_all / MT;
    a.ntx = a.row ? (Wo + 31) / 32 : (Wo + 15) / 16; a.nty = (Ho + 7) / 8; a.ntz = (Do + TZ - 1) / TZ;      // (the row kernel: 4 x 8 x 32 voxels per tile)
    a.ntiles = (unsigned)((size_t)a.ntx * a.nty * a.ntz * a.ncs * N);
    if (a.thin || a.flat) {                                       // (their statistics records; whether they leave planes out rides on the offset, below 32)
        const thin_runs_t t = mi_thin_runs(a.zi0, Do, Ho, Wo);
        a.zc = t.off | (a.zs0 > 0 || a.zs1 < Do ? 32 : 0); a.ntx = t.step; a.nty = (int)t.recs; a.ntz = (int)t.runs; a.ntiles = (unsigned)(t.recs * nmt_all * N);
        a.ngrp = (unsigned)((t.runs + 3) / 4);
    }
    if (a.s2row) { a.ntx = (Wo + 31) / 32; a.nty = (Ho + 3) / 4; a.ntz = Do; a.ntiles = (unsigned)((size_t)a.ntx * a.nty * Do * N); }
    // ---- weights ----
    int npairs_all = 0;
    for (int b0 = 0; b0 < a.nbt; b0 += a.CB) npairs_all += (27 * (a.nbt - b0 < a.CB ? a.nbt - b0 : a.CB) + 1) >> 1;
    if (a.row) npairs_all = 15 * a.nbt;              // (15 pairs per input block: its tap classes)
    // (sixteen pairs of padding: the kernels' weight loads run up to two ring stages ahead of the last pair)
    // (the wide kernel's weights are one buffer: codes and scale words interleaved pair by pair; its scale buffer is a stub)
    const size_t wq_bytes = (size_t)(npairs_all + 16) * nmt_all * (big ? WTILE + 256 : WTILE), wsc_bytes = big ? 256 : (size_t)(npairs_all + 16) * nmt_all * 256;
    a.wstride = (unsigned)((size_t)(npairs_all + 16) * MT * (WTILE + 256));
    const int memoCB = big ? -a.CB : a.CB;
    a.big = big;
    const int CxP = (Cx + 31) / 32 * 32;
    int dev = 0; MIRT(hipGetDevice(&dev));
    uint8_t *wq = nullptr, *wsc = nullptr; bool have = false;
    if (sp.wkey && !mi_ws_arena_on()) {
        std::lock_guard<std::mutex> lk(g_wmemo_mu);
        for (auto &m : g_wmemo)
            if (m.key == sp.wkey && m.w == w && m.fmt == fmt && m.Co == cout && m.Ci == Ci && m.Cx == Cx && m.nbt == a.nbt && m.CB == memoCB && m.nmt_all == nmt_all && m.dev == dev && m.lay == (big ? MT : a.row ? 100 : s2d ? 200 : a.thin ? 300 + stride : 0)) { wq = m.wq; wsc = m.wsc; have = true; break; }
        if (!have) {
            MIRT(hipMalloc((void **)&wq, wq_bytes)); MIRT(hipMalloc((void **)&wsc, wsc_bytes)); mi_count_alloc(); mi_count_alloc();
            if (!wq || !wsc) mi_die("%s: no device memory for the prepared weights", who);
            MIRT(hipMemsetAsync(wq, 0, wq_bytes, 0)); MIRT(hipMemsetAsync(wsc, 0, wsc_bytes, 0));
            g_wmemo.push_back(wmemo_t{sp.wkey, w, fmt, cout, Ci, Cx, a.nbt, memoCB, nmt_all, dev, big ? MT : a.row ? 100 : s2d ? 200 : a.thin ? 300 + stride : 0, wq, wsc});
        }
    } else { wq = (uint8_t *)mi_ws(MI_WS_WQ, wq_bytes); wsc = (uint8_t *)mi_ws(MI_WS_WSC, wsc_bytes); }
    if (!have) {
        const size_t nt = (size_t)npairs_all * nmt_all * 32;
        // 2-D fp4 weight scales (lp_set_w4_2d): the stride-1 e2m1 preps of more than 16 input channels, as src/lp_f4fwd.cuh:1163
        const int w2d = g_w2d_on() && fmt == 4 && stride == 1 && Ci > 16;
        if (fmt == 8) prep_w_k<8><<<nblk_(nt, 128), 128>>>(w, wq, (unsigned *)wsc, cout, Ci, Cx, CxP, a.nbt, a.CB, nmt_all, npairs_all, big ? MT : a.row ? -1 : s2d ? -2 : 0, 0);
        else prep_w_k<4><<<nblk_(nt, 128), 128>>>(w, wq, (unsigned *)wsc, cout, Ci, Cx, CxP, a.nbt, a.CB, nmt_all, npairs_all, big ? MT : a.row ? -1 : s2d ? -2 : 0, w2d);
        MICK();
    }
    a.wq = wq; a.wsc = wsc;
    a.stat_ch = osum && (cout / Go) % 4 ? 1 : 0;
    if (osum) a.part = (float *)mi_ws(MI_WS_MISC, (size_t)a.ntiles * (a.stat_ch ? 32 : a.wrec * MT * 8) * 2 * sizeof(float));
    const bool epi = act != 0;
    const int out = ybf == 3 ? 8 : ybf == 4 ? 4 : 0;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    const bool ktime = g_ktime && !mi_ws_arena_on();
    if (ktime) { MIRT(hipEventCreate(&ev0)); MIRT(hipEventCreate(&ev1)); MIRT(hipEventRecord(ev0, 0)); }
    if (s2d) {
        const dim3 grid((unsigned)((s2runs + 3) / 4), (unsigned)a.ncs, (unsigned)N);
        if (fmt == 8) conv3s2_launch_f8(out, MT, a, grid, smem); else conv3s2_launch_f4(out, MT, a, grid, smem);
    } else if (fmt == 8) { if (out == 8) conv3_launch_f8_o8(stride, epi, MT, NT, a, smem); else if (out == 4) conv3_launch_f8_o4(stride, epi, MT, NT, a, smem); else conv3_launch_f8_o0(stride, epi, MT, NT, a, smem); }
    else { if (out == 8) conv3_launch_f4_o8(stride, epi, MT, NT, a, smem); else if (out == 4) conv3_launch_f4_o4(stride, epi, MT, NT, a, smem); else conv3_launch_f4_o0(stride, epi, MT, NT, a, smem); }
    if (ktime) { MIRT(hipEventRecord(ev1, 0)); ktime_push(ev0, ev1, 2.0 * 27 * Ci * (double)cout * N * Do * Ho * Wo); }
    if (osum) conv_stats_reduce(who, a, MT, sp, osum);
    return 0;
}

// the consumer-side transform of a conv input (GroupNorm + SiLU while staging, re-quantisation to the compute format) done once into an MX
// tensor of the same channels, for a tensor several convs read: they then take y as a plain input and stage it as stored. Channels a
// multiple of 32. The bits of the convs' results do not change (the same pre-pass runs inside a conv otherwise).
extern "C" int mi_conv_prestage(const void *x, int xdt, shape5 s, gnp_t gp, void *y, int ybits) {
    if ((ybits != 8 && ybits != 4) || s.c % 32 || xdt < 0 || xdt > 4 || (gp.G > 0 && s.c % gp.G)) return -1;
    const size_t hw = (size_t)s.h * s.w;
    gn_for_slabs("mi_conv_prestage", gp, s.h * s.w, 0, s.d, [&](int z0, int z1, gnp_t gs) { mi_restage_sub(x, xdt, s.n, s.c, (size_t)(z1 - z0) * hw, gs, s.c, 0, y, ybits, (size_t)s.d * hw, (size_t)z0 * hw); });
    return 0;
}
extern "C" int mi_conv_prestage2(const void *x, shape5 s, gnp_t gp, void *y8, void *y4) {
    if (s.c % 32 || (gp.G > 0 && s.c % gp.G) || !y8 || !y4) return -1;
    const size_t hw = (size_t)s.h * s.w;
    gn_for_slabs("mi_conv_prestage2", gp, s.h * s.w, 0, s.d, [&](int z0, int z1, gnp_t gs) { mi_restage_sub2(x, 3, s.n, s.c, (size_t)(z1 - z0) * hw, gs, y8, y4, (size_t)s.d * hw, (size_t)z0 * hw); });
    return 0;
}
extern "C" int lp_conv_fwd_f8(const void *x, int xbf, shape5 xs, const float *w, const float *b, int cout, void *y, int ybf, gnp_t gp, double *osum, int Go, split_t sp) {
    return conv_dispatch("lp_conv_fwd_f8", 8, 1, x, xbf, xs, w, b, cout, y, ybf, gp, osum, Go, sp, nullptr, nullptr, 0);
}
extern "C" int lp_conv_fwd_f4(const void *x, int xbf, shape5 xs, const float *w, const float *b, int cout, void *y, int ybf, gnp_t gp, double *osum, int Go, split_t sp) {
    return conv_dispatch("lp_conv_fwd_f4", 4, 1, x, xbf, xs, w, b, cout, y, ybf, gp, osum, Go, sp, nullptr, nullptr, 0);
}
// prepared-weight memo id of the calling thread's next stride-2 conv, 3x3x3 or 2x2x2 (their signatures carry no split_t): 0 = prepare per call
static thread_local unsigned g_s2_wkey = 0;
extern "C" void mi_conv_s2_wkey(unsigned wkey) { g_s2_wkey = wkey; }
unsigned mi_take_s2_wkey(void) { const unsigned k = g_s2_wkey; g_s2_wkey = 0; return k; }      // (the 2x2x2 entries consume it too)
extern "C" void mi_conv_stem_zc(int zc) { g_stem_zc = zc; }
extern "C" int lp_conv_fwd_s2_f8(const void *x, int xbf, shape5 xs, const float *w, const float *b, int cout, void *y, int ybf, shape5 ys, gnp_t gp) {
    const int Do = (xs.d - 1) / 2 + 1, Ho = (xs.h - 1) / 2 + 1, Wo = (xs.w - 1) / 2 + 1;
    if (ys.d != Do || ys.h != Ho || ys.w != Wo || ys.c != cout || ys.n != xs.n) mi_die("lp_conv_fwd_s2_f8: output shape %d x %d x %d x %d x %d does not match a stride-2 conv of the input", ys.n, ys.c, ys.d, ys.h, ys.w);
    split_t sp; memset(&sp, 0, sizeof sp);
    sp.wkey = g_s2_wkey; g_s2_wkey = 0;
    // compute format as the reference's dispatch (src/lp_s2.cu:647-754): fp4 only for an MX-fp4 32 -> <= 32 channel conv on even dims, else fp8
    const bool f4 = xbf == 4 && xs.c == 32 && cout <= 32 && !(xs.d & 1) && !(xs.h & 1) && !(xs.w & 1);
    conv_dispatch("lp_conv_fwd_s2_f8", f4 ? 4 : 8, 2, x, xbf, xs, w, b, cout, y, ybf, gp, nullptr, 0, sp, nullptr, nullptr, 0);
    return f4 ? 3 : 0;
}
extern "C" int mi_conv_fwd_gn(int bits, const void *x, int xbf, shape5 xs, const float *w, const float *b, int cout, void *y, int ybf, gnp_t gp,
                              double *osum, int Go, split_t sp, float eps, float *omean, float *orstd) {
    if (bits != 8 && bits != 4) mi_die("mi_conv_fwd_gn: compute format %d (8 or 4)", bits);
    if (!osum || !omean || !orstd || Go <= 0) mi_die("mi_conv_fwd_gn: needs sum slots, mean and rstd buffers and groups");
    g_fin = gn_fin_t{omean, orstd, 0.0, eps};
    const int rc = conv_dispatch("mi_conv_fwd_gn", bits, 1, x, xbf, xs, w, b, cout, y, ybf, gp, osum, Go, sp, nullptr, nullptr, 0);
    g_fin = gn_fin_t{nullptr, nullptr, 0.0, 0.f};
    return rc;
}
extern "C" int mi_conv_fwd_gn_stage(int bits, const void *x, int xbf, shape5 xs, const float *w, const float *b, int cout, void *y, int ybf, gnp_t gp,
                                    double *osum, int Go, split_t sp, float eps, float *omean, float *orstd, const float *gamma, const float *beta, void *st8, void *st4) {
    if (cout % 32 || ybf < 3 || !gamma || !beta || (!st8 && !st4) || sp.Di || sp.yD || sp.zlo || sp.zhi || Go <= 0 || cout % Go || xs.n <= 0 || xs.c <= 0 || xs.d <= 0 || xs.h <= 0 || xs.w <= 0) { take_once(); return -1; }
    g_stage = gn_stage_t{gamma, beta, st8, st4};
    const int rc = mi_conv_fwd_gn(bits, x, xbf, xs, w, b, cout, y, ybf, gp, osum, Go, sp, eps, omean, orstd);
    g_stage.gamma = nullptr;
    return rc;
}
extern "C" int mi_conv_fwd_fused(int bits, const void *x, int xbf, shape5 xs, const float *w, const float *b, int cout, void *y, int ybf,
                                 const float *ep_a, const float *ep_b, int act, gnp_t gp, double *osum, int Go, split_t sp) {
    if (bits != 8 && bits != 4) mi_die("mi_conv_fwd_fused: compute format %d (8 or 4)", bits);
    if (act < 0 || act > 3 || (!act && ep_a) || (!ep_a != !ep_b)) mi_die("mi_conv_fwd_fused: activation %d / affine arguments", act);
    return conv_dispatch("mi_conv_fwd_fused", bits, 1, x, xbf, xs, w, b, cout, y, ybf, gp, osum, Go, sp, ep_a, ep_b, act);
}

// ---- the stride-1 convs for callers that cannot allocate (serving loops, harnesses that forbid hipMalloc) ----
// Every byte of device memory the conv needs beyond its inputs and outputs - prepared weights, re-staged operands, the coarse rows of a fused
// upsample, per-tile statistics partials, the constant page of out-of-volume rows - is carved from one file-scope device array. The array is a
// host-side stand-in by name: its device address is taken once per device and only that address is used from then on.
#define MI_STATIC_SCRATCH_BYTES ((size_t)64 << 20)
static __device__ __align__(256) unsigned char scratch[MI_STATIC_SCRATCH_BYTES];
static unsigned char *g_scratch_ptr[8];        // per device: the address of that device's copy of the array
static std::mutex g_scratch_mu;
extern "C" size_t mi_conv_static_scratch_bytes(void) { return MI_STATIC_SCRATCH_BYTES; }
// an upper bound of what conv_dispatch will request from mi_ws for this call, following its choices (every request rounded up to 256 bytes)
static size_t conv_scratch_bound(int fmt, const void *x2, int xbf, int ybf, shape5 xs, int cout, gnp_t gp, const double *osum, split_t sp) {
    auto al = [](size_t n) { return ((n + 255) & ~(size_t)255) + 256; };
    const int Ci = xs.c, Cx = x2 ? sp.c_split : Ci, C2 = Ci - Cx, N = xs.n, D = sp.Di ? sp.Di : xs.d;
    if (fmt == 4 && Ci <= 8) fmt = 8;
    const size_t S = (size_t)D * xs.h * xs.w, So = (size_t)xs.d * xs.h * xs.w;
    const int nmt_all = (cout + 31) / 32, fdt = fmt == 8 ? 3 : 4;
    // one-plane tiles of one channel tile: no launch has more (a z-range of one plane may still run the one-block row kernel: 512 bytes per tile of 32 voxels along x)
    const size_t tiles = (size_t)((xs.w + 15) / 16) * ((xs.h + 7) / 8) * (sp.Di && xs.d < 2 ? 2 : xs.d) * nmt_all * N;
    size_t need = 256;                                              // the constant page
    if (Ci <= 16 && !x2 && fmt == 8) need += al((size_t)9 * nmt_all * 2048) + al((size_t)9 * nmt_all * 256);      // the tap-packed kernels' weights
    const int nbt = (Cx + 31) / 32 + (x2 ? (C2 + 31) / 32 : 0);
    need += al(((size_t)(27 * nbt + 1) / 2 + 2 * nbt + 16) * nmt_all * 2304) + al(((size_t)(27 * nbt + 1) / 2 + 2 * nbt + 16) * nmt_all * 256);      // (at most 15 pairs per block)
    // the tap-packed kernels read their input as stored and apply its GroupNorm while staging: nothing is re-staged (conv_dispatch's routing)
    const bool stem = fmt == 8 && !x2 && ((xbf == 0 || xbf >= 2) && Ci <= (xbf == 0 ? 16 : 8) || (xbf >= 2 && Ci <= 16)) && (xbf == ybf || ybf >= 3);
    const bool s2g = x2 && sp.gp2.G;
    for (int s = 0; s < (x2 ? 2 : 1) && !stem; s++) {
        const gnp_t g = s2g ? (s ? sp.gp2 : gp) : gp;
        const bool upseg = s == 0 && sp.up, direct = xbf == fdt && !(g.G > 0) && !upseg;
        const int C = s ? C2 : Cx;
        if (!direct) need += al((size_t)N * ((C + 31) / 32) * S * 33);
        if (upseg) need += al((size_t)N * ((C + 31) / 32) * (S / 8) * 33);
    }
    const size_t thin_recs = xs.w <= flat_t<8>::WMAX || (So + 63) / 64 * nmt_all * N <= (size_t)(g_thin > 1024 ? g_thin : 1024) ? mi_thin_runs(sp.Di ? sp.zi0 : 0, xs.d, xs.h, xs.w).recs * nmt_all * N : 0;      // (the K-split kernel's, 64 bytes each: a few more than its runs)
    if (osum) need += al((tiles * 256 > thin_recs * 64 ? tiles * 256 : thin_recs * 64));
    return need;
}
// set-up, once per device with that device current: the array's address on this device, and the constant page at its head. mi_init calls it
// for the device it selects (a synchronous 128-byte copy: not something to meet for the first time inside a serving loop); the entry point
// repeats the call for a device nobody initialised through mi_init
int mi_conv_static_setup(const char *who) {
    int dv = 0; MIRT(hipGetDevice(&dv)); dv &= 7;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[dv]) return 0;
    unsigned char *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) { fprintf(stderr, "%s: the fixed scratch has no address on device %d: %s\n", who, dv, hipGetErrorString(e)); return -2; }
    uint8_t init[128]; memset(init, 0, 64); memset(init + 64, 1, 64);
    if (hipMemcpy(ptr, init, 128, hipMemcpyHostToDevice) != hipSuccess) { fprintf(stderr, "%s: cannot initialise the fixed scratch on device %d\n", who, dv); return -2; }
    g_scratch_ptr[dv] = ptr;
    return 0;
}
static int conv_fwd_static(const char *who, int fmt, const void *x, int xbf, shape5 xs, const float *w, const float *b, int cout, void *y, int ybf, gnp_t gp, double *osum, int Go, split_t sp) {
    int dv = 0; MIRT(hipGetDevice(&dv)); dv &= 7;
    if (!g_scratch_ptr[dv] && mi_conv_static_setup(who)) { take_once(); return -2; }
    const size_t need = conv_scratch_bound(fmt, sp.x2, xbf, ybf, xs, cout, gp, osum, sp);
    if (need > MI_STATIC_SCRATCH_BYTES) {
        fprintf(stderr, "%s: this call needs up to %zu bytes of scratch (prepared weights, re-staged operands, statistics partials); the fixed scratch holds %zu. "
                        "Use lp_conv_fwd_f8 / lp_conv_fwd_f4, which allocate, or pass an input that is already in the compute format without GroupNorm\n", who, need, (size_t)MI_STATIC_SCRATCH_BYTES);
        take_once();
        return -1;
    }
    unsigned char *ptr = g_scratch_ptr[dv];
    g_static_zpage = ptr;                                          // bytes [0, 128): zero rows, then scale bytes of value 1
    mi_ws_arena(ptr + 256, MI_STATIC_SCRATCH_BYTES - 256);         // everything else is carved per call, and fully written before it is read
    const int rc = conv_dispatch(who, fmt, 1, x, xbf, xs, w, b, cout, y, ybf, gp, osum, Go, sp, nullptr, nullptr, 0);
    mi_ws_arena(nullptr, 0);
    g_static_zpage = nullptr;
    return rc;
}
extern "C" int mi_conv_fwd_static(int bits, const void *x, int xbf, shape5 xs, const float *w, const float *b, int cout, void *y, int ybf, gnp_t gp, double *osum, int Go, split_t sp) {
    if (bits != 8 && bits != 4) { fprintf(stderr, "mi_conv_fwd_static: compute format %d (8 or 4)\n", bits); take_once(); return -1; }
    return conv_fwd_static("mi_conv_fwd_static", bits, x, xbf, xs, w, b, cout, y, ybf, gp, osum, Go, sp);
}
