// Prefill-sized routed-MoE layer on gfx950: grouped rows, the input transforms, two MFMA grouped GEMMs on trellis
// tiles decoded into registers, SwiGLU, output transform and weighted combine.
//
// The decode path (k_moe.hip) reproduces the reference's EXACT accumulation order, which keeps every product in a
// sequential fp32 chain; at prefill sizes (thousands of tokens) that order is an MFMA-free GEMM. This path instead
// accumulates with v_mfma_f32_16x16x32_f16: dequantized weights are the same bit-exact fp16 values, every rounding
// point of the reference's transforms is kept (prep_block, out_block, act_mul; ft_core.h:96-132), but the sums over
// the hidden dimension are formed in MFMA order. Its outputs therefore differ from EXACT by accumulation rounding
// only, the same way the reference's own fp64 expert does (ref_expert, ft_core.h:1674-1691).
//
// Operand layout: the trellis decode leaves lane l = 16q + n holding the four weights of column n at tile rows
// 2q + {0, 1, 8, 9}. That is exactly the B slice of lane l in v_mfma_f32_16x16x16_f16 when the k index 4q + jj stands
// for tile row 2q + {0, 1, 8, 9}[jj]; the inputs are stored with the same row permutation ([tk][q][jj] per tile row),
// so each decoded tile feeds the MFMA directly, with no transpose. gfx950's v_mfma_f32_16x16x32_f16 takes two such
// slices (tile rows r and r + 1) per lane as its 8 k-values.
#include <algorithm>
#include <type_traits>

#include "gfl_device.hpp"
#include "gfl_internal.hpp"

namespace gfl {

// ---------------------------------------------------------------------------------------------------------------
// grouped rows (tier_lut_build_grouped_rows semantics, ft_tier_ext.cpp:1047-1097) and the combine order
// ---------------------------------------------------------------------------------------------------------------

constexpr int GP_MT = 80;          // slots per GEMM pass (up to 5 MFMA row blocks)
constexpr int GP_PLAN_THREADS = GP_PLAN_CHUNK;   // one thread per pick of a chunk
constexpr int GP_PLAN_WAVES = GP_PLAN_THREADS / 64;
constexpr int GP_ORDER_THREADS = 256;

// Slots are expert-major, experts ascending, picks (hence tokens) ascending within an expert; picks with ids outside
// [0, E) are skipped (ids other than -1 are counted in hdr[1]). The combine order of a token's picks is the
// reference's job order: moe_forward (ft_core.h:1343-1349) scans picks token-major and opens a job for an expert at
// its first pick and after every 8 of its picks, so pick p (the c-th of its expert) lands in the job opened by that
// expert's pick number c - c % 8, and jobs are numbered in the order their opening picks appear. A call of one chunk
// takes one launch (gp_plan_kernel: 6.6 us at 184 picks, against 15.4 us of three), a longer one three launches over
// chunks of GP_PLAN_CHUNK picks: ranks within each chunk, then placement (every chunk sums the counts
// of the chunks before it), then each token's picks in job order.

// Bit mask of the lanes below this one.
__device__ __forceinline__ uint64_t gp_lanes_below(int lane)
{
    return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// Pass 1, one workgroup per chunk: each pick's rank among the same-expert picks of its chunk, in pick order (same
// expert lanes of a wave from ten ballots on the id bits, E <= 1024, plus the group sizes of the waves before), into
// pick_c; and the chunk's per-expert counts into ccnt[chunk][0, E), with its count of ids outside [-1, E) at [E].
__global__ __launch_bounds__(GP_PLAN_THREADS) void gp_rank_kernel(const int64_t* __restrict__ sel, int P, int E,
                                                                  GPlan g)
{
    __shared__ int s_cnt[MAX_EXPERTS];
    __shared__ unsigned char s_wcnt[GP_PLAN_WAVES][MAX_EXPERTS];   // group sizes (<= 64) of each wave
    __shared__ int s_bad;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int p = blockIdx.x * GP_PLAN_THREADS + t;
    const int64_t e64 = p < P ? sel[p] : -1;
    if (t < E) s_cnt[t] = 0;
    if (t == 0) s_bad = 0;
    for (int i = t; i < GP_PLAN_WAVES * MAX_EXPERTS / 4; i += GP_PLAN_THREADS)
        reinterpret_cast<int*>(&s_wcnt[0][0])[i] = 0;
    const bool ok = e64 >= 0 && e64 < E;
    const int e = ok ? (int)e64 : 0;
    uint64_t eq = __ballot(ok);
#pragma unroll
    for (int b = 0; b < 10; ++b)
    {
        const bool bit = ok && ((e >> b) & 1);
        const uint64_t m = __ballot(bit);
        eq &= bit ? m : ~m;
    }
    const int cin = __popcll(eq & gp_lanes_below(lane));
    const bool lead = ok && cin == 0;   // lowest lane of its expert's group
    __syncthreads();
    if (lead) s_wcnt[wv][e] = (unsigned char)__popcll(eq);
    else if (!ok && e64 != -1) atomicAdd(&s_bad, 1);
    __syncthreads();
    if (ok)
    {
        int r = cin;
        for (int v = 0; v < wv; ++v) r += s_wcnt[v][e];
        g.pick_c[p] = r;
    }
    if (lead) atomicAdd(&s_cnt[e], __popcll(eq));
    __syncthreads();
    int* cc = g.ccnt + (size_t)blockIdx.x * (E + 1);
    if (t < E) cc[t] = s_cnt[t];
    if (t == 0) cc[E] = s_bad;
}

// Inclusive scan over the 64 lanes of a wave.
__device__ __forceinline__ int gp_wave_scan(int v, int lane)
{
#pragma unroll
    for (int d = 1; d < 64; d <<= 1)
    {
        const int o = __shfl_up(v, d);
        if (lane >= d) v += o;
    }
    return v;
}

constexpr int GP_HIST = 256;   // sizes the items' counting sort tells apart (4 per lane of a wave)

// The GEMM's items: every expert's slots in passes of mt, a workgroup per pass (and column block), so that an expert
// with many slots runs its passes side by side. Whole passes first, then the remainders by descending size: the longest
// workgroups go first and the short ones fill the end of the launch. The remainders are placed by a counting sort over
// their sizes (mt <= GP_HIST; ties in any order, the items are independent). Comparing every expert with every other
// instead took about 10 us of the plan at E = 288. Whole workgroup of GP_PLAN_THREADS, thread t = expert t: tot slots
// from slot off; s_hist and s_full are LDS scratch; ends with a barrier.
__device__ __forceinline__ void gp_items(int t, int E, int mt, int tot, int off, const GPlan& g, int* s_hist,
                                         int* s_full)
{
    const int lane = t & 63, wv = t >> 6;
    const int full = t < E ? tot / mt : 0, rem = t < E ? tot - full * mt : 0;
    if (t < GP_HIST) s_hist[t] = 0;
    const int finc = gp_wave_scan(full, lane);
    if (lane == 63) s_full[wv] = finc;
    __syncthreads();
    int at = 0;   // place among the remainders of the same size
    if (rem > 0) at = atomicAdd(&s_hist[rem], 1);
    int fpre = 0, nfull = 0;
    for (int v = 0; v < GP_PLAN_WAVES; ++v)
    {
        fpre += v < wv ? s_full[v] : 0;
        nfull += s_full[v];
    }
    __syncthreads();
    if (wv == 0)
    {
        const int b = GP_HIST - 1 - 4 * lane;   // sizes descending over the lanes, four a lane
        const int v0 = s_hist[b], v1 = s_hist[b - 1], v2 = s_hist[b - 2], v3 = s_hist[b - 3];
        const int inc = gp_wave_scan(v0 + v1 + v2 + v3, lane);
        s_hist[b] = inc - v0 - v1 - v2 - v3;
        s_hist[b - 1] = inc - v1 - v2 - v3;
        s_hist[b - 2] = inc - v2 - v3;
        s_hist[b - 3] = inc - v3;
        if (lane == 63) g.hdr[2] = nfull + inc;
    }
    __syncthreads();
    const int f0 = fpre + finc - full;
    for (int k = 0; k < full; ++k) g.item[f0 + k] = make_int4(t, off + k * mt, mt, 0);
    if (rem > 0) g.item[nfull + s_hist[rem] + at] = make_int4(t, off + full * mt, rem, 0);
}

// Pass 2, one workgroup per chunk: expert e's picks in earlier chunks (base_e) and in all chunks (its slot count),
// slot offsets by a scan of the counts, and the jobs opened before the chunk, sum over e of ceil(base_e / 8) (the
// expert's ranks 0, 8, 16, ... below base_e); a pick's global rank is base_e plus its rank in the chunk, and a pick
// of rank r opens a job when r % 8 == 0, numbered after the chunk's earlier openers. Workgroup 0 also writes the
// counts, offsets, header and the GEMM's items (passes of up to mt slots of an expert).
__global__ __launch_bounds__(GP_PLAN_THREADS) void gp_place_kernel(const int64_t* __restrict__ sel, int P, int E,
                                                                   int mt, GPlan g)
{
    __shared__ int s_base[MAX_EXPERTS];
    __shared__ int s_off[MAX_EXPERTS];
    __shared__ int s_hist[GP_HIST];
    __shared__ int s_wtot[GP_PLAN_WAVES], s_wjob[GP_PLAN_WAVES], s_wop[GP_PLAN_WAVES];
    __shared__ int s_bad;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int c = blockIdx.x, nch = gridDim.x;
    const int p = c * GP_PLAN_THREADS + t;
    const int64_t e64 = p < P ? sel[p] : -1;
    const bool ok = e64 >= 0 && e64 < E;
    const int e = ok ? (int)e64 : 0;
    const int rc = ok ? g.pick_c[p] : 0;
    if (t == 0) s_bad = 0;
    int base = 0, tot = 0;
    if (t < E)
    {
#pragma unroll 8
        for (int k = 0; k < nch; ++k)
        {
            const int v = g.ccnt[(size_t)k * (E + 1) + t];
            tot += v;
            base += k < c ? v : 0;
        }
    }
    const int inc = gp_wave_scan(tot, lane);
    const int jinc = gp_wave_scan((base + 7) >> 3, lane);
    if (lane == 63)
    {
        s_wtot[wv] = inc;
        s_wjob[wv] = jinc;
    }
    __syncthreads();
    if (c == 0 && t < nch) atomicAdd(&s_bad, g.ccnt[(size_t)t * (E + 1) + E]);
    int pre = 0, jbase = 0;
    for (int v = 0; v < GP_PLAN_WAVES; ++v)
    {
        pre += v < wv ? s_wtot[v] : 0;
        jbase += s_wjob[v];
    }
    const int off_e = pre + inc - tot;
    if (t < E)
    {
        s_base[t] = base;
        s_off[t] = off_e;
        if (c == 0)
        {
            g.cnt[t] = tot;
            g.off[t] = off_e;
            if (t == E - 1)
            {
                g.off[E] = off_e + tot;
                g.hdr[0] = off_e + tot;
            }
        }
    }
    __syncthreads();
    if (c == 0)
    {
        if (t == 0) g.hdr[1] = s_bad;
        gp_items(t, E, mt, tot, off_e, g, s_hist, s_wop);
        __syncthreads();   // s_wop is used again below
    }
    const int r = ok ? s_base[e] + rc : 0;
    const bool opener = ok && (r & 7) == 0;
    const uint64_t om = __ballot(opener);
    if (lane == 0) s_wop[wv] = __popcll(om);
    __syncthreads();
    int job = jbase + __popcll(om & gp_lanes_below(lane));
    for (int v = 0; v < wv; ++v) job += s_wop[v];
    if (p < P)
    {
        if (ok)
        {
            const int s = s_off[e] + r;
            g.slot_pick[s] = p;
            g.slot_e[s] = e;
            if (opener) g.slot_job[s] = job;
            g.pick_slot[p] = s;
            g.pick_c[p] = r;
        }
        else g.pick_slot[p] = -1;
    }
}

// Pass 3, one thread per pick, whole tokens per workgroup: each token's picks in (job, pick) order with their fp32 weights
// and svh_down addresses. A pick of global rank c reads its job number from the slot of its job's opening pick, c % 8 slots
// before its own; its place is the number of the token's picks before it. (A thread per token, loading its picks' chains
// of addresses one after another, took 15.2 us at M = 2048, this 4.9 us.)
__global__ __launch_bounds__(GP_ORDER_THREADS) void gp_order_kernel(const uint64_t* __restrict__ ptrs, const void* w,
                                                                    int w_half, int M, int topk, GPlan g)
{
    __shared__ int s_job[GP_ORDER_THREADS];   // each pick's job, -1 if skipped
    const int t = threadIdx.x, toks = GP_ORDER_THREADS / topk;   // tokens per workgroup
    const int tl = t / topk, k = t - tl * topk, tk = blockIdx.x * toks + tl;
    const bool mine = tl < toks && tk < M;
    int s = -1, jb = -1;
    float wt = 0.f;
    uint64_t svh = 0;
    if (mine)
    {
        const int p = tk * topk + k;
        s = g.pick_slot[p];
        const int c = g.pick_c[p];   // a stale value where the pick is skipped, not used
        wt = w_half ? h2f_bits(reinterpret_cast<const uint16_t*>(w)[p]) : reinterpret_cast<const float*>(w)[p];
        if (s >= 0)
        {
            jb = g.slot_job[s - (c & 7)];
            if (ptrs) svh = ptrs[(size_t)g.slot_e[s] * 9 + 8];
        }
    }
    s_job[t] = jb;
    __syncthreads();
    if (!mine) return;
    int r = 0, n = 0;
    for (int k2 = 0; k2 < topk; ++k2)
    {
        const int j2 = s_job[tl * topk + k2];
        n += j2 >= 0;
        r += j2 >= 0 && (j2 < jb || (j2 == jb && k2 < k));
    }
    if (s >= 0)
    {
        g.tok_slot[tk * topk + r] = s;
        g.tok_w[tk * topk + r] = wt;
        g.tok_svh[tk * topk + r] = svh;
    }
    if (k == 0) g.tok_npk[tk] = n;
}

// The three passes in one launch for a call of one chunk (P <= GP_PLAN_CHUNK): one workgroup, a thread per pick (and per
// expert). Ranks as gp_rank_kernel, placement as gp_place_kernel with nothing before the chunk, and each pick's place in
// its token's (job, pick) order by counting the token's picks before it.
__global__ __launch_bounds__(GP_PLAN_THREADS) void gp_plan_kernel(const uint64_t* __restrict__ ptrs,
                                                                  const int64_t* __restrict__ sel, const void* w,
                                                                  int w_half, int P, int topk, int E, int mt, GPlan g)
{
    __shared__ unsigned char s_wcnt[GP_PLAN_WAVES][MAX_EXPERTS];   // group sizes (<= 64) of each wave
    __shared__ int s_off[MAX_EXPERTS];
    __shared__ int s_job[GP_PLAN_THREADS];    // job number of the slot, at the slots of job-opening picks
    __shared__ int s_pjob[GP_PLAN_THREADS];   // each pick's job, -1 if skipped
    __shared__ int s_hist[GP_HIST];
    __shared__ int s_wtot[GP_PLAN_WAVES], s_wop[GP_PLAN_WAVES], s_full[GP_PLAN_WAVES];
    __shared__ int s_bad;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int64_t e64 = t < P ? sel[t] : -1;
    float wt = 0.f;
    if (t < P) wt = w_half ? h2f_bits(reinterpret_cast<const uint16_t*>(w)[t]) : reinterpret_cast<const float*>(w)[t];
    if (t == 0) s_bad = 0;
    for (int i = t; i < GP_PLAN_WAVES * MAX_EXPERTS / 4; i += GP_PLAN_THREADS)
        reinterpret_cast<int*>(&s_wcnt[0][0])[i] = 0;
    const bool ok = e64 >= 0 && e64 < E;
    const int e = ok ? (int)e64 : 0;
    const uint64_t svh = ok && ptrs ? ptrs[(size_t)e * 9 + 8] : 0;
    uint64_t eq = __ballot(ok);
#pragma unroll
    for (int b = 0; b < 10; ++b)
    {
        const bool bit = ok && ((e >> b) & 1);
        const uint64_t m = __ballot(bit);
        eq &= bit ? m : ~m;
    }
    const int cin = __popcll(eq & gp_lanes_below(lane));
    __syncthreads();
    if (ok && cin == 0) s_wcnt[wv][e] = (unsigned char)__popcll(eq);
    else if (!ok && e64 != -1) atomicAdd(&s_bad, 1);
    __syncthreads();
    int r = cin, tot = 0;
#pragma unroll
    for (int v = 0; v < GP_PLAN_WAVES; ++v)
    {
        r += v < wv ? s_wcnt[v][e] : 0;
        tot += s_wcnt[v][t];
    }
    if (t >= E) tot = 0;
    const int inc = gp_wave_scan(tot, lane);
    const bool opener = ok && (r & 7) == 0;
    const uint64_t om = __ballot(opener);
    if (lane == 63) s_wtot[wv] = inc;
    if (lane == 0) s_wop[wv] = __popcll(om);
    __syncthreads();
    int off_e = inc - tot, job = __popcll(om & gp_lanes_below(lane));
    for (int v = 0; v < wv; ++v)
    {
        off_e += s_wtot[v];
        job += s_wop[v];
    }
    s_off[t] = off_e;
    if (t < E)
    {
        g.cnt[t] = tot;
        g.off[t] = off_e;
        if (t == E - 1)
        {
            g.off[E] = off_e + tot;
            g.hdr[0] = off_e + tot;
        }
    }
    if (t == 0) g.hdr[1] = s_bad;
    gp_items(t, E, mt, tot, off_e, g, s_hist, s_full);   // its first barrier also orders s_off
    const int s = ok ? s_off[e] + r : -1;
    if (opener) s_job[s] = job;
    __syncthreads();
    const int jb = ok ? s_job[s - (r & 7)] : -1;
    s_pjob[t] = jb;
    if (t < P)
    {
        g.pick_slot[t] = s;
        if (ok)
        {
            g.slot_pick[s] = t;
            g.slot_e[s] = e;
        }
    }
    __syncthreads();
    if (t >= P) return;
    const int tk = t / topk, k = t - tk * topk;
    int rank = 0, npk = 0;
    for (int k2 = 0; k2 < topk; ++k2)
    {
        const int j2 = s_pjob[tk * topk + k2];
        npk += j2 >= 0;
        rank += j2 >= 0 && (j2 < jb || (j2 == jb && k2 < k));
    }
    if (ok)
    {
        g.tok_slot[tk * topk + rank] = s;
        g.tok_w[tk * topk + rank] = wt;
        g.tok_svh[tk * topk + rank] = svh;
    }
    if (k == 0) g.tok_npk[tk] = npk;
}

// ---------------------------------------------------------------------------------------------------------------
// transforms: one wave per slot, or per (token, group of blocks); each 16-lane row of the wave takes one 128-block,
// 8 elements per lane (16-byte loads), 4 blocks per round; exact rounding points. Small calls are bound by the latency of
// their dependent loads and give a slot to more waves (184 picks: input transform 11.4 -> 6.4 us, SwiGLU 9.9 -> 6.0 us)
// ---------------------------------------------------------------------------------------------------------------

constexpr int GP_TW = 4;   // waves per transform workgroup
constexpr int GP_TU = 2;   // rounds of 4 blocks per chunk of the input transform (two chunks' loads in flight)
constexpr int GP_TA = 3;   // rounds of 4 blocks per SwiGLU-transform wave (one wave covers I = 1536)
constexpr int GP_SMALL = 1024;   // picks up to which a SwiGLU-transform wave takes one round

// Elements 8li..8li+7 of 128-block b (one lane of a 16-lane row), rounded to fp16, into the accumulator-chain input
// layout: fp32, position tk * 16 + 4j + q holds row 2q + {0, 1, 8, 9}[j] of tile row tk (the rows chain j of every
// output column reads in tile row tk, in its order)
__device__ __forceinline__ void xg_store_row(float* dst, int b, int li, const float (&v)[8])
{
    float r[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) r[k] = h2f_bits((uint16_t)f2h_bits(v[k]));
    float* d = dst + (size_t)b * 128 + (li >> 1) * 16 + 8 * (li & 1);
    *reinterpret_cast<float4*>(d) = float4{ r[0], r[2], r[4], r[6] };
    *reinterpret_cast<float4*>(d + 4) = float4{ r[1], r[3], r[5], r[7] };
}

// prep_block (ft_core.h:97-102) of the gate and up inputs of slot s, `parts` waves per slot (prep_parts). XL: fp32 in the
// accumulator-chain layout (xg_store_row), else fp16 in the MFMA layout (gp_store_row), NT:
// with non-temporal stores.
template <bool XL, bool NT>
__global__ __launch_bounds__(GP_TW * 64) void gp_prep_kernel(const uint64_t* __restrict__ ptrs,
                                                             const uint16_t* __restrict__ x, int H, int topk, int cap,
                                                             int parts, GPlan g, void* __restrict__ xt_out)
{
    uint16_t* xt = static_cast<uint16_t*>(xt_out);
    float* xtf = static_cast<float*>(xt_out);
    const int lane = threadIdx.x & 63, rl = lane >> 4, li = lane & 15;
    const int w = blockIdx.x * GP_TW + (threadIdx.x >> 6), s = w / parts;
    const int e = g.slot_e[s], pick = g.slot_pick[s];   // read beside the slot count: past it stale entries, not used
    if (s >= g.hdr[0]) return;
    constexpr int CH = 4 * GP_TU;   // blocks per chunk
    const int nall = H / 128, span = (nall + parts * CH - 1) / (parts * CH) * CH;
    const int b0 = (w - s * parts) * span, nblk = min(nall, b0 + span);   // this wave's blocks [b0, nblk)
    if (b0 >= nblk) return;
    const int tok = pick / topk;
    const gptr<uint16_t> su0 = gaddr<uint16_t>(ptrs[(size_t)e * 9 + 3]);
    const gptr<uint16_t> su1 = gaddr<uint16_t>(ptrs[(size_t)e * 9 + 5]);
    const uint16_t* xr = x + (size_t)tok * H;
    uint16_t* d0 = xt + (size_t)s * H;
    uint16_t* d1 = xt + ((size_t)cap + s) * H;
    float* f0 = xtf + (size_t)s * H;
    float* f1 = xtf + ((size_t)cap + s) * H;
    uint4 xv[2][GP_TU], g0[2][GP_TU], g1[2][GP_TU];
    auto load = [&](int buf, int c0) {
#pragma unroll
        for (int k = 0; k < GP_TU; ++k)
        {
            const int o = min(c0 + 4 * k + rl, nblk - 1) * 128 + li * 8;
            xv[buf][k] = *reinterpret_cast<const uint4*>(xr + o);
            g0[buf][k] = gld16(su0, o);
            g1[buf][k] = gld16(su1, o);
        }
    };
    auto work = [&](int buf, int c0) {
#pragma unroll
        for (int k = 0; k < GP_TU; ++k)
        {
            const int b = c0 + 4 * k + rl;
            if constexpr (XL)
            {
                float u[8], v[8];
                prep_block_row_p(u, xv[buf][k], g0[buf][k]);
                prep_block_row_p(v, xv[buf][k], g1[buf][k]);
                if (b < nblk)
                {
                    xg_store_row(f0, b, li, u);
                    xg_store_row(f1, b, li, v);
                }
            }
            else
            {
                uint32_t u[4], v[4];
                prep_block_row_h(u, xv[buf][k], g0[buf][k]);
                prep_block_row_h(v, xv[buf][k], g1[buf][k]);
                if (b < nblk)
                {
                    gp_store_row<NT>(d0, b, li, u);
                    gp_store_row<NT>(d1, b, li, v);
                }
            }
        }
    };
    // two chunk buffers: the next chunk's loads are in flight while the current one is transformed
    load(0, b0);
    for (int c0 = b0; c0 < nblk; c0 += 2 * CH)
    {
        if (c0 + CH < nblk) load(1, c0 + CH);
        work(0, c0);
        if (c0 + 2 * CH < nblk) load(0, c0 + 2 * CH);
        if (c0 + CH < nblk) work(1, c0 + CH);
    }
}

// fwd_phase phase 1 (ft_core.h:974-991), one wave per (slot, 4 * TA blocks of I): per 128-block, out_block of
// gate and up, r16(act_mul), down prep_block, stored in the GEMM input layout
template <bool XL, int TA>
__global__ __launch_bounds__(GP_TW * 64) void gp_act_kernel(const uint64_t* __restrict__ ptrs, int I, int cap, GPlan g,
                                                            const uint16_t* __restrict__ ygu, const float* silu_tab,
                                                            float act_limit, void* __restrict__ xd_out)
{
    uint16_t* xd = static_cast<uint16_t*>(xd_out);
    const int lane = threadIdx.x & 63, rl = lane >> 4, li = lane & 15;
    const int nbi = I / 128, nch = (nbi + 4 * TA - 1) / (4 * TA);
    const int item = blockIdx.x * GP_TW + (threadIdx.x >> 6);
    const int s = item / nch, c0 = (item % nch) * 4 * TA;
    const int e = g.slot_e[s];   // read beside the slot count: past it a stale entry, not used
    if (s >= g.hdr[0]) return;
    const gptr<uint16_t> svh_g = gaddr<uint16_t>(ptrs[(size_t)e * 9 + 4]);
    const gptr<uint16_t> svh_u = gaddr<uint16_t>(ptrs[(size_t)e * 9 + 6]);
    const gptr<uint16_t> suh_d = gaddr<uint16_t>(ptrs[(size_t)e * 9 + 7]);
    const uint16_t* yg = ygu + (size_t)s * I;
    const uint16_t* yu = ygu + ((size_t)cap + s) * I;
    uint16_t* dst = xd + (size_t)s * I;
    float* dstf = static_cast<float*>(xd_out) + (size_t)s * I;
    // TA rounds of 4 blocks in three phases kept apart by scheduling barriers (left to itself the compiler sinks
    // each round's loads next to their use): all loads; the output transforms and every silu lookup; the
    // activation, input transform and stores
    {
        float gv[TA][8], uv[TA][8], ev[TA][8];
        uint4 gh[TA], uh[TA], sg[TA], su[TA], sd[TA];
#pragma unroll
        for (int k = 0; k < TA; ++k)
        {
            const int o = min(c0 + 4 * k + rl, nbi - 1) * 128 + li * 8;
            gh[k] = *reinterpret_cast<const uint4*>(yg + o);
            uh[k] = *reinterpret_cast<const uint4*>(yu + o);
            sg[k] = gld16(svh_g, o);
            su[k] = gld16(svh_u, o);
            sd[k] = gld16(suh_d, o);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < TA; ++k)
        {
            out_block_row_h(gv[k], gh[k], sg[k]);
            out_block_row_h(uv[k], uh[k], su[k]);
        }
#pragma unroll
        for (int k = 0; k < TA; ++k)
#pragma unroll
            for (int j = 0; j < 8; ++j) ev[k][j] = silu_tab[f2h_bits(gv[k][j]) & 0xFFFFu];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < TA; ++k)
        {
            const int b = c0 + 4 * k + rl;
            float av[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) av[j] = r16(act_mul_s(ev[k][j], uv[k][j], act_limit));
            if constexpr (XL)
            {
                prep_block_row_fp(av, sd[k]);
                if (b < nbi) xg_store_row(dstf, b, li, av);
            }
            else
            {
                uint32_t ah[4];
                prep_block_row_fh(ah, av, sd[k]);
                if (b < nbi) gp_store_row(dst, b, li, ah);
            }
        }
    }
}

// The same for calls of many picks, with the middle of the silu table in LDS. Each gate element is a lookup at an
// address of its own, which from L1 takes the kernel a cycle per lane: at M = 8192 (top-8, I = 1536) about 160 of its
// 274 us. A workgroup of 16 waves fills a CU's registers, holds the binades [2^-12, 16) of both signs (128 KB; other
// gates read the table in memory) and goes through the (slot, 12 blocks) items, consecutive ones side by side, so that
// the fill is paid once per CU. At M = 8192 it moves its 604 MB at 3.1 TB/s (before 2.2). Measured, gp_act_kernel ->
// this one, us, MFMA grouped inputs | fp32 chain inputs, E = 288: M = 250 12.2 -> 15.6 | 12.7 -> 15.1, M = 512 19.4 ->
// 17.8 | 20.6 -> 18.1, M = 768 27.2 -> 27.9 | 29.6 -> 27.9, M = 1024 34.7 -> 30.3 | 39.4 -> 29.9, M = 2048 71.0 -> 56.9
// | 74.6 -> 51.0, M = 8192 274 -> 196 | 299 -> 185: taken from 8,192 picks on: from there every measured size gains (at
// I = 1536 a wave has two items there; other I, which change a slot's items, and calls with skipped picks were not
// measured for the line).
constexpr int GL_NW = 16;          // waves per workgroup
constexpr int GL_CUS = 256;        // workgroups: one per CU of an undivided MI355X
constexpr int GL_MIN = 8192;       // picks from which the launch is taken
constexpr int GL_LO = 3 << 10;     // first fp16 pattern held (2^-12), and how many of each sign
constexpr int GL_N = 16 << 10;

template <bool XL>
__global__ __launch_bounds__(GL_NW * 64) void gl_act_kernel(const uint64_t* __restrict__ ptrs, int I, int cap, GPlan g,
                                                            const uint16_t* __restrict__ ygu,
                                                            const float* __restrict__ silu_tab, float act_limit,
                                                            void* __restrict__ xd_out)
{
    __shared__ __align__(16) float tab[2 * GL_N];
    for (int i = threadIdx.x; i < 2 * GL_N / 4; i += GL_NW * 64)
        reinterpret_cast<float4*>(tab)[i] =
            reinterpret_cast<const float4*>(silu_tab + GL_LO + (i < GL_N / 4 ? 0 : 0x8000 - GL_N))[i];
    __syncthreads();
    const int lane = threadIdx.x & 63, rl = lane >> 4, li = lane & 15;
    const int nbi = I / 128, nch = (nbi + 4 * GP_TA - 1) / (4 * GP_TA), items = g.hdr[0] * nch;
    for (int item = blockIdx.x * GL_NW + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); item < items;
         item += gridDim.x * GL_NW)
    {
        const int s = item / nch, c0 = (item % nch) * 4 * GP_TA;
        const uint64_t* pe = ptrs + (size_t)g.slot_e[s] * 9;
        const gptr<uint16_t> svh_g = gaddr<uint16_t>(pe[4]);
        const gptr<uint16_t> svh_u = gaddr<uint16_t>(pe[6]);
        const gptr<uint16_t> suh_d = gaddr<uint16_t>(pe[7]);
        const uint16_t* yg = ygu + (size_t)s * I;
        const uint16_t* yu = ygu + ((size_t)cap + s) * I;
        uint4 gh[GP_TA], uh[GP_TA], sg[GP_TA], su[GP_TA], sd[GP_TA];
#pragma unroll
        for (int k = 0; k < GP_TA; ++k)
        {
            const int o = min(c0 + 4 * k + rl, nbi - 1) * 128 + li * 8;
            gh[k] = *reinterpret_cast<const uint4*>(yg + o);
            uh[k] = *reinterpret_cast<const uint4*>(yu + o);
            sg[k] = gld16(svh_g, o);
            su[k] = gld16(svh_u, o);
            sd[k] = gld16(suh_d, o);
        }
        __builtin_amdgcn_sched_barrier(0);   // every load goes out before the first is used
#pragma unroll
        for (int k = 0; k < GP_TA; ++k)
        {
            float gv[8], uv[8];
            out_block_row_h(gv, gh[k], sg[k]);
            uint32_t gb[8], far = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j)
            {
                gb[j] = f2h_bits(gv[j]) & 0xFFFFu;
                const uint32_t m = (gb[j] & 0x7FFFu) - (uint32_t)GL_LO;
                far = max(far, m);
                gv[j] = tab[min(m, (uint32_t)GL_N - 1) + (gb[j] >> 15) * GL_N];
            }
            if (far >= (uint32_t)GL_N)
            {
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if ((gb[j] & 0x7FFFu) - (uint32_t)GL_LO >= (uint32_t)GL_N) gv[j] = silu_tab[gb[j]];
            }
            out_block_row_h(uv, uh[k], su[k]);
#pragma unroll
            for (int j = 0; j < 8; ++j) gv[j] = r16(act_mul_s(gv[j], uv[j], act_limit));
            const int b = c0 + 4 * k + rl;
            if constexpr (XL)
            {
                prep_block_row_fp(gv, sd[k]);
                if (b < nbi) xg_store_row(static_cast<float*>(xd_out) + (size_t)s * I, b, li, gv);
            }
            else
            {
                uint32_t ah[4];
                prep_block_row_fh(ah, gv, sd[k]);
                if (b < nbi) gp_store_row(static_cast<uint16_t*>(xd_out) + (size_t)s * I, b, li, ah);
            }
        }
    }
}

// out_block (ft_core.h:1016) of every expert output block and the weighted sum in job order (ft_core.h:1020-1033),
// one wave per (token, group of 4 blocks): each 16-lane row takes one block; lane k < npk holds the token's k-th pick
// (slot, weight, output scales), read back per pick with readlane; eight picks' loads are issued before their eight
// terms are added in order (against four: M = 2048 47.2 -> 46.1 us). Rows of tokens without a valid pick become 0.
constexpr int GP_CK = 8;   // picks whose loads a combine wave keeps in flight (all of a top-8 token's)

__global__ __launch_bounds__(GP_TW * 64) void gp_comb_kernel(int H, int M, int topk, GPlan g, const uint16_t* __restrict__ yraw,
                                                             float* __restrict__ out)
{
    const int lane = threadIdx.x & 63, rl = lane >> 4, li = lane & 15;
    const int nbh = H / 128, ngr = (nbh + 3) / 4;
    const int item = blockIdx.x * GP_TW + (threadIdx.x >> 6);
    const int tok = item / ngr, b = (item % ngr) * 4 + rl;
    if (tok >= M) return;
    const int npk = g.tok_npk[tok];
    // entries past the token's picks hold stale values, which are not used
    const int ml = tok * topk + min(lane, topk - 1);
    const int my_s = g.tok_slot[ml];
    const float my_w = g.tok_w[ml];
    const uint64_t my_p = g.tok_svh[ml];
    const int o = min(b, nbh - 1) * 128 + li * 8;
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.f;
    for (int k0 = 0; k0 < npk; k0 += GP_CK)
    {
        uint4 yh[GP_CK];
        uint4 sv[GP_CK];
        float wk[GP_CK];
#pragma unroll
        for (int i = 0; i < GP_CK; ++i)
        {
            const int k = min(k0 + i, npk - 1);
            const int s = __builtin_amdgcn_readlane(my_s, k);
            wk[i] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_w), k));
            const uint64_t pa = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(my_p >> 32), k) << 32) |
                                (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)my_p, k);
            yh[i] = *reinterpret_cast<const uint4*>(yraw + (size_t)s * H + o);
            sv[i] = gld16(gaddr<uint16_t>(pa), o);
        }
#pragma unroll
        for (int i = 0; i < GP_CK; ++i)
        {
            if (k0 + i >= npk) break;
            float v[8];
            out_block_row_h(v, yh[i], sv[i]);
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[j] = acc[j] + wk[i] * v[j];
        }
    }
    if (b < nbh)
    {
        float* orow = out + (size_t)tok * H + b * 128 + li * 8;
        *reinterpret_cast<float4*>(orow) = float4{ acc[0], acc[1], acc[2], acc[3] };
        *reinterpret_cast<float4*>(orow + 4) = float4{ acc[4], acc[5], acc[6], acc[7] };
    }
}

// ---------------------------------------------------------------------------------------------------------------
// MFMA grouped GEMM: y[slot][n] = sum_k x[slot][k] W_e[k][n] for every slot of every expert
// ---------------------------------------------------------------------------------------------------------------

constexpr int GP_NW = 8;           // waves per GEMM workgroup
constexpr int GP_CPW = 2;          // tile columns per wave (each A fragment read from LDS feeds GP_CPW MFMAs)
constexpr int GP_WCOLS = 16 * GP_NW * GP_CPW;   // output columns per workgroup (256)
constexpr int GP_XPW = GP_MT / GP_NW;           // slots whose input chunk each wave loads per group
constexpr int GP_NG = 2;           // ring depth (groups of 8 tile rows): 2 keeps two workgroups per CU
constexpr int GP_XS = 136;         // fp16 stride of one slot's group chunk in LDS (128 + 8: conflict-free reads)

typedef __attribute__((address_space(3))) void gp_lds_void;

template <int N>
__device__ __forceinline__ void gp_wait_vmcnt()
{
    static_assert(N >= 0 && N < 64, "vmcnt range");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Workgroup barrier without __syncthreads' release fence: that fence waits for vmcnt(0), i.e. for every LDS-direct load
// still in flight, which would drain the prefetch ring at every group. Each wave has already waited for its own loads
// of the group it is about to read; the barrier only has to order those waits and the previous group's LDS reads
// (waited for here, nothing else is outstanding on that counter) across the waves. The "memory" clobber keeps the
// compiler from moving LDS accesses across it.
__device__ __forceinline__ void gp_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

struct GemmArgs
{
    const uint64_t* ptrs;
    int mat_base, nmat;        // first matrix of the launch (0 gate, 1 up, 2 down) and how many
    int kdim, ndim, cap, nit;  // nit: items the grid covers
    GPlan g;
    const uint16_t* xin;       // [mats][cap][kdim] fp16, GEMM input layout
    uint16_t* yout;            // [mats][cap][ndim] fp16: out_block's leading r16 (ft_core.h:109) applied here
};

// Grid: 8 * ceil(items / 8) * (ndim / 256) * matrices, XCD-major. Workgroup = 8 waves x 2 tile columns = 256 output
// columns of one matrix for one item, a pass of up to GP_MT slots of an expert. Per group of 8 tile rows every
// wave decodes its 16 tiles and, per pair of tile rows, reads one A fragment (16 slots x 32 k) per row block of the
// pass and runs 2 MFMAs (16x16x32) with it, one per column. The tiles stream through per-wave LDS rings and the slots'
// inputs through a shared ring, both filled by LDS-direct loads GP_NG - 1 groups ahead; one workgroup barrier per group
// (group g landed for every wave; every wave is past group g - 1, whose slots are refilled after it).
template <int K>
__global__ __launch_bounds__(GP_NW * 64) void gp_gemm_kernel(GemmArgs a)
{
    constexpr int TB = 32 * K, RB = GP_CPW * TB, GB = 8 * RB, NG = GP_NG;
    constexpr int NLD = GB / 256;                 // trellis dword loads per lane per group
    constexpr int NV = NLD + GP_XPW;              // vector memory instructions per wave per group
    static_assert(GB % 256 == 0, "group of tiles must split into whole wave loads");
    extern __shared__ __align__(16) uint8_t gp_lds[];
    // the wave index in a scalar register, so every LDS-DMA destination (M0) is scalar arithmetic
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    // XCD-aware order: workgroups are dispatched round-robin over the 8 XCDs (XCD = linear id % 8), so every
    // workgroup of the it-th item of the dispatch order gets a linear id = it (mod 8) and the item's slot inputs are
    // fetched into one L2
    const int nch = a.ndim / GP_WCOLS, per = nch * a.nmat;
    const int xcd = blockIdx.x % 8, j = blockIdx.x / 8;
    const int it = (j / per) * 8 + xcd, rr0 = j % per;
    if (it >= a.nit || it >= a.g.hdr[2]) return;
    const int4 item = a.g.item[it];   // a pass of up to GP_MT slots of an expert
    const int e = item.x, c0 = item.y, T = item.z;
    const int nc = rr0 % nch;
    const int mat = a.mat_base + rr0 / nch;
    const int TN = a.ndim / 16, TK = a.kdim / 16, ngroups = TK / 8;
    const int t0 = (nc * GP_NW + wave) * GP_CPW;                     // this wave's first tile column
    uint8_t* ring = gp_lds + wave * NG * GB;                          // [NG][8 tile rows][GP_CPW columns][TB]
    uint16_t* xring = reinterpret_cast<uint16_t*>(gp_lds + GP_NW * NG * GB);   // [NG][GP_MT slots][GP_XS]
    const uint8_t* tr = reinterpret_cast<const uint8_t*>(a.ptrs[(size_t)e * 9 + mat]);
    const size_t gstride = (size_t)TN * TB;                           // bytes per tile row of the matrix
    uint8_t* cb = const_cast<uint8_t*>(uniform_ptr(tr + (size_t)t0 * TB));
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(cb, (short)0, (int)((size_t)TK * gstride),
                                                                        0x00020000);
    const int gs = (int)gstride;
    int voff[NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i)
    {
        const int byte = i * 256 + lane * 4;   // within the group's [8][GP_CPW][TB] block
        voff[i] = (byte / RB) * gs + (byte % RB);
    }
    const LaneDec d = lane_dec(lane, K);
    const uint16_t* xin = a.xin + (size_t)(mat - a.mat_base) * a.cap * a.kdim;
    // the slots' inputs through a buffer resource too: the lane's 4 bytes as the vector offset, row and group in the
    // scalar offset
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(uniform_ptr(reinterpret_cast<const uint8_t*>(xin))), (short)0,
        (int)((size_t)a.cap * a.kdim * 2), 0x00020000);
    uint16_t* yout = a.yout + (size_t)(mat - a.mat_base) * a.cap * a.ndim;
    const int q = lane >> 4, i16 = lane & 15;

    // byte offsets of the input rows this wave loads, the same in every lane (slots past the pass read the pass's
    // last slot): the scalar offset of its LDS-direct loads, whose vector offset is the lane's 4 bytes
    int xrow[GP_XPW];
#pragma unroll
    for (int j = 0; j < GP_XPW; ++j) xrow[j] = (c0 + min(wave * GP_XPW + j, T - 1)) * a.kdim * 2;
    const int xl = lane * 4;
    auto issue = [&](int g) {
        uint8_t* dst = ring + (g % NG) * GB;
#pragma unroll
        for (int i = 0; i < NLD; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (gp_lds_void*)(dst + i * 256), 4, voff[i], g * 8 * gs, 0,
                                                     0);
        uint16_t* xd = xring + (size_t)(g % NG) * GP_MT * GP_XS;
#pragma unroll
        for (int j = 0; j < GP_XPW; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (gp_lds_void*)(xd + (wave * GP_XPW + j) * GP_XS), 4, xl,
                                                     xrow[j] + g * 256, 0, 0);
    };
    // the pass with its NMB = ceil(T / 16) row blocks of 16 slots: MFMAs and input fragments of empty blocks
    // are not issued
    auto pass = [&](auto nmb_c) {
        constexpr int NMB = decltype(nmb_c)::value;
        float4v acc[GP_CPW][NMB];
#pragma unroll
        for (int c = 0; c < GP_CPW; ++c)
#pragma unroll
            for (int mb = 0; mb < NMB; ++mb) acc[c][mb] = float4v{ 0.f, 0.f, 0.f, 0.f };
#pragma unroll
        for (int g = 0; g < NG - 1; ++g)
            if (g < ngroups) issue(g);
        for (int g = 0; g < ngroups; ++g)
        {
            if (g + NG - 2 < ngroups) gp_wait_vmcnt<(NG - 2) * NV>();   // this wave's loads of group g landed
            else gp_wait_vmcnt<0>();
            gp_barrier();   // every wave's loads of group g landed; every wave is done with group g - 1
            if (g + NG - 1 < ngroups) issue(g + NG - 1);   // into the slots of group g - 1
            const uint8_t* sl = ring + (g % NG) * GB;
            const uint16_t* xs = xring + (size_t)(g % NG) * GP_MT * GP_XS;
#pragma unroll
            for (int rp = 0; rp < 4; ++rp)
            {
                // the trellis words of this pair of tile rows (the next pair's reads go out under this decode)
                uint32_t wd[GP_CPW][2][2];
#pragma unroll
                for (int c = 0; c < GP_CPW; ++c)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                    {
                        const uint8_t* tp = sl + (2 * rp + h) * RB + c * TB;
                        wd[c][h][0] = *reinterpret_cast<const uint32_t*>(tp + d.o0);
                        wd[c][h][1] = *reinterpret_cast<const uint32_t*>(tp + d.o1);
                    }
                half8 A[NMB];
#pragma unroll
                for (int mb = 0; mb < NMB; ++mb)
                    A[mb] = *reinterpret_cast<const half8*>(xs + (mb * 16 + i16) * GP_XS + q * 32 + rp * 8);
                half8 B[GP_CPW];
#pragma unroll
                for (int c = 0; c < GP_CPW; ++c)
                {
                    const half4 B0 = decode4<K>(wd[c][0][0], wd[c][0][1], d.sh);
                    const half4 B1 = decode4<K>(wd[c][1][0], wd[c][1][1], d.sh);
                    B[c] = half8{ B0[0], B0[1], B0[2], B0[3], B1[0], B1[1], B1[2], B1[3] };
                }
                // raised wave priority while this wave issues its MFMAs: the matrix pipe is refilled as soon as
                // it frees, and the other waves of the SIMD take the VALU slots in between
                __builtin_amdgcn_s_setprio(1);
#pragma unroll
                for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
                    for (int c = 0; c < GP_CPW; ++c)
                        acc[c][mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[mb], B[c], acc[c][mb], 0, 0, 0);
                __builtin_amdgcn_s_setprio(0);
            }
        }
        // D[i][n]: lane holds rows 4q + rr of each 16-slot block, column (t0 + c) * 16 + i16
#pragma unroll
        for (int c = 0; c < GP_CPW; ++c)
#pragma unroll
            for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
                for (int rr = 0; rr < 4; ++rr)
                {
                    const int sl = mb * 16 + q * 4 + rr;
                    if (sl < T)
                        yout[(size_t)(c0 + sl) * a.ndim + (t0 + c) * 16 + i16] = (uint16_t)f2h_bits(acc[c][mb][rr]);
                }
    };
    static_assert(GP_MT == 80, "one case per row-block count");
    switch ((T + 15) / 16)
    {
        case 1: pass(std::integral_constant<int, 1>{}); break;
        case 2: pass(std::integral_constant<int, 2>{}); break;
        case 3: pass(std::integral_constant<int, 3>{}); break;
        case 4: pass(std::integral_constant<int, 4>{}); break;
        default: pass(std::integral_constant<int, 5>{}); break;
    }
}

// The same GEMM for experts with many slots: passes of up to GW_MT, so that a weight is decoded half as often. What bounds
// it: the decode (72 VALU cycles per tile) and the MFMAs (8 per tile and 16 slots) share the SIMD's issue and overlap in
// part. The accumulators take 80 VGPRs; the kernel fits 128 (4 waves per SIMD, two workgroups per CU) with groups of 4 tile
// rows, whose input ring is 40 KB, and one input fragment in flight at a time. The input rows are swizzled instead of
// padded: a load brings two rows, and their 128-byte chunks have to lie next to each other in LDS.
// Measured against passes of 80 (ms per layer, E = 288 top-8, mean slots in brackets): M = 2048 [57] 1.60 -> 1.70, M =
// 2500 [69] 1.76 -> 1.80, M = 2700 [75] 2.00 -> 1.87, M = 4096 [114] 3.07 -> 2.42, M = 5000 [139] 3.43 -> 2.80, M =
// 8192 [228] 5.42 -> 4.86. Passes of 144: 4096 2.41, 5000 3.02, 8192 4.80; of 176 (two registers spilled): 2.43, 2.80,
// 4.99.
constexpr int GW_MT = 160;         // slots per pass (up to 10 MFMA row blocks)
constexpr int GW_GR = 4;           // tile rows per group
constexpr int GW_XPW = GW_MT / 2 / GP_NW;       // pairs of input rows each wave loads per group
constexpr int GW_XROW = GW_GR * 16 * 2;         // input bytes of one slot per group

template <int K>
__global__ __launch_bounds__(GP_NW * 64) __attribute__((amdgpu_waves_per_eu(4))) void gw_gemm_kernel(GemmArgs a)
{
    constexpr int TB = 32 * K, RB = GP_CPW * TB, GB = GW_GR * RB;
    constexpr int NLD = GB / 256;                 // trellis dword loads per lane per group
    static_assert(GB % 256 == 0 && GW_MT % (2 * GP_NW) == 0, "whole wave loads");
    extern __shared__ __align__(16) uint8_t gp_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int nch = a.ndim / GP_WCOLS, per = nch * a.nmat;
    const int xcd = blockIdx.x % 8, j = blockIdx.x / 8;
    const int it = (j / per) * 8 + xcd, rr0 = j % per;
    if (it >= a.nit || it >= a.g.hdr[2]) return;
    const int4 item = a.g.item[it];
    const int e = item.x, c0 = item.y, T = item.z;
    const int nc = rr0 % nch;
    const int mat = a.mat_base + rr0 / nch;
    const int TN = a.ndim / 16, TK = a.kdim / 16, ngroups = TK / GW_GR;
    const int t0 = (nc * GP_NW + wave) * GP_CPW;                     // this wave's first tile column
    uint8_t* ring = gp_lds + wave * 2 * GB;                           // [2][GW_GR tile rows][GP_CPW columns][TB]
    uint8_t* xring = gp_lds + GP_NW * 2 * GB;                         // [2][GW_MT slots][GW_XROW], swizzled
    const uint8_t* tr = reinterpret_cast<const uint8_t*>(a.ptrs[(size_t)e * 9 + mat]);
    const size_t gstride = (size_t)TN * TB;                           // bytes per tile row of the matrix
    uint8_t* cb = const_cast<uint8_t*>(uniform_ptr(tr + (size_t)t0 * TB));
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(cb, (short)0, (int)((size_t)TK * gstride),
                                                                        0x00020000);
    const int gs = (int)gstride;
    int voff[NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i)
    {
        const int byte = i * 256 + lane * 4;   // within the group's [GW_GR][GP_CPW][TB] block
        voff[i] = (byte / RB) * gs + (byte % RB);
    }
    const LaneDec d = lane_dec(lane, K);
    const uint16_t* xin = a.xin + (size_t)(mat - a.mat_base) * a.cap * a.kdim;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(uniform_ptr(reinterpret_cast<const uint8_t*>(xin))), (short)0,
        (int)((size_t)a.cap * a.kdim * 2), 0x00020000);
    uint16_t* yout = a.yout + (size_t)(mat - a.mat_base) * a.cap * a.ndim;
    const int q = lane >> 4, i16 = lane & 15;
    // A load brings the group's chunks of two slots: lane l the 4 bytes at l % 32 of slot row l / 32. The chunk's
    // 16-byte unit 2q + rp (rows 2rp, 2rp + 1 of lane group q) is at byte 64 q + 16 rp of the stored group of 8 tile
    // rows; it lands at unit (2q + rp) ^ (pair % 8), so that the 16 rows of a fragment read lie in different banks.
    const int un = (lane & 31) >> 2;
    const int x1 = (un >> 1) * 64 + (un & 1) * 16 + (lane & 3) * 4;   // a pair whose second slot is past the pass repeats
    const int x2 = x1 + (lane >> 5) * a.kdim * 2;                     // its first
    auto issue = [&](int g) {
        uint8_t* dst = ring + (g & 1) * GB;
#pragma unroll
        for (int i = 0; i < NLD; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (gp_lds_void*)(dst + i * 256), 4, voff[i], g * GW_GR * gs, 0, 0);
        uint8_t* xd = xring + (g & 1) * GW_MT * GW_XROW;
#pragma unroll
        for (int k = 0; k < GW_XPW; ++k)
        {
            const int pr = wave + GP_NW * k;   // pair of slots, dealt over the waves
            if (2 * pr < T)
            {
                const int sw = ((pr & 6) << 5) | ((pr & 1) << 4);   // unit pr % 8 as source bytes
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (gp_lds_void*)(xd + pr * 2 * GW_XROW), 4,
                                                         (2 * pr + 1 < T ? x2 : x1) ^ sw,
                                                         (c0 + 2 * pr) * a.kdim * 2 + (g >> 1) * 256 + (g & 1) * 32, 0, 0);
            }
        }
    };
    auto pass = [&](auto nmb_c) {
        constexpr int NMB = decltype(nmb_c)::value;
        float4v acc[GP_CPW][NMB];
#pragma unroll
        for (int c = 0; c < GP_CPW; ++c)
#pragma unroll
            for (int mb = 0; mb < NMB; ++mb) acc[c][mb] = float4v{ 0.f, 0.f, 0.f, 0.f };
        // slot 16 mb + i16 is row i16 % 2 of pair 8 mb + i16 / 2
        const int xr = i16 * GW_XROW + (((2 * q) ^ (i16 >> 1)) << 4);
        issue(0);
        for (int g = 0; g < ngroups; ++g)
        {
            gp_wait_vmcnt<0>();
            gp_barrier();   // every wave's loads of group g landed; every wave is done with group g - 1
            if (g + 1 < ngroups) issue(g + 1);
            const uint8_t* sl = ring + (g & 1) * GB;
            const uint8_t* xs = xring + (g & 1) * GW_MT * GW_XROW;
            half8 B[2][GP_CPW];
            auto dec = [&](int rp, half8 (&o)[GP_CPW]) {
#pragma unroll
                for (int c = 0; c < GP_CPW; ++c)
                {
                    const uint8_t* tp = sl + 2 * rp * RB + c * TB;
                    const half4 B0 = decode4<K>(ld_u32(tp + d.o0), ld_u32(tp + d.o1), d.sh);
                    const half4 B1 = decode4<K>(ld_u32(tp + RB + d.o0), ld_u32(tp + RB + d.o1), d.sh);
                    o[c] = half8{ B0[0], B0[1], B0[2], B0[3], B1[0], B1[1], B1[2], B1[3] };
                }
            };
            // the whole group's decode first, then its MFMAs in one run (decode and MFMAs of each row pair in turn: M = 4096
            // 2.38 ms against 2.31)
            dec(0, B[0]);
            dec(1, B[1]);
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int rp = 0; rp < GW_GR / 2; ++rp)
#pragma unroll
                for (int mb = 0; mb < NMB; ++mb)
                {
                    const half8 A = *reinterpret_cast<const half8*>(xs + mb * 16 * GW_XROW + (xr ^ (rp << 4)));
#pragma unroll
                    for (int c = 0; c < GP_CPW; ++c)
                        acc[c][mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, B[rp][c], acc[c][mb], 0, 0, 0);
                }
            __builtin_amdgcn_s_setprio(0);
        }
#pragma unroll
        for (int c = 0; c < GP_CPW; ++c)
#pragma unroll
            for (int mb = 0; mb < NMB; ++mb)
#pragma unroll
                for (int rr = 0; rr < 4; ++rr)
                {
                    const int sl = mb * 16 + q * 4 + rr;
                    if (sl < T)
                        yout[(size_t)(c0 + sl) * a.ndim + (t0 + c) * 16 + i16] = (uint16_t)f2h_bits(acc[c][mb][rr]);
                }
    };
    static_assert(GW_MT == 160, "one case per row-block count");
    switch ((T + 15) / 16)
    {
        case 1: pass(std::integral_constant<int, 1>{}); break;
        case 2: pass(std::integral_constant<int, 2>{}); break;
        case 3: pass(std::integral_constant<int, 3>{}); break;
        case 4: pass(std::integral_constant<int, 4>{}); break;
        case 5: pass(std::integral_constant<int, 5>{}); break;
        case 6: pass(std::integral_constant<int, 6>{}); break;
        case 7: pass(std::integral_constant<int, 7>{}); break;
        case 8: pass(std::integral_constant<int, 8>{}); break;
        case 9: pass(std::integral_constant<int, 9>{}); break;
        default: pass(std::integral_constant<int, 10>{}); break;
    }
}

// ---------------------------------------------------------------------------------------------------------------
// EXACT for many slots: the reference's accumulator chains, each weight decoded once per pass of an expert's slots
// ---------------------------------------------------------------------------------------------------------------
//
// The reference's EXACT sum (tile_accum<M,EXACT>, ft_core.h:313-345) gives every output column n four fp32
// accumulators; accumulator j takes, in each tile row tk, the products of rows 2q + {0, 1, 8, 9}[j] for q = 0..3, in
// that order, tile rows ascending, and the four are reduced (a0 + a1) + (a2 + a3) (gemv_block, ft_core.h:377-386).
// Here each chain step runs on the matrix cores. v_mfma_f32_16x16x1_4b_f32 computes four independent 16x16 rank-1
// updates D_b = C_b + A_b B_b^T with K = 1. Per element that is one product added to one accumulator, and both
// operands are fp16 values, so the product is exact in fp32 and D = RN(C + A B) = fmaf(A, B, C), the reference's
// chain step. v_mfma_f32_4x4x1_16b_f32 does the same for sixteen 4x4 blocks. Probes on MI355X matched both with fmaf bit
// for bit on millions of elements (zeros, signed zeros and near-cancelling sums included).
//   - Weights: a lane decodes four consecutive stream indices of a tile (decode4: column n, step q, chains 0..3), as the
//     decode kernels do, and the transposing fp16 MFMA (a 0/1 permutation, exact) turns them into chain j's four steps of
//     column n in lane 16j + n, as fp32. Decoding the lane's own four steps from four windows instead took 8 LDS reads and
//     22 VALU instructions per tile (four funnel shifts, four conversions to fp32) against 2 and 15, and no fp32 MFMA
//     hides VALU issue. With the groups of four below: M = 2048 layer 8.26 -> 7.36 ms, M = 333 2.42 -> 2.08 ms.
//   - Whole blocks of 16 slots, 16x16x1: B is the weight register, A lane 16j + m holds slot m's input for chain j at
//     step q (one ds_read_b128 per lane gives q = 0..3); chain j of (slot 4 (l / 16) + i, column l % 16) is register
//     4j + i of lane l, and the reduction is four registers of one lane.
//   - The slots past them: groups of four by 4x4x1 with the same two registers (cbsz = 2, abid = s: each chain's four
//     blocks of 4 columns take A from its slots 4s..4s+3), then up to two single slots as v_fmac_f32 chains. A group
//     costs 37 cycles of the SIMD per tile, a single slot 12 and a block of 16 128: a remainder of 13 to 15 slots is a
//     padded block, 3, 7 and 11 are padded groups. Each remainder has a loop of its own: with the groups and single
//     slots under branches inside one loop, the reads and decodes of a tile row could not move across them
//     (M = 64 decode call 1151 -> 1087 us, M = 2048 7364 -> 7128 us).
// A wave takes one tile column (16 outputs) with its 4 chains for every slot of the pass. Every accumulator is one chain
// of fused multiply-adds in the reference's order, so the results are bit-identical to the decode path's.
//
// What bounds it: issue. Per tile about 80 cycles of VALU decode plus 8 cycles per slot of fp32 MFMA, which do not
// overlap (the fp32 MFMA holds the SIMD's FMA units). Counters of the gate|up launch, shares of the SIMDs' cycles with the
// MFMAs busy / issuing other VALU / both: 64-slot passes (M = 2048, 57 slots per expert) 78 / 14 / 2%, 32-slot ones (M = 333,
// 3 of 4 picks held) 48 / 40 / 6%, 16-slot ones (M = 64) 26 / 76 / 10%; 8-18% are neither.

constexpr int XG_NW = 8;                    // waves per workgroup: 8 tile columns share one input ring
constexpr int XG_MS = 64;                   // most slots per pass (xg_slots picks 16, 32 or 64 for a call)
constexpr int XG_COLS = 16 * XG_NW;         // output columns per workgroup (a tile column per wave)
constexpr int XG_TC = XG_COLS / 16;         // tile columns per workgroup
constexpr int XG_NG = 2;                    // ring depth (groups of 8 tile rows)
constexpr int XG_XROW = 8 * 16 * 4;         // input bytes of one slot per group: 8 tile rows x 16 rows x fp32
typedef float xg_acc __attribute__((ext_vector_type(16)));   // one 16-slot block of a wave's 4 x 16 x 16 accumulators

struct XgArgs
{
    const uint64_t* ptrs;
    int mat_base, nmat;        // first matrix of the launch (0 gate, 1 up, 2 down) and how many
    int kdim, ndim, cap, nit;  // nit: items the grid covers
    GPlan g;
    const float* xin;          // [mats][cap][kdim] fp32 (fp16-valued), accumulator-chain layout
    uint16_t* yout;            // [mats][cap][ndim] fp16: out_block's leading r16 (ft_core.h:109) applied here
};

// Grid: 8 * ceil(items / 8) * (ndim / XG_COLS) * matrices, XCD-major as the MFMA GEMM. Workgroup = XG_NW waves x 16
// columns (a tile column each, all 4 chains) of one matrix for one item, a pass of up to MS slots of an expert. Per group
// of 8 tile rows the trellis of the XG_TC tile columns and the pass's inputs arrive by LDS-direct loads one group ahead
// (one workgroup barrier per group); at the end each lane reduces its outputs' 4 chains.
// Input rows are swizzled by the loads' source addresses: the 16-byte unit u of slot m's row chunk lands at unit
// u ^ (m % 8), so that the 16 slots a fragment read takes at one unit lie in different banks (row stride 512 bytes).
// Occupancy: the accumulators take MS VGPRs, so 16-, 32- and 64-slot passes fit 64, 80 and 128 registers (8, 6 and 4
// waves per SIMD, 4, 3 and 2 workgroups per CU), with nothing spilled as long as the trellis loads' addresses are scalar: a
// register per load left seven of the twelve instantiations 2 to 5 short, reloaded inside the loops at K = 4 and 5 (4/4/4
// bits, M = 64 1148 -> 1108 us, M = 128 1558 -> 1499, M = 333 2300 -> 2216; 3 bits M = 333 2186 -> 2151, others equal). LDS:
// 4 K + MS KB a workgroup, so all of these fit but K = 5 at 64 slots, which has one workgroup per CU (xg_slots). With few
// slots the loop lives from other waves' issue slots: M = 64 decode call, 16-slot passes at 6 and 8 waves 1087 and 1073 us,
// 32-slot ones at 4 and 6 waves 1263 and 1098 us.
template <int K, int MS>
__global__ __launch_bounds__(XG_NW * 64) __attribute__((amdgpu_waves_per_eu(MS >= 64 ? 4 : MS >= 32 ? 6 : 8))) void
xg_gemm_kernel(XgArgs a)
{
    constexpr int TB = 32 * K, RB = XG_TC * TB, GB = 8 * RB, NG = XG_NG, XGB = MS * XG_XROW;
    constexpr int NLD = RB / 256;              // trellis dword loads per lane per group: wave r brings tile row r
    constexpr int RPW = MS / XG_NW;            // input rows each wave loads per group
    static_assert(XG_NW == 8 && RB % 256 == 0, "a tile row of the group is whole loads of one wave");
    extern __shared__ __align__(16) uint8_t xg_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int nch = a.ndim / XG_COLS, per = nch * a.nmat;
    const int xcd = blockIdx.x % 8, jb = blockIdx.x / 8;
    const int it = (jb / per) * 8 + xcd, rr0 = jb % per;
    if (it >= a.nit || it >= a.g.hdr[2]) return;
    const int4 item = a.g.item[it];
    const int e = item.x, c0 = item.y, T = item.z;
    const int nc = rr0 % nch;
    const int mat = a.mat_base + rr0 / nch;
    const int TN = a.ndim / 16, TK = a.kdim / 16, ngroups = TK / 8;
    uint8_t* tring = xg_lds;                                   // [NG][8 tile rows][XG_TC tile columns][TB]
    uint8_t* xring = xg_lds + NG * GB;                         // [NG][MS slots][8 tile rows][4 chains][4] fp32, swizzled
    const uint8_t* tr = reinterpret_cast<const uint8_t*>(a.ptrs[(size_t)e * 9 + mat]);
    const int gs = TN * TB;                                    // bytes per tile row of the matrix
    uint8_t* cb = const_cast<uint8_t*>(uniform_ptr(tr + (size_t)nc * XG_TC * TB));
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(cb, (short)0, (int)((size_t)TK * gs),
                                                                        0x00020000);
    const float* xin = a.xin + (size_t)(mat - a.mat_base) * a.cap * a.kdim;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(uniform_ptr(reinterpret_cast<const uint8_t*>(xin))), (short)0,
        (int)((size_t)a.cap * a.kdim * 4), 0x00020000);
    uint16_t* yout = a.yout + (size_t)(mat - a.mat_base) * a.cap * a.ndim;
    // chain j of column n of the wave's tile column
    const int j = lane >> 4, n = lane & 15;
    const LaneDec d = lane_dec(lane, K);
    half4 Pm;
#pragma unroll
    for (int r = 0; r < 4; ++r) Pm[r] = (_Float16)((j == (n & 3) && r == (n >> 2)) ? 1.0f : 0.0f);
    const float4v zero = { 0.f, 0.f, 0.f, 0.f };
    // byte of unit 4 c + j (tile row c of 4, chain j) of slot n's row chunk, stored at unit (4 c + j) ^ (n % 8)
    int xu[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) xu[c] = n * XG_XROW + (((4 * c + j) ^ (n & 7)) << 4);

    auto issue = [&](int g, int nsl) {
        uint8_t* dst = tring + (g % NG) * GB;
#pragma unroll
        for (int i = 0; i < NLD; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (gp_lds_void*)(dst + (wave * NLD + i) * 256), 4, lane * 4,
                                                     (g * 8 + wave) * gs + i * 256, 0, 0);
        // this wave's RPW slot rows of the group (rows of slots past the pass repeat its last slot); the lane's source
        // unit is permuted so that the row's 16-byte units land swizzled
        uint8_t* xd = xring + (g % NG) * XGB;
        if (wave * RPW < nsl)
        {
#pragma unroll
            for (int r = 0; r < RPW; ++r)
            {
                const int sl = wave * RPW + r;
                const int srow = (c0 + min(sl, T - 1)) * a.kdim * 4 + g * XG_XROW;
                const int vo = (((lane >> 2) ^ (sl & 7)) << 4) + (lane & 3) * 4;
#pragma unroll
                for (int h = 0; h < XG_XROW / 256; ++h)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (gp_lds_void*)(xd + sl * XG_XROW + h * 256), 4,
                                                             h * 256 + vo, srow, 0, 0);
            }
        }
    };
    // NB blocks of 16 slots, then NQ groups of 4 and NV single slots
    auto pass = [&](auto nb_c, auto nq_c, auto nv_c) {
        constexpr int NB = decltype(nb_c)::value, NQ = decltype(nq_c)::value, NV = decltype(nv_c)::value;
        constexpr int NSL = 16 * NB;
        xg_acc acc[NB > 0 ? NB : 1];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[b][r] = 0.f;
        float4v qacc[NQ > 0 ? NQ : 1];
        float racc[NV > 0 ? NV : 1];
#pragma unroll
        for (int m = 0; m < NQ; ++m) qacc[m] = zero;
#pragma unroll
        for (int m = 0; m < NV; ++m) racc[m] = 0.f;
        issue(0, T);
        for (int g = 0; g < ngroups; ++g)
        {
            gp_wait_vmcnt<0>();
            gp_barrier();   // group g landed for every wave; every wave is done with group g - 1
            if (g + 1 < ngroups) issue(g + 1, T);
            const uint8_t* tl = tring + (g % NG) * GB + wave * TB;
            const uint8_t* xl = xring + (g % NG) * XGB;
#pragma unroll
            for (int t8 = 0; t8 < 8; ++t8)
            {
                const uint8_t* tp = tl + t8 * RB;
                const uint32_t hi = *reinterpret_cast<const uint32_t*>(tp + d.o0);
                const uint32_t lo = *reinterpret_cast<const uint32_t*>(tp + d.o1);
                const float4v w = __builtin_amdgcn_mfma_f32_16x16x16f16(Pm, decode4<K>(hi, lo, d.sh), zero, 0, 0, 0);
                const uint8_t* xt = xl + (t8 >> 2) * 256 + xu[t8 & 3];
                float4 xv[NB > 0 ? NB : 1];
#pragma unroll
                for (int b = 0; b < NB; ++b) xv[b] = *reinterpret_cast<const float4*>(xt + b * 16 * XG_XROW);
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    acc[b] = __builtin_amdgcn_mfma_f32_16x16x1f32(xv[b].x, w[0], acc[b], 0, 0, 0);
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    acc[b] = __builtin_amdgcn_mfma_f32_16x16x1f32(xv[b].y, w[1], acc[b], 0, 0, 0);
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    acc[b] = __builtin_amdgcn_mfma_f32_16x16x1f32(xv[b].z, w[2], acc[b], 0, 0, 0);
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    acc[b] = __builtin_amdgcn_mfma_f32_16x16x1f32(xv[b].w, w[3], acc[b], 0, 0, 0);
                if constexpr (NQ > 0)
                {
                    const float4 xq = *reinterpret_cast<const float4*>(xt + NSL * XG_XROW);
                    const float xs[4] = { xq.x, xq.y, xq.z, xq.w };
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                    {
                        qacc[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(xs[q], w[q], qacc[0], 2, 0, 0);
                        if constexpr (NQ > 1)
                            qacc[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(xs[q], w[q], qacc[1], 2, 1, 0);
                        if constexpr (NQ > 2)
                            qacc[2] = __builtin_amdgcn_mfma_f32_4x4x1f32(xs[q], w[q], qacc[2], 2, 2, 0);
                    }
                }
#pragma unroll
                for (int m = 0; m < NV; ++m)
                {
                    constexpr int S0 = NSL + 4 * NQ;
                    const float4 x4 = *reinterpret_cast<const float4*>(
                        xl + (t8 >> 2) * 256 + (S0 + m) * XG_XROW + (((4 * (t8 & 3) + j) ^ ((S0 + m) & 7)) << 4));
                    racc[m] = __builtin_fmaf(x4.x, w[0], racc[m]);
                    racc[m] = __builtin_fmaf(x4.y, w[1], racc[m]);
                    racc[m] = __builtin_fmaf(x4.z, w[2], racc[m]);
                    racc[m] = __builtin_fmaf(x4.w, w[3], racc[m]);
                }
            }
        }
        // chain c of (slot 16 b + 4 (lane / 16) + i, column lane % 16) is register 4c + i of acc[b]: the
        // reference's (a0 + a1) + (a2 + a3), rounded to fp16 (out_block's leading r16)
        const int col = nc * XG_COLS + wave * 16 + n;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                const int s = 16 * b + 4 * j + i;
                const float y = (acc[b][i] + acc[b][4 + i]) + (acc[b][8 + i] + acc[b][12 + i]);
                if (s < T) yout[(size_t)(c0 + s) * a.ndim + col] = (uint16_t)f2h_bits(y);
            }
        auto put = [&](float v, int s) {
            const float a1 = __shfl(v, n + 16), a2 = __shfl(v, n + 32), a3 = __shfl(v, n + 48);
            const float y = (v + a1) + (a2 + a3);
            if (j == 0 && s < T) yout[(size_t)(c0 + s) * a.ndim + col] = (uint16_t)f2h_bits(y);
        };
#pragma unroll
        for (int m = 0; m < NQ; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) put(qacc[m][i], NSL + 4 * m + i);
#pragma unroll
        for (int m = 0; m < NV; ++m) put(racc[m], NSL + 4 * NQ + m);
    };
    // T slots: nb whole blocks of 16, then a remainder of R <= 12 as groups of four and single slots (13 to 15 fill
    // one more block)
    const int R = T % 16 > 12 ? 0 : T % 16, nb = (T - R + 15) / 16;
    auto n0 = std::integral_constant<int, 0>{};
    auto n1 = std::integral_constant<int, 1>{};
    auto n2 = std::integral_constant<int, 2>{};
    auto n3 = std::integral_constant<int, 3>{};
    auto rest = [&](auto nb_c) {
        switch (R)
        {
            case 0:
                if constexpr (decltype(nb_c)::value > 0) pass(nb_c, n0, n0);
                break;
            case 1: pass(nb_c, n0, n1); break;
            case 2: pass(nb_c, n0, n2); break;
            case 3:
            case 4: pass(nb_c, n1, n0); break;
            case 5: pass(nb_c, n1, n1); break;
            case 6: pass(nb_c, n1, n2); break;
            case 7:
            case 8: pass(nb_c, n2, n0); break;
            case 9: pass(nb_c, n2, n1); break;
            case 10: pass(nb_c, n2, n2); break;
            default: pass(nb_c, n3, n0); break;
        }
    };
    if (nb == MS / 16) pass(std::integral_constant<int, MS / 16>{}, n0, n0);
    else if (nb == 0) rest(n0);
    if constexpr (MS > 16)
        if (nb == 1) rest(n1);
    if constexpr (MS > 32)
    {
        if (nb == 2) rest(n2);
        else if (nb == 3) rest(n3);
    }
}

// ---------------------------------------------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------------------------------------------

template <int K>
static size_t gp_gemm_lds()
{
    return (size_t)GP_NW * GP_NG * 8 * GP_CPW * 32 * K + (size_t)GP_NG * GP_MT * GP_XS * 2;
}

template <int K>
static int gp_gemm_launch(const GemmArgs& a, int nmat, hipStream_t st)
{
    const size_t lds = gp_gemm_lds<K>();
    // opened to what the kernel needs once per process (thread-safe static initialisation)
    static const bool opened = hipFuncSetAttribute(reinterpret_cast<const void*>(gp_gemm_kernel<K>),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
    if (!opened) return -1;
    GemmArgs b = a;
    b.nmat = nmat;
    const unsigned grid = (unsigned)(((a.nit + 7) / 8) * 8 * (a.ndim / GP_WCOLS) * nmat);
    hipLaunchKernelGGL(gp_gemm_kernel<K>, dim3(grid), dim3(GP_NW * 64), lds, st, b);
    return 0;
}

template <int K>
static int gw_gemm_launch(const GemmArgs& a, int nmat, hipStream_t st)
{
    constexpr size_t lds = (size_t)GP_NW * 2 * GW_GR * GP_CPW * 32 * K + (size_t)2 * GW_MT * GW_XROW;
    static const bool opened = hipFuncSetAttribute(reinterpret_cast<const void*>(gw_gemm_kernel<K>),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
    if (!opened) return -1;
    GemmArgs b = a;
    b.nmat = nmat;
    const unsigned grid = (unsigned)(((a.nit + 7) / 8) * 8 * (a.ndim / GP_WCOLS) * nmat);
    hipLaunchKernelGGL(gw_gemm_kernel<K>, dim3(grid), dim3(GP_NW * 64), lds, st, b);
    return 0;
}

// Slots per pass of an MFMA call of P picks (skipped ones included) over E experts: passes of GP_MT while an expert's mean
// share fits one with room for its spread (measured at gw_gemm_kernel).
static int gp_slots(int P, int E) { return P < 72 * E ? GP_MT : GW_MT; }

template <int K>
static int gp_gemm_k(int mt, const GemmArgs& a, int nmat, hipStream_t st)
{
    return mt == GW_MT ? gw_gemm_launch<K>(a, nmat, st) : gp_gemm_launch<K>(a, nmat, st);
}

static int gp_gemm(int K, int mt, const GemmArgs& a, int nmat, hipStream_t st)
{
    switch (K)
    {
        case 2: return gp_gemm_k<2>(mt, a, nmat, st);
        case 3: return gp_gemm_k<3>(mt, a, nmat, st);
        case 4: return gp_gemm_k<4>(mt, a, nmat, st);
        case 5: return gp_gemm_k<5>(mt, a, nmat, st);
        default: return -1;
    }
}

template <int K, int MS>
static int xg_gemm_launch(const XgArgs& a, int nmat, hipStream_t st)
{
    constexpr size_t lds = (size_t)XG_NG * 8 * XG_TC * 32 * K + (size_t)XG_NG * MS * XG_XROW;
    static const bool opened = hipFuncSetAttribute(reinterpret_cast<const void*>(xg_gemm_kernel<K, MS>),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
    if (!opened) return -1;
    XgArgs b = a;
    b.nmat = nmat;
    const unsigned grid = (unsigned)(((a.nit + 7) / 8) * 8 * (a.ndim / XG_COLS) * nmat);
    hipLaunchKernelGGL((xg_gemm_kernel<K, MS>), dim3(grid), dim3(XG_NW * 64), lds, st, b);
    return 0;
}

// Slots per pass of a call of P picks (skipped ones included: the host does not see them) over E experts: 16 below 8
// picks per expert, 32 below 28, else 64. A smaller pass leaves more waves per SIMD, a larger one decodes an expert's
// weights less often. Measured at E = 288, top-8, 3 bits (ms per layer with 16 / 32 / 64; P / E in brackets): M = 64
// [1.8] 1.05 / 1.07 / 1.27, M = 333 [9.3] 1.62 / 1.64 / 1.80, M = 500 [14] 2.75 / 2.59 / 2.77, M = 700 [19] 3.71 / 3.12
// / 3.35, M = 1024 [28] 5.05 / 4.21 / 4.22, M = 2048 [57] 9.39 / 7.84 / 7.07.
// With 5 bits a 64-slot pass takes 84 KB of LDS, one workgroup per CU (2 waves per SIMD): where all three matrices have
// 5, 32 slots from 28 picks on too, and where two have, below 48 picks (64 -> 32 slots, ms; bits gate/up/down): 5/5/5 M
// = 1024 5.55 -> 4.56, M = 1500 6.83 -> 6.54, M = 2048 8.68 -> 8.34, M = 4096 16.7 -> 15.6, E = 72 M = 300 [33] 1.63 ->
// 1.41, M = 1200 [133] 5.07 -> 4.62, H = 4096 I = 2048 M = 2048 9.26 -> 8.78; 5/5/3 M = 1024 5.14 -> 4.40, M = 1500
// [42] 6.45 -> 6.40, M = 2048 8.13 -> 8.13 and 8.13 -> 8.22, M = 4096 [114] 15.8 -> 15.5; 5/2/5 M = 1024 5.26 -> 4.41,
// M = 1500 6.56 -> 6.43, M = 2048 8.24 -> 8.17 and 8.21 -> 8.21. With one matrix of 5 bits 64 stays: 3/3/5 M = 1500
// 5.99 -> 6.33, M = 2048 7.72 -> 8.08, M = 4096 15.1 -> 15.4 (but M = 1024 4.72 -> 4.37); 3/5/4 M = 2048 7.74 -> 8.13.
// A rank that holds 72 of 288 experts and skips the other picks (us with 16 / 32 / 64): M = 64 [7.1] 316 / 318 / 363, M
// = 128 [14] 412 / 421 / 467, M = 333 [37] 612 / 616 / 651, M = 1024 [114] 1368 / 1162 / 1148, M = 2048 [228] 2506 /
// 2109 / 1900; all 288 registered and 3 of 4 picks skipped: M = 128 [3.6] 733 / 767 / 895, M = 333 1269 / 1281 / 1415,
// M = 1024 [28] 1982 / 1972 / 2102, M = 2048 [57] 2927 / 2673 / 2823: the size chosen is up to 7% from the best of the
// three.
static int xg_slots(int P, int E, int Kg, int Ku, int Kd)
{
    const int five = (Kg == 5) + (Ku == 5) + (Kd == 5);
    return P < 8 * E ? 16 : P < 28 * E || five == 3 || (five == 2 && P < 48 * E) ? 32 : XG_MS;
}

template <int K>
static int xg_gemm_k(int ms, const XgArgs& a, int nmat, hipStream_t st)
{
    return ms == 16   ? xg_gemm_launch<K, 16>(a, nmat, st)
           : ms == 32 ? xg_gemm_launch<K, 32>(a, nmat, st)
                      : xg_gemm_launch<K, XG_MS>(a, nmat, st);
}

static int xg_gemm(int K, int ms, const XgArgs& a, int nmat, hipStream_t st)
{
    switch (K)
    {
        case 2: return xg_gemm_k<2>(ms, a, nmat, st);
        case 3: return xg_gemm_k<3>(ms, a, nmat, st);
        case 4: return xg_gemm_k<4>(ms, a, nmat, st);
        case 5: return xg_gemm_k<5>(ms, a, nmat, st);
        default: return -1;
    }
}

void launch_grouped_plan(const uint64_t* ptrs, const int64_t* sel, const void* w, int w_half, int P, int topk, int E,
                         int mt, const GPlan& g, hipStream_t st)
{
    const int M = P / topk;
    const unsigned nch = (unsigned)((P + GP_PLAN_CHUNK - 1) / GP_PLAN_CHUNK);
    if (nch == 1)
    {
        hipLaunchKernelGGL(gp_plan_kernel, dim3(1), dim3(GP_PLAN_THREADS), 0, st, ptrs, sel, w, w_half, P, topk, E, mt, g);
        return;
    }
    hipLaunchKernelGGL(gp_rank_kernel, dim3(nch), dim3(GP_PLAN_THREADS), 0, st, sel, P, E, g);
    hipLaunchKernelGGL(gp_place_kernel, dim3(nch), dim3(GP_PLAN_THREADS), 0, st, sel, P, E, mt, g);
    const int toks = GP_ORDER_THREADS / topk;
    hipLaunchKernelGGL(gp_order_kernel, dim3((unsigned)((M + toks - 1) / toks)), dim3(GP_ORDER_THREADS), 0, st, ptrs, w,
                       w_half, M, topk, g);
}

// Waves per slot of the input transform: one where the slots alone make about 4 waves per SIMD, else up to one per chunk
// of blocks.
static int prep_parts(int P, int H)
{
    const int most = (H / 128 + 4 * GP_TU - 1) / (4 * GP_TU);
    return std::max(1, std::min(most, 4096 / P));
}

template <bool XL, int TA>
static void act_launch_ta(const uint64_t* ptrs, int P, int I, int cap, const GPlan& g, const uint16_t* ygu,
                          const float* silu_tab, float act_limit, void* xd, hipStream_t st)
{
    const long items = (long)P * ((I / 128 + 4 * TA - 1) / (4 * TA));
    hipLaunchKernelGGL((gp_act_kernel<XL, TA>), dim3((unsigned)((items + GP_TW - 1) / GP_TW)), dim3(GP_TW * 64), 0, st,
                       ptrs, I, cap, g, ygu, silu_tab, act_limit, xd);
}

template <bool XL>
static void act_launch(const uint64_t* ptrs, int P, int I, int cap, const GPlan& g, const uint16_t* ygu,
                       const float* silu_tab, float act_limit, void* xd, hipStream_t st)
{
    if (P <= GP_SMALL) act_launch_ta<XL, 1>(ptrs, P, I, cap, g, ygu, silu_tab, act_limit, xd, st);
    else if (P < GL_MIN) act_launch_ta<XL, GP_TA>(ptrs, P, I, cap, g, ygu, silu_tab, act_limit, xd, st);
    else
        hipLaunchKernelGGL(gl_act_kernel<XL>, dim3(GL_CUS), dim3(GL_NW * 64), 0, st, ptrs, I, cap, g, ygu, silu_tab,
                           act_limit, xd);
}

static void comb_launch(int H, int M, int topk, const GPlan& g, const uint16_t* yraw, float* out, hipStream_t st)
{
    const long items = (long)M * ((H / 128 + 3) / 4);
    hipLaunchKernelGGL(gp_comb_kernel, dim3((unsigned)((items + GP_TW - 1) / GP_TW)), dim3(GP_TW * 64), 0, st, H, M,
                       topk, g, yraw, out);
}

int launch_grouped(const uint64_t* ptrs, const int64_t* sel, const void* w, int w_half, int P, int topk, int E, int H,
                   int I, int Kg, int Ku, int Kd, const uint16_t* x, const GPlan& g, int cap, uint16_t* xt,
                   uint16_t* ygu, uint16_t* xd, uint16_t* yraw, const float* silu_tab, float act_limit, float* out,
                   hipStream_t st)
{
    const int M = P / topk;
    const int mt = gp_slots(P, E);
    launch_grouped_plan(ptrs, sel, w, w_half, P, topk, E, mt, g, st);
    const int parts = prep_parts(P, H);
    // inputs of 512 MB and more, which no cache keeps until the GEMM reads them, are stored non-temporally: H = 4096, M = 8192
    // (1.07 GB) 318 -> 261 us, whole call at H = 5120 4478 -> 4386; of 134 MB 39.4 -> 37.4, of 268 MB 72.0 -> 73.1, whole call
    // of 2,048 tokens at H = 5120 1582 -> 1584
    const auto prep = (long)P * H < (1L << 27) ? gp_prep_kernel<false, false> : gp_prep_kernel<false, true>;
    hipLaunchKernelGGL(prep, dim3((unsigned)(((long)P * parts + GP_TW - 1) / GP_TW)), dim3(GP_TW * 64), 0, st,
                       ptrs, x, H, topk, cap, parts, g,
                       static_cast<void*>(xt));
    GemmArgs a;
    a.ptrs = ptrs; a.kdim = H; a.ndim = I; a.cap = cap; a.nit = gemm_items(P, E, mt); a.g = g; a.xin = xt; a.yout = ygu;
    if (Kg == Ku)
    {
        a.mat_base = 0;
        if (gp_gemm(Kg, mt, a, 2, st)) return -1;
    }
    else
    {
        a.mat_base = 0;
        if (gp_gemm(Kg, mt, a, 1, st)) return -1;
        GemmArgs b = a;
        b.mat_base = 1;
        b.xin = xt + (size_t)cap * H;
        b.yout = ygu + (size_t)cap * I;
        if (gp_gemm(Ku, mt, b, 1, st)) return -1;
    }
    act_launch<false>(ptrs, P, I, cap, g, ygu, silu_tab, act_limit, xd, st);
    GemmArgs c = a;
    c.mat_base = 2; c.kdim = I; c.ndim = H; c.xin = xd; c.yout = yraw;
    if (gp_gemm(Kd, mt, c, 1, st)) return -1;
    comb_launch(H, M, topk, g, yraw, out, st);
    return 0;
}

int launch_chains_gate_up(const uint64_t* ptrs, const int64_t* sel, const void* w, int w_half, int P, int topk, int E,
                          int H, int I, int Kg, int Ku, int Kd, const uint16_t* x, const GPlan& g, int cap,
                          float* xt, uint16_t* ygu, float* xd, const float* silu_tab, float act_limit, hipStream_t st)
{
    // the chain GEMM addresses its fp32 inputs with 32-bit byte offsets
    if ((size_t)cap * (size_t)(H > I ? H : I) * 4 > (size_t)0x7fffffff) return -1;
    const int ms = xg_slots(P, E, Kg, Ku, Kd);
    launch_grouped_plan(ptrs, sel, w, w_half, P, topk, E, ms, g, st);
    const int parts = prep_parts(P, H);
    hipLaunchKernelGGL((gp_prep_kernel<true, false>), dim3((unsigned)(((long)P * parts + GP_TW - 1) / GP_TW)), dim3(GP_TW * 64), 0, st,
                       ptrs, x, H, topk, cap, parts, g, static_cast<void*>(xt));
    XgArgs a;
    a.ptrs = ptrs; a.kdim = H; a.ndim = I; a.cap = cap; a.nit = gemm_items(P, E, ms); a.g = g; a.xin = xt; a.yout = ygu;
    a.mat_base = 0;
    if (Kg == Ku)
    {
        if (xg_gemm(Kg, ms, a, 2, st)) return -1;
    }
    else
    {
        if (xg_gemm(Kg, ms, a, 1, st)) return -1;
        a.mat_base = 1;
        a.xin = xt + (size_t)cap * H;
        a.yout = ygu + (size_t)cap * I;
        if (xg_gemm(Ku, ms, a, 1, st)) return -1;
    }
    act_launch<true>(ptrs, P, I, cap, g, ygu, silu_tab, act_limit, xd, st);
    return 0;
}

int launch_chains_down(const uint64_t* ptrs, int P, int topk, int E, int H, int I, int Kg, int Ku, int Kd, const GPlan& g,
                       int cap, const float* xd, uint16_t* yraw, float* out, hipStream_t st)
{
    const int ms = xg_slots(P, E, Kg, Ku, Kd);
    XgArgs a;
    a.ptrs = ptrs; a.mat_base = 2; a.kdim = I; a.ndim = H; a.cap = cap; a.nit = gemm_items(P, E, ms); a.g = g;
    a.xin = xd; a.yout = yraw;
    if (xg_gemm(Kd, ms, a, 1, st)) return -1;
    comb_launch(H, P / topk, topk, g, yraw, out, st);
    return 0;
}

size_t grouped_gemm_lds_bytes(int K)
{
    switch (K)
    {
        case 2: return gp_gemm_lds<2>();
        case 3: return gp_gemm_lds<3>();
        case 4: return gp_gemm_lds<4>();
        case 5: return gp_gemm_lds<5>();
        default: return 0;
    }
}

}  // namespace gfl
