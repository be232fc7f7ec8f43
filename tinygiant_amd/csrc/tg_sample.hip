// tg_sample.hip -- temperature / top-p token sampling over a vocabulary of
// logits on the GPU (tinygiant/engine.py:348-357; greedy, :358-359, is the
// argmax of tg_legacy.hip).
//
// The reference samples in numpy:
//   probs = exp((logits - max(logits)) / T);  probs /= sum(probs)
//   order = argsort(probs) descending;  cs = cumsum(probs[order])
//   cutoff = searchsorted(cs, top_p) + 1;  candidates = order[:cutoff]
//   cp = probs[candidates];  cp /= sum(cp);  token = choice(candidates, p=cp)
// where RandomState.choice widens cp to float64, forms cdf = cumsum(cp) /
// cdf[-1], draws one uniform u and takes the first candidate whose cdf value
// exceeds u.  This file computes the same token from the same u, step by
// step in the same arithmetic:
//   z = (l - m) / T in fp32 (correctly rounded division);
//   p = exp(z) as the fp32 rounding of a float64 exp.  numpy's own float32 exp
//       is within 2 ulp of that and differs between CPUs; this build fixes
//       the correctly rounded value;
//   S = np.sum's order: 8192-value buffers added one after another from 0,
//       each buffer by numpy's pairwise recursion (halves rounded down to a
//       multiple of 8 until 128 or fewer values, those by 8 interleaved
//       accumulators combined as ((r0+r1)+(r2+r3))+((r4+r5)+(r6+r7)) and the
//       last n % 8 values added in order; fewer than 8 values in order from 0);
//   q = p / S;  the fp32 running sum of q in descending order, compared in
//       double with top_p (searchsorted widens the float32 sums);
//   the candidates' sum in np.sum's order, cp = q / that sum, the float64
//       running sum of cp, each value divided by the last, first one > u.
// Ties in q are ordered by ascending token id (numpy's default argsort does
// not fix an order for ties).
//
// Launches of one call (one host synchronisation at the end):
//   k_smp_max     per-block max of the logits and a non-finite flag; clears
//                 the histogram
//   k_smp_exp     p
//   k_smp_chunks  one wave per 8192-value buffer: its pairwise sum
//   k_smp_norm    S from the buffer sums; q = p / S; a histogram of q's top
//                 12 bits with counts and exact mass (units of 2^-40)
//   k_smp_final   the fewest top buckets whose mass provably carries the fp32
//                 running sum past top_p (they hold the candidates); when
//                 they hold at most 8192 elements, their keys (descending q,
//                 ascending id) gathered into LDS, sorted by a bitonic network
//                 8 keys per thread, and the ordered sums as block scans
// More candidates (flat distributions, top_p near 1): the host then launches a
// radix sort of every q (k_rs_count, k_rs_place), and k_smp_cut, k_smp_chunks
// and k_smp_draw finish.  top_p >= 1 or NaN with more than 8192 tokens goes
// there at once, without the selection and its wait.
#include <algorithm>

#include "tg_device.h"
#include "tg_internal.h"

namespace tg {

constexpr int SMP_T = 256;
constexpr int PW_LEVELS = 8;   // depth of numpy's pairwise tree over <= 8192 values is 7

TG_DEV uint32_t smp_bucket(float q) {
    const uint32_t b = __float_as_uint(q) >> SMP_BUCKET_SHIFT;
    return b < (uint32_t)SMP_BUCKETS ? b : (uint32_t)SMP_BUCKETS - 1;  // NaN with the sign bit
}
// q in [0, 1] in units of 2^-40, rounded down (exact: a power-of-two scale)
TG_DEV unsigned long long smp_mass(float q) {
    return (q >= 0.0f && q <= 1.0f) ? (unsigned long long)(q * 0x1p40f) : 0ull;
}
// ascending key order = descending q, then ascending id
TG_DEV unsigned long long smp_key(float q, uint32_t id) {
    return ((unsigned long long)(0x7FFFFFFFu - (__float_as_uint(q) & 0x7FFFFFFFu)) << 32) | id;
}
TG_DEV float smp_key_q(unsigned long long k) { return __uint_as_float(0x7FFFFFFFu - (uint32_t)(k >> 32)); }

TG_DEV float rdl(float v, int i) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), i)); }
TG_DEV double rdl(double v, int i) {
    const unsigned long long b = __double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, i);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), i);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// ------------------------------------------------ numpy's pairwise sum
// Base case of numpy's pairwise summation, n <= 128 values v[0..n).
TG_DEV float pw_leaf(const float *v, int n) {
    if (n < 8) {
        float r = 0.0f;
        for (int i = 0; i < n; i++) r = r + v[i];
        return r;
    }
    float r0 = v[0], r1 = v[1], r2 = v[2], r3 = v[3], r4 = v[4], r5 = v[5], r6 = v[6], r7 = v[7];
    const int main = n & ~7;
    for (int i = 8; i < main; i += 8) {
        r0 = r0 + v[i]; r1 = r1 + v[i + 1]; r2 = r2 + v[i + 2]; r3 = r3 + v[i + 3];
        r4 = r4 + v[i + 4]; r5 = r5 + v[i + 5]; r6 = r6 + v[i + 6]; r7 = r7 + v[i + 7];
    }
    float res = ((r0 + r1) + (r2 + r3)) + ((r4 + r5) + (r6 + r7));
    for (int i = main; i < n; i++) res = res + v[i];
    return res;
}

// The recursion's nodes level by level (at most 64 per level for n <= 8192):
// node (start, len) splits into len/2 rounded down to a multiple of 8 and
// the rest while len > 128.  ch = index of the left child in the next level,
// -1 for a leaf.
struct PwTree {
    short st[PW_LEVELS][WAVE], ln[PW_LEVELS][WAVE], ch[PW_LEVELS][WAVE];
    float v[PW_LEVELS][WAVE];
};

// numpy's pairwise sum of v[0..n), 1 <= n <= 8192, by one whole wave (every
// lane returns it).  Leaves are summed one per lane, inner nodes level by
// level from the bottom, each as left + right.
TG_DEV float wave_pw_sum(const float *v, int n, PwTree &t) {
    const int lane = __lane_id();
    int cnt[PW_LEVELS];
    if (lane == 0) { t.st[0][0] = 0; t.ln[0][0] = (short)n; }
    wave_lds_sync();
    int c = 1;
#pragma unroll
    for (int d = 0; d < PW_LEVELS; d++) {
        cnt[d] = c;
        const bool have = lane < c;
        const int s0 = have ? t.st[d][lane] : 0, l0 = have ? t.ln[d][lane] : 0;
        const bool split = have && l0 > 128 && d + 1 < PW_LEVELS;
        const uint64_t m = __ballot(split);
        const int r = __popcll(m & ((1ull << lane) - 1));
        if (split) {
            const int n2 = (l0 >> 1) & ~7;
            t.st[d + 1][2 * r] = (short)s0;
            t.ln[d + 1][2 * r] = (short)n2;
            t.st[d + 1][2 * r + 1] = (short)(s0 + n2);
            t.ln[d + 1][2 * r + 1] = (short)(l0 - n2);
        }
        if (have) t.ch[d][lane] = (short)(split ? 2 * r : -1);
        c = 2 * __popcll(m);
        wave_lds_sync();
    }
#pragma unroll
    for (int d = PW_LEVELS - 1; d >= 0; d--) {
        if (lane < cnt[d]) {
            const int ch = t.ch[d][lane];
            const int dn = d + 1 < PW_LEVELS ? d + 1 : d;  // children exist only above the last level
            const float val = ch < 0 ? pw_leaf(v + t.st[d][lane], t.ln[d][lane])
                                     : t.v[dn][ch] + t.v[dn][ch + 1];
            t.v[d][lane] = val;
        }
        wave_lds_sync();
    }
    return t.v[0][0];
}

// ------------------------------------------------ ordered running sums, in parallel
// The running sum s_k = round(s_{k-1} + v_k) of descending values v_k >= 0
// (fp32, or float64 of fp32 values) is defined by its order; walked by one
// wave, 151,936 of them took 1,230 us in fp32 and two walks 1,690 us in
// float64.  While the sum stays inside one binade [2^e, 2^(e+1)) it is a
// multiple of the binade's ulp, and what a run of additions adds to it depends
// on where it starts only through the parity of that multiple (it decides the
// ties).  So each lane adds its run to 2^e and to 2^e + ulp: the differences
// are what the run adds to an even and to an odd sum, and these pairs compose
// associatively.  A scan over the lanes' pairs gives every lane the exact sum
// before its run, and the lane then makes its own additions from there.  The
// first lane whose sum reaches 2^(e+1) still ends on the true sum (it made
// every addition itself); the lanes after it are scanned again from that sum,
// once per binade.  v_k <= v_0 <= s throughout; pairs past a crossing may be
// inexact and are not used.  The same 151,936 values now take 36 us (fp32 cut)
// and 72 us (float64 draw): one block, bound by its additions and 19 tiles of
// two barriers each.  (Values loaded one dword at a time instead of two float4
// per lane: 95 and 113 us.  Ulps counted as 64-bit integers: 166 and 192 us.)
template <class F> struct Grid;  // the sum's binade as 2^e, its ulp, a value's parity in ulps
template <> struct Grid<float> {
    TG_DEV static float binade(float s) { return __uint_as_float(__float_as_uint(s) & 0x7F800000u); }
    static constexpr float ULP = 0x1p-23f;
    TG_DEV static bool odd(float v) { return __float_as_uint(v) & 1u; }
};
template <> struct Grid<double> {
    TG_DEV static double binade(double s) {
        return __longlong_as_double(__double_as_longlong(s) & 0x7FF0000000000000ll);
    }
    static constexpr double ULP = 0x1p-52;
    TG_DEV static bool odd(double v) { return __double_as_longlong(v) & 1; }
};
// what a run of additions adds to a sum that is an even / odd number of ulps
template <class F> struct Hop { F d0, d1; };
// run a, then run b, in binade c
template <class F> TG_DEV Hop<F> hop_join(F c, const Hop<F> &a, const Hop<F> &b) {
    return {a.d0 + (Grid<F>::odd(c + a.d0) ? b.d1 : b.d0), a.d1 + (Grid<F>::odd(c + a.d1) ? b.d0 : b.d1)};
}
// lanes without a source read 0
template <int CTRL, int ROWS> TG_DEV float dpp_0(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xF, false));
}
template <int CTRL, int ROWS> TG_DEV double dpp_0(double v) {
    const unsigned long long b = __double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROWS, 0xF, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROWS, 0xF, false);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <int CTRL, int ROWS, class F> TG_DEV Hop<F> hop_from(const Hop<F> &v) {
    return {dpp_0<CTRL, ROWS>(v.d0), dpp_0<CTRL, ROWS>(v.d1)};
}
// inclusive scan over groups of 16 lanes, then over the wave ({0, 0} is the identity)
template <class F> TG_DEV Hop<F> hop_scan16(F c, Hop<F> v) {
    v = hop_join(c, hop_from<0x111, 0xF>(v), v);  // row_shr:1
    v = hop_join(c, hop_from<0x112, 0xF>(v), v);  // row_shr:2
    v = hop_join(c, hop_from<0x114, 0xF>(v), v);  // row_shr:4
    v = hop_join(c, hop_from<0x118, 0xF>(v), v);  // row_shr:8
    return v;
}
template <class F> TG_DEV Hop<F> hop_scan(F c, Hop<F> v) {
    v = hop_scan16(c, v);
    v = hop_join(c, hop_from<0x142, 0xA>(v), v);  // row_bcast:15 into rows 1 and 3
    v = hop_join(c, hop_from<0x143, 0xC>(v), v);  // row_bcast:31 into rows 2 and 3
    return v;
}

constexpr int ORD_R = 8;        // values per lane and scan
constexpr int ORD_NW = 16;      // waves of a block scan
constexpr int ORD_HEAD = 1024;  // values summed by one wave first (most of the binades lie there)
constexpr int ORD_TILE = ORD_NW * WAVE * ORD_R;
constexpr int ORD_LOG = 2 + SMP_VMAX / ORD_TILE;
struct OrdLds {
    Hop<double> t[ORD_NW];  // the waves' totals
    double s[ORD_NW];       // per wave, its first event: the sum after that lane's run (no event: after its last),
    int end[ORD_NW];        // that lane's end (INT_MAX: no event)
    int hit[ORD_NW];        // and the index that satisfies the predicate (-1: the binade's end)
    double s0;              // the head's result
    float s2;               // the candidates' sum
    int pos0, pick;
    double log[ORD_LOG];    // the sum before each tile
};

// Continues the running sum s of the values before pos (a multiple of 8; at 0,
// s = v[0] and the sum goes on from v[1]) over v[pos..n) (each divided by div
// when DIV), by NW waves (NW == 1: any one wave; else the whole block of ORD_NW
// waves).  v is 16-byte aligned and readable to the next multiple of 8 values.
// Returns the first index whose running sum satisfies pred (monotone), or -1
// with s the sum of all.  log: the sum before each tile.
template <class F, int NW, bool DIV, class Pred>
TG_DEV int ord_run(const float *v, float div, int n, int pos, F &s, Pred pred, OrdLds &L, double *log) {
    constexpr int TILE = NW * WAVE * ORD_R;
    const int lane = __lane_id(), w = NW == 1 ? 0 : (int)threadIdx.x / WAVE, slot = (w * WAVE + lane) * ORD_R;
    float raw[ORD_R];
    F x[ORD_R];
    // two 16-byte loads, unconditional (at the last group of 8 past the end,
    // whose values are not used), so that they stay in flight during a scan
    auto load = [&](int p0) {
        const float4 *g = reinterpret_cast<const float4 *>(v + min(p0 + slot, (n - 1) & ~(ORD_R - 1)));
        const float4 a = g[0], b = g[1];
        raw[0] = a.x; raw[1] = a.y; raw[2] = a.z; raw[3] = a.w;
        raw[4] = b.x; raw[5] = b.y; raw[6] = b.z; raw[7] = b.w;
    };
    load(pos);
    for (; pos < n; pos += TILE) {
#pragma unroll
        for (int j = 0; j < ORD_R; j++) {
            const int i = pos + slot + j;
            const float q = DIV ? raw[j] / div : raw[j];
            x[j] = i > 0 && i < n ? (F)q : (F)0;
        }
        load(pos + TILE);
        if (NW > 1 && log && threadIdx.x == 0) *log++ = (double)s;
        const int end = min(pos + slot + ORD_R, n);  // of this lane's run
        for (;;) {
            // x: this tile's values not yet in s (those that are, and past n: 0)
            const F c = Grid<F>::binade(s), c1 = c + c * Grid<F>::ULP;
            F a0 = c, a1 = c1;
#pragma unroll
            for (int j = 0; j < ORD_R; j++) {
                a0 = a0 + x[j];
                a1 = a1 + x[j];
            }
            const Hop<F> inc = hop_scan(c, Hop<F>{a0 - c, a1 - c1});
            Hop<F> ex = hop_from<0x138, 0xF>(inc);  // wave_shr:1
            if (NW > 1) {
                if (lane == WAVE - 1) L.t[w] = {(double)inc.d0, (double)inc.d1};
                lds_barrier();  // (the next tile's loads stay in flight)
                const Hop<double> td = L.t[lane & (NW - 1)];
                const Hop<F> ti = hop_scan16(c, Hop<F>{(F)td.d0, (F)td.d1});
                if (w > 0) ex = hop_join(c, Hop<F>{rdl(ti.d0, w - 1), rdl(ti.d1, w - 1)}, ex);
            }
            const F sl = s + (Grid<F>::odd(s) ? ex.d1 : ex.d0);
            F se = sl;
#pragma unroll
            for (int j = 0; j < ORD_R; j++) se = se + x[j];
            const uint64_t m = __ballot(se >= c + c || pred(se));
            int first = WAVE - 1, at = INT_MAX, hit = -1;
            if (m) {
                first = __ffsll((unsigned long long)m) - 1;
                at = __builtin_amdgcn_readlane(end, first);
                F r = sl;
                int k = 0;
#pragma unroll
                for (int j = 0; j < ORD_R; j++) {
                    r = r + x[j];
                    k += pred(r) ? 0 : 1;
                }
                k = __builtin_amdgcn_readlane(k, first);
                if (k < ORD_R) hit = pos + (w * WAVE + first) * ORD_R + k;
            }
            F sn = rdl(se, first);
            if (NW > 1) {
                if (lane == 0) { L.end[w] = at; L.s[w] = (double)sn; L.hit[w] = hit; }
                lds_barrier();
                const uint64_t me = __ballot(lane < NW && L.end[lane & (NW - 1)] != INT_MAX);
                const int fw = me ? __ffsll((unsigned long long)me) - 1 : NW - 1;
                at = L.end[fw];
                sn = (F)L.s[fw];
                hit = L.hit[fw];
            }
            s = sn;
            if (at == INT_MAX) break;  // the whole tile is in s
            if (hit >= 0) return hit;
#pragma unroll
            for (int j = 0; j < ORD_R; j++)
                if (end <= at) x[j] = (F)0;
        }
    }
    return -1;
}

// The running sum of v[0..n) (n >= 1) by a block of ORD_NW waves: its first
// index that satisfies pred, or -1 and s the whole sum.
template <class F, bool DIV, class Pred>
TG_DEV int ord_block(const float *v, float div, int n, F &s, Pred pred, OrdLds &L, double *log) {
    if (threadIdx.x < WAVE) {
        F h = (F)(DIV ? v[0] / div : v[0]);
        int at = 0;
        if (!pred(h)) at = ord_run<F, 1, DIV>(v, div, min(n, ORD_HEAD), 0, h, pred, L, nullptr);
        if (threadIdx.x == 0) { L.s0 = (double)h; L.pos0 = at; }
    }
    __syncthreads();
    s = (F)L.s0;
    const int at = L.pos0;
    if (at >= 0 || n <= ORD_HEAD) return at;
    return ord_run<F, ORD_NW, DIV>(v, div, n, ORD_HEAD, s, pred, L, log);
}

// First k whose float64 running sum of (double)(v[k] / s2), divided by the
// last one, exceeds u (cdf.searchsorted(u, side='right')), by a block of
// ORD_NW waves: the sums of the tiles, then the tile that holds the draw.
TG_DEV int ord_draw(const float *v, int n, float s2, double u, OrdLds &L) {
    double tot;
    ord_block<double, true>(v, s2, n, tot, [](double) { return false; }, L, L.log + 1);
    const int nt = 1 + (n > ORD_HEAD ? (n - ORD_HEAD + ORD_TILE - 1) / ORD_TILE : 0);  // the head, then tiles
    if (threadIdx.x == 0) L.pick = nt - 1;
    __syncthreads();
    for (int t = threadIdx.x; t + 1 < nt; t += ORD_NW * WAVE)
        if (L.log[t + 1] / tot > u) atomicMin(&L.pick, t);
    __syncthreads();
    const int t = L.pick;
    auto hit = [=](double s) { return s / tot > u; };
    double s;
    int at;
    if (t == 0) {
        at = ord_block<double, true>(v, s2, min(n, ORD_HEAD), s, hit, L, nullptr);
    } else {
        const int p0 = ORD_HEAD + (t - 1) * ORD_TILE;
        s = L.log[t];
        at = ord_run<double, ORD_NW, true>(v, s2, min(n, p0 + ORD_TILE), p0, s, hit, L, nullptr);
    }
    return at < 0 ? n - 1 : at;
}

// np.sum of v[0..n) as buffers of 8192 added from 0, by one wave
TG_DEV float wave_np_sum(const float *v, int n, PwTree &t) {
    float s = 0.0f;
    for (int c0 = 0; c0 < n; c0 += NP_BUFSIZE) s = s + wave_pw_sum(v + c0, min(NP_BUFSIZE, n - c0), t);
    return s;
}

// The candidates' draw from their q in descending order (v[0..n), n <= 8192)
// by a block of ORD_NW waves: writes cut and the token drawn.
TG_DEV void block_finish(const float *v, int n, int V, double top_p, double u, PwTree &t, OrdLds &L, SmpCtl *ctl,
                         const uint32_t *ids) {
    float s;
    int cut = ord_block<float, false>(v, 1.0f, n, s, [=](float r) { return (double)r >= top_p; }, L, nullptr);
    if (cut < 0) {
        if (n != V) {  // the selection bound guarantees a crossing inside a strict prefix
            if (threadIdx.x == 0) ctl->status = SMP_ST_BOUND;
            return;
        }
        cut = V;  // searchsorted past the end: every token is a candidate
    } else {
        cut += 1;
    }
    __syncthreads();
    if (threadIdx.x < WAVE) {
        const float s2 = wave_np_sum(v, cut, t);
        if (threadIdx.x == 0) L.s2 = s2;
    }
    __syncthreads();
    const float s2 = L.s2;
    const int pos = ord_draw(v, cut, s2, u, L);
    if (threadIdx.x == 0) {
        ctl->cut = cut;
        ctl->token = (int)ids[pos];
        ctl->status = SMP_ST_OK;
    }
}

// ------------------------------------------------ kernels
__global__ __launch_bounds__(SMP_T) void k_smp_max(const float *__restrict__ l, int V, float *__restrict__ pmax,
                                                   int *__restrict__ pbad, uint32_t *__restrict__ hcnt,
                                                   unsigned long long *__restrict__ hmass, SmpCtl *ctl) {
    const int tid = threadIdx.x, gt = blockIdx.x * SMP_T + tid, gn = gridDim.x * SMP_T;
    for (int b = gt; b < SMP_BUCKETS; b += gn) { hcnt[b] = 0; hmass[b] = 0; }
    if (gt == 0) { ctl->n = 0; ctl->done = 0; ctl->large = 0; ctl->status = SMP_ST_PENDING; ctl->token = -1; ctl->cut = 0; }
    float m = -INFINITY;
    int bad = 0;
    for (int i = gt; i < V; i += gn) {
        const float x = l[i];
        bad |= (x != x) | (x == INFINITY);
        m = fmaxf(m, x);
    }
    for (int s = WAVE / 2; s >= 1; s >>= 1) {
        m = fmaxf(m, __shfl_xor(m, s, WAVE));
        bad |= __shfl_xor(bad, s, WAVE);
    }
    __shared__ float sm[SMP_T / WAVE];
    __shared__ int sb[SMP_T / WAVE];
    if ((tid & (WAVE - 1)) == 0) { sm[tid / WAVE] = m; sb[tid / WAVE] = bad; }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < SMP_T / WAVE; w++) { m = fmaxf(m, sm[w]); bad |= sb[w]; }
        pmax[blockIdx.x] = m;
        pbad[blockIdx.x] = bad;
    }
}

__global__ __launch_bounds__(SMP_T) void k_smp_exp(const float *__restrict__ l, int V, const float *__restrict__ pmax,
                                                   const int *__restrict__ pbad, int nb, float T,
                                                   float *__restrict__ p, SmpCtl *ctl) {
    __shared__ float s_m;
    const int tid = threadIdx.x;
    if (tid < WAVE) {
        float m = -INFINITY;
        int bad = 0;
        for (int b = tid; b < nb; b += WAVE) { m = fmaxf(m, pmax[b]); bad |= pbad[b]; }
        for (int s = WAVE / 2; s >= 1; s >>= 1) {
            m = fmaxf(m, __shfl_xor(m, s, WAVE));
            bad |= __shfl_xor(bad, s, WAVE);
        }
        if (tid == 0) {
            s_m = m;
            if (blockIdx.x == 0) { ctl->m = m; ctl->bad = bad | (m == -INFINITY); }
        }
    }
    __syncthreads();
    const float m = s_m;
    for (int i = blockIdx.x * SMP_T + tid; i < V; i += gridDim.x * SMP_T) {
        const float z = (l[i] - m) / T;
        p[i] = (float)exp((double)z);
    }
}

// One wave per 8192-value buffer of v[0..n): its pairwise sum.  n is the
// argument, or, when n_from_ctl, the candidate count ctl->cut.
__global__ __launch_bounds__(WAVE) void k_smp_chunks(const float *__restrict__ v, int n, int n_from_ctl,
                                                     const SmpCtl *ctl, float *__restrict__ sums) {
    __shared__ PwTree t;
    if (n_from_ctl) {
        if (ctl->status != SMP_ST_PENDING) return;
        n = ctl->cut;
    }
    const int c0 = blockIdx.x * NP_BUFSIZE;
    if (c0 >= n) return;
    const float s = wave_pw_sum(v + c0, min(NP_BUFSIZE, n - c0), t);
    if (threadIdx.x == 0) sums[blockIdx.x] = s;
}

// The candidates lie in the top buckets: with C elements and exact mass M
// (2^-40 units, rounded down per element) in buckets >= b, the fp32 running
// sum over those elements in descending order ends at or above
// M 2^-40 - C 2^-24 (each addition rounds by at most half an ulp of a sum
// below 2), so M 2^-40 >= top_p + C 2^-24 puts the crossing inside them.
// The largest such b is taken; none (top_p near or above 1, or NaN) = all.
// A block of NT threads; the histogram is read at device scope (other
// blocks' atomics).  Leaves bstar and C in ctl.
template <int NT>
TG_DEV void smp_select(const uint32_t *hcnt, const unsigned long long *hmass, int V, double top_p, SmpCtl *ctl) {
    constexpr int PER = SMP_BUCKETS / NT;
    __shared__ uint32_t wc[NT / WAVE];
    __shared__ unsigned long long wm[NT / WAVE];
    __shared__ int s_best;
    __shared__ uint32_t s_C;
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), w = tid / WAVE;
    // descending position d = PER tid + k holds bucket SMP_BUCKETS - 1 - d
    uint32_t c[PER];
    unsigned long long ms[PER];
    uint32_t tc = 0;
    unsigned long long tm = 0;
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const int b = SMP_BUCKETS - 1 - (PER * tid + k);
        c[k] = __hip_atomic_load(hcnt + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        ms[k] = __hip_atomic_load(hmass + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        tc += c[k];
        tm += ms[k];
    }
    uint32_t ic = tc;  // inclusive scan of the thread totals over the wave, then over waves
    unsigned long long im = tm;
    for (int s = 1; s < WAVE; s <<= 1) {
        const uint32_t oc = __shfl_up(ic, s, WAVE);
        const unsigned long long om = __shfl_up(im, s, WAVE);
        if (lane >= s) { ic += oc; im += om; }
    }
    if (lane == WAVE - 1) { wc[w] = ic; wm[w] = im; }
    if (tid == 0) { s_best = INT_MAX; s_C = (uint32_t)V; }
    __syncthreads();
    uint32_t cc = ic - tc;
    unsigned long long cm = im - tm;
    for (int j = 0; j < w; j++) { cc += wc[j]; cm += wm[j]; }
    int best = INT_MAX;
    uint32_t bestC = 0;
#pragma unroll
    for (int k = 0; k < PER; k++) {
        cc += c[k];
        cm += ms[k];
        const double need = (top_p + (double)cc * 0x1p-24) * 0x1p40 + 1024.0;
        if (best == INT_MAX && cc >= 1 && (double)cm >= need) { best = PER * tid + k; bestC = cc; }
    }
    atomicMin(&s_best, best);
    __syncthreads();
    if (best != INT_MAX && best == s_best) s_C = bestC;
    __syncthreads();
    if (tid == 0) {
        const int d = s_best;
        ctl->bstar = d == INT_MAX ? 0 : SMP_BUCKETS - 1 - d;
        ctl->C = d == INT_MAX ? (uint32_t)V : s_C;
    }
}

// q = p / S; SELECT: also the histogram, and the candidate buckets from it
template <bool SELECT>
__global__ __launch_bounds__(SMP_T) void k_smp_norm(const float *__restrict__ p, int V,
                                                    const float *__restrict__ sums, int nchunks, double top_p,
                                                    SmpCtl *ctl, float *__restrict__ q, uint32_t *hcnt,
                                                    unsigned long long *hmass) {
    __shared__ uint32_t lc[SELECT ? SMP_BUCKETS : 1];
    __shared__ unsigned long long lm[SELECT ? SMP_BUCKETS : 1];
    __shared__ float s_S;
    __shared__ int s_last;
    const int tid = threadIdx.x;
    if constexpr (SELECT)
        for (int b = tid; b < SMP_BUCKETS; b += SMP_T) { lc[b] = 0; lm[b] = 0; }
    if (tid == 0) {
        float S = 0.0f;
        for (int c = 0; c < nchunks; c++) S = S + sums[c];
        s_S = S;
        if (blockIdx.x == 0) ctl->S = S;
    }
    __syncthreads();
    const float S = s_S;
    for (int i = blockIdx.x * SMP_T + tid; i < V; i += gridDim.x * SMP_T) {
        const float v = p[i] / S;
        q[i] = v;
        if constexpr (SELECT) {
            const uint32_t b = smp_bucket(v);
            atomicAdd(&lc[b], 1u);
            atomicAdd(&lm[b], smp_mass(v));
        }
    }
    if constexpr (!SELECT) return;
    __syncthreads();
    for (int b = tid; b < SMP_BUCKETS; b += SMP_T)
        if (lc[b]) {
            atomicAdd(&hcnt[b], lc[b]);
            atomicAdd(&hmass[b], lm[b]);
        }
    // the last block to finish picks the candidate buckets
    __threadfence();
    __syncthreads();
    if (tid == 0) s_last = atomicAdd(&ctl->done, 1u) == gridDim.x - 1;
    __syncthreads();
    if (s_last) {
        __threadfence();
        smp_select<SMP_T>(hcnt, hmass, V, top_p, ctl);
    }
}

// Bitonic network, 8 keys per thread: thread t holds keys 8t .. 8t+7 of a
// run whose first key is key g0 of the whole network (g0 a multiple of 8192;
// the direction of stage kk at key i is ascending when (i & kk) == 0).  One
// step (kk, j): j < 8 in registers, 8 <= j < 512 with lane t ^ (j / 8) of the
// same wave, larger through LDS (x, 8 keys per thread).  Every thread of the
// block calls it; threads with 8t >= n hold no keys (n a power of two >= 8).
template <int J>
TG_DEV void bt_reg_step(unsigned long long (&k)[8], uint32_t g, int kk) {
#pragma unroll
    for (int r = 0; r < 8; r++) {
        const int l = r ^ J;
        if (l > r) {
            const bool asc = ((g + (uint32_t)r) & (uint32_t)kk) == 0;
            const unsigned long long a = k[r], b = k[l];
            if ((a > b) == asc) { k[r] = b; k[l] = a; }
        }
    }
}

TG_DEV unsigned long long shfl_xor_u64(unsigned long long v, int m) {
    const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)v, m, WAVE);
    const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(v >> 32), m, WAVE);
    return ((unsigned long long)hi << 32) | lo;
}

TG_DEV unsigned long long bt_pick(unsigned long long a, unsigned long long o, bool keep_min) {
    return keep_min ? (a < o ? a : o) : (a > o ? a : o);
}

TG_DEV void bt_step(unsigned long long (&k)[8], int n, uint32_t g0, int kk, int j, unsigned long long *x) {
    const int t = threadIdx.x;
    const bool act = (t << 3) < n;
    const uint32_t g = g0 + ((uint32_t)t << 3);
    if (j >= 512) {
        if (act) {
#pragma unroll
            for (int r = 0; r < 8; r++) x[(t << 3) + r] = k[r];
        }
        __syncthreads();
        if (act) {
#pragma unroll
            for (int r = 0; r < 8; r++) {
                const int i = (t << 3) + r;
                const bool keep_min = (((g + (uint32_t)r) & (uint32_t)kk) == 0) == ((i & j) == 0);
                k[r] = bt_pick(k[r], x[i ^ j], keep_min);
            }
        }
        __syncthreads();
    } else if (j >= 8) {
        const int m = j >> 3;  // partner lane t ^ m, in the same wave (m < 64)
#pragma unroll
        for (int r = 0; r < 8; r++) {
            const unsigned long long o = shfl_xor_u64(k[r], m);
            const bool keep_min = (((g + (uint32_t)r) & (uint32_t)kk) == 0) == ((t & m) == 0);
            k[r] = bt_pick(k[r], o, keep_min);
        }
    } else if (j == 4) {
        bt_reg_step<4>(k, g, kk);
    } else if (j == 2) {
        bt_reg_step<2>(k, g, kk);
    } else {
        bt_reg_step<1>(k, g, kk);
    }
}

// Ascending sort of n keys (8 <= n <= 8192, a power of two) held 8 per thread.
TG_DEV void bitonic_regs(unsigned long long (&k)[8], int n, unsigned long long *x) {
    for (int kk = 2; kk <= n; kk <<= 1)
        for (int j = kk >> 1; j > 0; j >>= 1) bt_step(k, n, 0, kk, j, x);
}

// The last launch of a call: at most 8192 candidates (keys[0..C) from
// k_smp_compact) sorted in registers and LDS, then the scans by wave 0.
// More candidates: ctl->large for the host.
__global__ __launch_bounds__(1024) void k_smp_final(const unsigned long long *__restrict__ keys, int V,
                                                    double top_p, double u, SmpCtl *ctl) {
    extern __shared__ __align__(16) uint8_t smem[];
    unsigned long long *sk = reinterpret_cast<unsigned long long *>(smem);
    PwTree &t = *reinterpret_cast<PwTree *>(smem + sizeof(unsigned long long) * SMP_SMALL);
    const int tid = threadIdx.x;
    if (ctl->bad) {
        if (tid == 0) ctl->status = SMP_ST_INPUT;
        return;
    }
    const uint32_t C = ctl->C;
    if (C > (uint32_t)SMP_SMALL) {
        if (tid == 0) ctl->large = 1;
        return;
    }
    int P = 8;
    while (P < (int)C) P <<= 1;
    unsigned long long k[8];
#pragma unroll
    for (int r = 0; r < 8; r++) {
        const int i = (tid << 3) + r;
        k[r] = i < (int)C ? keys[i] : ~0ull;
    }
    bitonic_regs(k, P, sk);
    __syncthreads();
    // sorted keys -> q (first half of the array) and ids (second half)
    float *sq = reinterpret_cast<float *>(smem);
    uint32_t *sid = reinterpret_cast<uint32_t *>(smem) + SMP_SMALL;
#pragma unroll
    for (int r = 0; r < 8; r++) {
        const int i = (tid << 3) + r;
        if (i < (int)C) {
            sq[i] = smp_key_q(k[r]);
            sid[i] = (uint32_t)k[r];
        }
    }
    __syncthreads();
    __shared__ OrdLds ord;
    block_finish(sq, (int)C, V, top_p, u, t, ord, ctl, sid);
}

// ------------------------------------------------ more than 8192 candidates
// The candidates' keys (bucket >= ctl->bstar) into keys[0..C): per block a
// count, one global slot range, then the keys.
__global__ __launch_bounds__(SMP_T) void k_smp_compact(const float *__restrict__ q, int V, SmpCtl *ctl,
                                                       unsigned long long *__restrict__ keys) {
    __shared__ uint32_t s_cnt, s_base;
    const uint32_t bstar = (uint32_t)ctl->bstar;
    const int lane = __lane_id();
    if (threadIdx.x == 0) s_cnt = 0;
    __syncthreads();
    for (int i = blockIdx.x * SMP_T + threadIdx.x; i < V; i += gridDim.x * SMP_T)
        if (smp_bucket(q[i]) >= bstar) atomicAdd(&s_cnt, 1u);
    __syncthreads();
    if (threadIdx.x == 0) {
        s_base = atomicAdd(&ctl->n, s_cnt);
        s_cnt = 0;
    }
    __syncthreads();
    for (int i0 = blockIdx.x * SMP_T; i0 < V; i0 += gridDim.x * SMP_T) {
        const int i = i0 + threadIdx.x;
        float v = 0.0f;
        bool take = false;
        if (i < V) {
            v = q[i];
            take = smp_bucket(v) >= bstar;
        }
        const uint64_t m = __ballot(take);
        if (m) {
            const int leader = __ffsll((long long)m) - 1;
            uint32_t base = 0;
            if (lane == leader) base = atomicAdd(&s_cnt, (uint32_t)__popcll(m));
            base = (uint32_t)__shfl((int)base, leader, WAVE);
            if (take) keys[s_base + base + __popcll(m & ((1ull << lane) - 1))] = smp_key(v, (uint32_t)i);
        }
    }
}

// All V probabilities in descending order, ties by ascending id: a stable
// radix sort of 0x3F800000 - bits(q) (q <= 1: 30 bits) in three passes of 10
// bits.  Per pass one launch counts each block's digits (table [block][digit])
// and one places the block's RS_TILE keys: every block sums the table's columns
// itself (no scan launch between), and inside a block a key's rank among its
// equals is its wave's count so far plus its lane's place among the lanes with
// the same digit (one ballot per digit bit).  Bound by the latency of these
// steps, not by its 1.2 MB a pass: at 151,936 values (38 blocks) 2.6-4.5 us to
// count and 12-15 us to place, 53 us in all; the bitonic network it replaces
// took 21 launches and 215 us there, and grew with the next power of two.
constexpr int RS_T = 1024, RS_R = 4, RS_TILE = RS_T * RS_R, RS_BITS = 10, RS_BINS = 1 << RS_BITS;
static_assert(RS_BINS == RS_T, "one digit per thread");
static_assert(SMP_RS_TABLE >= (SMP_VMAX + RS_TILE - 1) / RS_TILE * RS_BINS, "table size");
template <int PASS>
TG_DEV unsigned long long rs_load(const float *q, const unsigned long long *src, int i) {
    if constexpr (PASS == 0) return ((unsigned long long)(0x3F800000u - __float_as_uint(q[i])) << 32) | (uint32_t)i;
    return src[i];
}
template <int PASS>
TG_DEV uint32_t rs_digit(unsigned long long k) { return (uint32_t)(k >> (32 + PASS * RS_BITS)) & (RS_BINS - 1); }

template <int PASS>
__global__ __launch_bounds__(RS_T) void k_rs_count(const float *__restrict__ q,
                                                   const unsigned long long *__restrict__ src, int n,
                                                   uint32_t *__restrict__ table) {
    __shared__ uint32_t h[RS_BINS];
    const int tid = threadIdx.x, i0 = blockIdx.x * RS_TILE;
    unsigned long long k[RS_R];
#pragma unroll
    for (int r = 0; r < RS_R; r++) k[r] = rs_load<PASS>(q, src, min(i0 + r * RS_T + tid, n - 1));
    h[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS_R; r++)
        if (i0 + r * RS_T + tid < n) atomicAdd(&h[rs_digit<PASS>(k[r])], 1u);
    __syncthreads();
    table[(size_t)blockIdx.x * RS_BINS + tid] = h[tid];
}

template <int PASS>
__global__ __launch_bounds__(RS_T) void k_rs_place(const float *__restrict__ q,
                                                   const unsigned long long *__restrict__ src, int n,
                                                   const uint32_t *__restrict__ table,
                                                   unsigned long long *__restrict__ dst, float *__restrict__ sq,
                                                   uint32_t *__restrict__ sid) {
    constexpr int NW = RS_T / WAVE;
    __shared__ uint16_t cnt[NW][RS_BINS];  // per wave and digit: its keys so far, then the keys of earlier waves
    __shared__ uint32_t base[RS_BINS], wt[NW];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), w = tid / WAVE;
    const int i0 = blockIdx.x * RS_TILE + w * (RS_TILE / NW);  // a wave's keys are contiguous
    unsigned long long k[RS_R];
#pragma unroll
    for (int r = 0; r < RS_R; r++) k[r] = rs_load<PASS>(q, src, min(i0 + r * WAVE + lane, n - 1));
    uint32_t tot = 0, before = 0;
#pragma unroll 8
    for (int b = 0; b < (int)gridDim.x; b++) {
        const uint32_t c = table[(size_t)b * RS_BINS + tid];
        tot += c;
        before += b < (int)blockIdx.x ? c : 0u;
    }
    for (int j = 0; j < NW; j++) cnt[j][tid] = 0;
    uint32_t inc = tot;  // exclusive scan of the digits' totals over the block
    for (int s = 1; s < WAVE; s <<= 1) {
        const uint32_t o = __shfl_up(inc, s, WAVE);
        if (lane >= s) inc += o;
    }
    if (lane == WAVE - 1) wt[w] = inc;
    __syncthreads();
    uint32_t off = inc - tot + before;
    for (int j = 0; j < w; j++) off += wt[j];
    base[tid] = off;
    uint32_t rank[RS_R];
#pragma unroll
    for (int r = 0; r < RS_R; r++) {
        const bool live = i0 + r * WAVE + lane < n;
        const uint32_t d = rs_digit<PASS>(k[r]);
        uint64_t peers = __ballot(live);
#pragma unroll
        for (int bit = 0; bit < RS_BITS; bit++) {
            const bool set = (d >> bit) & 1u;
            const uint64_t m = __ballot(set);
            peers &= set ? m : ~m;
        }
        const uint32_t below = (uint32_t)__popcll(peers & ((1ull << lane) - 1));
        rank[r] = cnt[w][d] + below;
        wave_lds_sync();
        if (live && below == 0) cnt[w][d] = (uint16_t)(cnt[w][d] + __popcll(peers));
        wave_lds_sync();
    }
    __syncthreads();
    uint32_t run = 0;
    for (int j = 0; j < NW; j++) {
        const uint32_t c = cnt[j][tid];
        cnt[j][tid] = (uint16_t)run;
        run += c;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS_R; r++) {
        if (i0 + r * WAVE + lane >= n) continue;
        const uint32_t d = rs_digit<PASS>(k[r]), at = base[d] + cnt[w][d] + rank[r];
        if constexpr (PASS == 2) {
            sq[at] = __uint_as_float(0x3F800000u - (uint32_t)(k[r] >> 32));
            sid[at] = (uint32_t)k[r];
        } else {
            dst[at] = k[r];
        }
    }
}

__global__ __launch_bounds__(1024) void k_smp_cut(const float *__restrict__ sq, int V, double top_p, SmpCtl *ctl) {
    __shared__ OrdLds ord;
    float s;
    const int c = ord_block<float, false>(sq, 1.0f, V, s, [=](float r) { return (double)r >= top_p; }, ord, nullptr);
    if (threadIdx.x == 0) ctl->cut = c >= 0 ? c + 1 : V;
}

// The draw over cut candidates in global memory.
__global__ __launch_bounds__(1024) void k_smp_draw(const float *__restrict__ sq, const uint32_t *__restrict__ sid,
                                                   const float *__restrict__ sums, double u, SmpCtl *ctl) {
    __shared__ OrdLds ord;
    if (ctl->status != SMP_ST_PENDING) return;
    const int cut = ctl->cut;
    float s2 = 0.0f;
    for (int c = 0; c * NP_BUFSIZE < cut; c++) s2 = s2 + sums[c];
    const int pos = ord_draw(sq, cut, s2, u, ord);
    if (threadIdx.x == 0) {
        ctl->token = (int)sid[pos];
        ctl->status = SMP_ST_OK;
    }
}

// ------------------------------------------------ launchers
static unsigned smp_grid(long n, long per) { return (unsigned)std::max<long>(1, std::min<long>(256, (n + per - 1) / per)); }

size_t smp_small_lds() { return sizeof(unsigned long long) * SMP_SMALL + sizeof(PwTree); }

// p and the buffer sums; then q with or without the candidate selection
static void launch_probs(const SmpBufs &b, const float *logits, int V, float T, double top_p, bool select,
                         hipStream_t st) {
    const unsigned nb = smp_grid(V, SMP_T * 4);
    const int nchunks = (V + NP_BUFSIZE - 1) / NP_BUFSIZE;
    TG_LAUNCH(k_smp_max, dim3(nb), dim3(SMP_T), 0, st, logits, V, b.pmax, b.pbad, b.hcnt, b.hmass, b.ctl);
    TG_LAUNCH(k_smp_exp, dim3(smp_grid(V, SMP_T * 2)), dim3(SMP_T), 0, st, logits, V, b.pmax, b.pbad, (int)nb, T,
              b.p, b.ctl);
    TG_LAUNCH(k_smp_chunks, dim3(nchunks), dim3(WAVE), 0, st, b.p, V, 0, b.ctl, b.sums);
    if (select)
        TG_LAUNCH(k_smp_norm<true>, dim3(smp_grid(V, SMP_T * 8)), dim3(SMP_T), 0, st, b.p, V, b.sums, nchunks,
                  top_p, b.ctl, b.q, b.hcnt, b.hmass);
    else
        TG_LAUNCH(k_smp_norm<false>, dim3(smp_grid(V, SMP_T * 2)), dim3(SMP_T), 0, st, b.p, V, b.sums, nchunks,
                  top_p, b.ctl, b.q, b.hcnt, b.hmass);
}

hipError_t launch_sample_main(const SmpBufs &b, const float *logits, int V, float T, double top_p, double u,
                              hipStream_t st) {
    if (V <= 0 || V > SMP_VMAX) return hipErrorInvalidValue;
    launch_probs(b, logits, V, T, top_p, true, st);
    TG_LAUNCH(k_smp_compact, dim3(smp_grid(V, SMP_T * 8)), dim3(SMP_T), 0, st, b.q, V, b.ctl, b.keys);
    TG_LAUNCH(k_smp_final, dim3(1), dim3(1024), smp_small_lds(), st, b.keys, V, top_p, u, b.ctl);
    return hipGetLastError();
}

hipError_t launch_sample_large(const SmpBufs &b, int V, double top_p, double u, hipStream_t st) {
    if (V <= 0 || V > SMP_VMAX) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((V + RS_TILE - 1) / RS_TILE)), block(RS_T);
    TG_LAUNCH(k_rs_count<0>, grid, block, 0, st, b.q, b.keys, V, b.table);
    TG_LAUNCH(k_rs_place<0>, grid, block, 0, st, b.q, b.keys, V, b.table, b.keys, b.sq, b.sid);
    TG_LAUNCH(k_rs_count<1>, grid, block, 0, st, b.q, b.keys, V, b.table);
    TG_LAUNCH(k_rs_place<1>, grid, block, 0, st, b.q, b.keys, V, b.table, b.keys2, b.sq, b.sid);
    TG_LAUNCH(k_rs_count<2>, grid, block, 0, st, b.q, b.keys2, V, b.table);
    TG_LAUNCH(k_rs_place<2>, grid, block, 0, st, b.q, b.keys2, V, b.table, b.keys, b.sq, b.sid);
    const int nchunks = (V + NP_BUFSIZE - 1) / NP_BUFSIZE;
    TG_LAUNCH(k_smp_cut, dim3(1), dim3(1024), 0, st, b.sq, V, top_p, b.ctl);
    TG_LAUNCH(k_smp_chunks, dim3(nchunks), dim3(WAVE), 0, st, b.sq, 0, 1, b.ctl, b.sums);
    TG_LAUNCH(k_smp_draw, dim3(1), dim3(1024), 0, st, b.sq, b.sid, b.sums, u, b.ctl);
    return hipGetLastError();
}

hipError_t launch_sample_all(const SmpBufs &b, const float *logits, int V, float T, double top_p, double u,
                             hipStream_t st) {
    if (V <= 0 || V > SMP_VMAX) return hipErrorInvalidValue;
    launch_probs(b, logits, V, T, top_p, false, st);
    return launch_sample_large(b, V, top_p, u, st);
}

hipError_t sample_prepare() {
    return hipFuncSetAttribute((const void *)k_smp_final, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)smp_small_lds());
}

}  // namespace tg
