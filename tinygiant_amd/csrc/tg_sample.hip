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
//   k_smp_exp_chunks  p, and the pairwise sum of each 8192-value buffer
//   k_smp_norm_select  S from the buffer sums; q = p / S; a histogram of q in
//                 1/16 binades with counts and exact mass (units of 2^-40),
//                 and from it the fewest top buckets whose mass provably
//                 carries the fp32 running sum past top_p (they hold the
//                 candidates)
//   k_smp_compact their keys (descending q, ascending id)
//   k_smp_rank    at most 8192 of them: each key to its place
//   k_smp_final   the cutoff, the candidates' sum and the draw
// More candidates (flat distributions, top_p near 1): the host then launches a
// radix sort of every q (k_rs_count, k_rs_place), and k_smp_cut, k_smp_chunks
// and k_smp_draw finish.  top_p >= 1 or NaN with more than 8192 tokens goes
// there at once, without the selection and its wait.
#include <algorithm>
#include <type_traits>

#include "tg_device.h"
#include "tg_internal.h"

namespace tg {

constexpr int SMP_T = 256;
constexpr int PW_LEVELS = 8;   // depth of numpy's pairwise tree over <= 8192 values is 7

// 1/16 binades below 1; everything below 2^-63 (and zero) in bucket 0
TG_DEV uint32_t smp_bucket(float q) {
    const int b = (int)(__float_as_uint(q) >> SMP_BUCKET_SHIFT) - SMP_BUCKET_LOW;
    return (uint32_t)min(max(b, 0), SMP_BUCKETS - 1);
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
// Base case of numpy's pairwise summation, n <= 128 values v[0..n), by 8
// adjacent lanes (j = lane % 8): each keeps one of the 8 interleaved
// accumulators; every lane returns the sum.
TG_DEV float pw_leaf8(const float *v, int n, int j) {
    if (n < 8) {
        float r = 0.0f;
        for (int i = 0; i < n; i++) r = r + v[i];
        return r;
    }
    const int main = n & ~7;
    float r = v[j];
    for (int i = 8; i < main; i += 8) r = r + v[i + j];
    auto dpp = [](float x, auto c) {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(c)::value, 0xF, 0xF, false));
    };
    r = r + dpp(r, std::integral_constant<int, 0xB1>{});   // lane ^ 1
    r = r + dpp(r, std::integral_constant<int, 0x4E>{});   // lane ^ 2
    r = r + dpp(r, std::integral_constant<int, 0x141>{});  // the other quad of 8
    for (int i = main; i < n; i++) r = r + v[i];
    return r;
}

// The recursion's nodes level by level (at most 64 per level for n <= 8192):
// node (start, len) splits into len/2 rounded down to a multiple of 8 and
// the rest while len > 128.  ch = index of the left child in the next level,
// -1 for a leaf.
struct PwTree {
    short st[PW_LEVELS][WAVE], ln[PW_LEVELS][WAVE], ch[PW_LEVELS][WAVE];
    float v[PW_LEVELS][WAVE];
    short leaf[PW_LEVELS * WAVE];  // level * 64 + index
    int nleaf;
};

// numpy's pairwise sum of v[0..n), 1 <= n <= 8192, by the whole block (1024
// threads; every thread returns it): wave 0 lays out the tree, every leaf is
// summed by 8 lanes, and wave 0 adds the inner nodes up, each as left + right.
// (Leaves one per lane of one wave read 64 lines per load: 6.1 us a buffer.)
TG_DEV float block_pw_sum(const float *v, int n, PwTree &t) {
    const int tid = threadIdx.x, lane = tid & (WAVE - 1);
    int cnt[PW_LEVELS];
    if (tid < WAVE) {
        if (lane == 0) { t.st[0][0] = 0; t.ln[0][0] = (short)n; }
        wave_lds_sync();
        int c = 1, nl = 0;
#pragma unroll
        for (int d = 0; d < PW_LEVELS; d++) {
            cnt[d] = c;
            const bool have = lane < c;
            const int s0 = have ? t.st[d][lane] : 0, l0 = have ? t.ln[d][lane] : 0;
            const bool split = have && l0 > 128 && d + 1 < PW_LEVELS;
            const uint64_t m = __ballot(split), mf = __ballot(have && !split), lt = (1ull << lane) - 1;
            const int r = __popcll(m & lt);
            if (split) {
                const int n2 = (l0 >> 1) & ~7;
                t.st[d + 1][2 * r] = (short)s0;
                t.ln[d + 1][2 * r] = (short)n2;
                t.st[d + 1][2 * r + 1] = (short)(s0 + n2);
                t.ln[d + 1][2 * r + 1] = (short)(l0 - n2);
            } else if (have) {
                t.leaf[nl + __popcll(mf & lt)] = (short)(d * WAVE + lane);
            }
            if (have) t.ch[d][lane] = (short)(split ? 2 * r : -1);
            c = 2 * __popcll(m);
            nl += __popcll(mf);
            wave_lds_sync();
        }
        if (lane == 0) t.nleaf = nl;
    }
    __syncthreads();
    const int nl = t.nleaf;
    for (int g = tid >> 3; g < nl; g += (int)blockDim.x >> 3) {
        const int at = t.leaf[g], d = at / WAVE, i = at % WAVE;
        const float r = pw_leaf8(v + t.st[d][i], t.ln[d][i], tid & 7);
        if ((tid & 7) == 0) t.v[d][i] = r;
    }
    __syncthreads();
    if (tid < WAVE) {
#pragma unroll
        for (int d = PW_LEVELS - 2; d >= 0; d--) {
            if (lane < cnt[d]) {
                const int ch = t.ch[d][lane];
                if (ch >= 0) t.v[d][lane] = t.v[d + 1][ch] + t.v[d + 1][ch + 1];
            }
            wave_lds_sync();
        }
    }
    __syncthreads();
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
// inexact and are not used.  The same 151,936 values now take 25 us (fp32 cut)
// and 56 us (float64 draw): one block, bound by its additions and 10 tiles of
// two barriers each.  (With 8 values per lane 36 and 72 us, loaded one dword at a
// time instead of by float4 95 and 113 us.  Ulps counted as 64-bit integers: 166 and 192 us.)
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

// values per lane and scan: by a block (8: cut 36, draw 72 us instead of 25 and
// 56 at 151,936 values), by one wave (which scans its values once per binade)
constexpr int ORD_R = 16, ORD_R1 = 8;
static_assert(SMP_PAD % ORD_R == 0 && SMP_PAD % ORD_R1 == 0, "loads of whole runs stay in sq");
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

// Continues the running sum s of the values before pos (a multiple of 16; at 0,
// s = v[0] and the sum goes on from v[1]) over v[pos..n) (each divided by div
// when DIV), by NW waves (NW == 1: any one wave; else the whole block of ORD_NW
// waves).  v is 16-byte aligned and readable to the next multiple of 16 values.
// Returns the first index whose running sum satisfies pred (monotone), or -1
// with s the sum of all.  log: the sum before each tile.
template <class F, int NW, bool DIV, class Pred>
TG_DEV int ord_run(const float *v, float div, int n, int pos, F &s, Pred pred, OrdLds &L, double *log) {
    constexpr int R = NW == 1 ? ORD_R1 : ORD_R, TILE = NW * WAVE * R;
    const int lane = __lane_id(), w = NW == 1 ? 0 : (int)threadIdx.x / WAVE, slot = (w * WAVE + lane) * R;
    float raw[R];
    F x[R];
    // 16-byte loads, unconditional (at the last group past the end, whose
    // values are not used), so that they stay in flight during a scan
    auto load = [&](int p0) {
        const float4 *g = reinterpret_cast<const float4 *>(v + min(p0 + slot, (n - 1) & ~(R - 1)));
#pragma unroll
        for (int q = 0; q < R / 4; q++) {
            const float4 f = g[q];
            raw[4 * q] = f.x; raw[4 * q + 1] = f.y; raw[4 * q + 2] = f.z; raw[4 * q + 3] = f.w;
        }
    };
    load(pos);
    for (; pos < n; pos += TILE) {
#pragma unroll
        for (int j = 0; j < R; j++) {
            const int i = pos + slot + j;
            const float q = DIV ? raw[j] / div : raw[j];
            x[j] = i > 0 && i < n ? (F)q : (F)0;
        }
        load(pos + TILE);
        if (NW > 1 && log && threadIdx.x == 0) *log++ = (double)s;
        const int end = min(pos + slot + R, n);  // of this lane's run
        for (;;) {
            // x: this tile's values not yet in s (those that are, and past n: 0)
            const F c = Grid<F>::binade(s), c1 = c + c * Grid<F>::ULP;
            F a0 = c, a1 = c1;
#pragma unroll
            for (int j = 0; j < R; j++) {
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
            for (int j = 0; j < R; j++) se = se + x[j];
            const uint64_t m = __ballot(se >= c + c || pred(se));
            int first = WAVE - 1, at = INT_MAX, hit = -1;
            if (m) {
                first = __ffsll((unsigned long long)m) - 1;
                at = __builtin_amdgcn_readlane(end, first);
                F r = sl;
                int k = 0;
#pragma unroll
                for (int j = 0; j < R; j++) {
                    r = r + x[j];
                    k += pred(r) ? 0 : 1;
                }
                k = __builtin_amdgcn_readlane(k, first);
                if (k < R) hit = pos + (w * WAVE + first) * R + k;
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
            for (int j = 0; j < R; j++)
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

// One block per 8192-value buffer: p = exp((l - max) / T) and its pairwise sum,
// read from LDS.  Few candidates leave a call bound by the host's launches, so the
// two are one (a call over 8192 tokens with few candidates 50 us; as two launches 62).
__global__ __launch_bounds__(1024) void k_smp_exp_chunks(const float *__restrict__ l, int V,
                                                         const float *__restrict__ pmax, const int *__restrict__ pbad,
                                                         int nb, float T, float *__restrict__ p,
                                                         float *__restrict__ sums, SmpCtl *ctl) {
    constexpr int R = NP_BUFSIZE / 1024;
    __shared__ float ps[NP_BUFSIZE];
    __shared__ PwTree t;
    __shared__ float s_m;
    const int tid = threadIdx.x, c0 = blockIdx.x * NP_BUFSIZE;
    float x[R];
#pragma unroll
    for (int r = 0; r < R; r++) x[r] = l[min(c0 + r * 1024 + tid, V - 1)];
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
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int j = r * 1024 + tid;
        if (c0 + j < V) {
            const float z = (x[r] - m) / T, e = (float)exp((double)z);
            p[c0 + j] = e;
            ps[j] = e;
        }
    }
    __syncthreads();
    const float s = block_pw_sum(ps, min(NP_BUFSIZE, V - c0), t);
    if (tid == 0) sums[blockIdx.x] = s;
}

// One block per 8192-value buffer of the candidates v[0..ctl->cut): its pairwise sum.
__global__ __launch_bounds__(1024) void k_smp_chunks(const float *__restrict__ v, const SmpCtl *ctl,
                                                     float *__restrict__ sums) {
    __shared__ PwTree t;
    if (ctl->status != SMP_ST_PENDING) return;
    const int n = ctl->cut, c0 = blockIdx.x * NP_BUFSIZE;
    if (c0 >= n) return;
    const float s = block_pw_sum(v + c0, min(NP_BUFSIZE, n - c0), t);
    if (threadIdx.x == 0) sums[blockIdx.x] = s;
}
// np.sum from the buffer sums: added one after another from 0 (n <= 64; every
// lane of the wave)
TG_DEV float smp_total(const float *sums, int n) {
    const int lane = __lane_id();
    const float x = lane < n ? sums[lane] : 0.0f;
    float s = 0.0f;
    for (int c = 0; c < n; c++) s = s + rdl(x, c);
    return s;
}

// The candidates lie in the top buckets: with C elements and exact mass M
// (2^-40 units, rounded down per element) in buckets >= b, the fp32 running
// sum over those elements in descending order ends at or above
// M 2^-40 - C 2^-24 (each addition rounds by at most half an ulp of a sum
// below 2), so M 2^-40 >= top_p + C 2^-24 puts the crossing inside them.
// The largest such b is taken; none (top_p near or above 1, or NaN) = all.
// A block of SL_T threads; the histogram is read at device scope (other
// blocks' atomics).  Leaves bstar and C in ctl.
constexpr int SL_T = 1024, SL_R = 8;  // threads, values per thread of the selection's launches
static_assert(SMP_BUCKETS == SL_T, "one bucket per thread");
TG_DEV void smp_select(const uint32_t *hcnt, const unsigned long long *hmass, int V, double top_p, SmpCtl *ctl) {
    constexpr int NW = SL_T / WAVE;
    __shared__ uint32_t wc[NW], hC[NW];
    __shared__ unsigned long long wm[NW];
    __shared__ int hd[NW];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), w = tid / WAVE;
    // descending position tid holds bucket SMP_BUCKETS - 1 - tid
    const int b = SMP_BUCKETS - 1 - tid;
    const uint32_t c = __hip_atomic_load(hcnt + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long m = __hip_atomic_load(hmass + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    uint32_t cc = c;  // inclusive scan over the wave, then over waves
    unsigned long long cm = m;
    for (int s = 1; s < WAVE; s <<= 1) {
        const uint32_t oc = __shfl_up(cc, s, WAVE);
        const unsigned long long om = __shfl_up(cm, s, WAVE);
        if (lane >= s) { cc += oc; cm += om; }
    }
    if (lane == WAVE - 1) { wc[w] = cc; wm[w] = cm; }
    __syncthreads();
    for (int j = 0; j < w; j++) { cc += wc[j]; cm += wm[j]; }
    const double need = (top_p + (double)cc * 0x1p-24) * 0x1p40 + 1024.0;
    const uint64_t hit = __ballot(cc >= 1 && (double)cm >= need);
    const int first = hit ? __ffsll((unsigned long long)hit) - 1 : 0;
    const uint32_t fc = (uint32_t)__builtin_amdgcn_readlane((int)cc, first);
    if (lane == 0) { hd[w] = hit ? w * WAVE + first : INT_MAX; hC[w] = fc; }
    __syncthreads();
    if (tid == 0) {
        int d = INT_MAX;
        uint32_t C = (uint32_t)V;
        for (int j = NW - 1; j >= 0; j--)
            if (hd[j] != INT_MAX) { d = hd[j]; C = hC[j]; }
        ctl->bstar = d == INT_MAX ? 0 : SMP_BUCKETS - 1 - d;
        ctl->C = C;
    }
}

__global__ __launch_bounds__(SMP_T) void k_smp_norm(const float *__restrict__ p, int V,
                                                    const float *__restrict__ sums, int nchunks, SmpCtl *ctl,
                                                    float *__restrict__ q) {
    const float S = smp_total(sums, nchunks);
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl->S = S;
    for (int i = blockIdx.x * SMP_T + threadIdx.x; i < V; i += gridDim.x * SMP_T) q[i] = p[i] / S;
}

// The same with the histogram; the last block to finish picks the candidate
// buckets.  Bound by the device-scope atomics on the histogram: few blocks (8
// values per thread of 1024) so that a bucket takes few of them, and no fence
// (its write-back of the L2 cost 10 us): 8.3 us at 151,936 values, from 20.
__global__ __launch_bounds__(SL_T) void k_smp_norm_select(const float *__restrict__ p, int V,
                                                          const float *__restrict__ sums, int nchunks, double top_p,
                                                          SmpCtl *ctl, float *__restrict__ q, uint32_t *hcnt,
                                                          unsigned long long *hmass) {
    __shared__ uint32_t lc[SMP_BUCKETS];
    __shared__ unsigned long long lm[SMP_BUCKETS];
    __shared__ int s_last;
    const int tid = threadIdx.x, i0 = blockIdx.x * SL_T * SL_R + tid;
    float x[SL_R];
#pragma unroll
    for (int r = 0; r < SL_R; r++) x[r] = p[min(i0 + r * SL_T, V - 1)];
    lc[tid] = 0;
    lm[tid] = 0;
    const float S = smp_total(sums, nchunks);
    if (blockIdx.x == 0 && tid == 0) ctl->S = S;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < SL_R; r++) {
        const int i = i0 + r * SL_T;
        if (i < V) {
            const float v = x[r] / S;
            q[i] = v;
            const uint32_t b = smp_bucket(v);
            atomicAdd(&lc[b], 1u);
            atomicAdd(&lm[b], smp_mass(v));
        }
    }
    __syncthreads();
    if (lc[tid]) {
        atomicAdd(&hcnt[tid], lc[tid]);
        atomicAdd(&hmass[tid], lm[tid]);
    }
    // this thread's histogram atomics are done at device scope (a fence would
    // also write the L2's q back); the last block reads them at device scope
    __builtin_amdgcn_s_waitcnt(VMCNT0);
    __syncthreads();
    if (tid == 0)
        s_last = __hip_atomic_fetch_add(&ctl->done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    __syncthreads();
    if (s_last) smp_select(hcnt, hmass, V, top_p, ctl);
}

// The candidates' keys (bucket >= ctl->bstar) into keys[0..C), in any order:
// per block one global slot range.
__global__ __launch_bounds__(SL_T) void k_smp_compact(const float *__restrict__ q, int V, SmpCtl *ctl,
                                                      unsigned long long *__restrict__ keys) {
    __shared__ uint32_t wc[SL_T / WAVE], s_base;
    const uint32_t bstar = (uint32_t)ctl->bstar;
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), w = tid / WAVE, i0 = blockIdx.x * SL_T * SL_R + tid;
    float v[SL_R];
#pragma unroll
    for (int r = 0; r < SL_R; r++) v[r] = q[min(i0 + r * SL_T, V - 1)];
    uint64_t m[SL_R];
    uint32_t n = 0;
#pragma unroll
    for (int r = 0; r < SL_R; r++) {
        m[r] = __ballot(i0 + r * SL_T < V && smp_bucket(v[r]) >= bstar);
        n += (uint32_t)__popcll(m[r]);
    }
    if (lane == 0) wc[w] = n;
    __syncthreads();
    if (tid == 0) {
        uint32_t t = 0;
        for (int j = 0; j < SL_T / WAVE; j++) t += wc[j];
        s_base = t ? atomicAdd(&ctl->n, t) : 0u;
    }
    __syncthreads();
    uint32_t at = s_base;
    for (int j = 0; j < w; j++) at += wc[j];
#pragma unroll
    for (int r = 0; r < SL_R; r++) {
        if ((m[r] >> lane) & 1)
            keys[at + __popcll(m[r] & ((1ull << lane) - 1))] = smp_key(v[r], (uint32_t)(i0 + r * SL_T));
        at += (uint32_t)__popcll(m[r]);
    }
}

// At most SMP_SMALL candidates in order: a key's place is the number of
// smaller keys (they are distinct).  A block places 64 keys, one per lane, its
// 16 waves each counting over a sixteenth of all keys, read lane by lane: at
// 1,400 candidates 22 blocks and 6 rounds of 16 keys a wave, 8.8 us, and the
// scans after it 17 us; with a bitonic network of 66 dependent steps in one
// block before the scans the two took 57 us.
__global__ __launch_bounds__(1024) void k_smp_rank(const unsigned long long *__restrict__ keys,
                                                   const SmpCtl *__restrict__ ctl, float *__restrict__ sq,
                                                   uint32_t *__restrict__ sid) {
    constexpr int NW = 1024 / WAVE;
    __shared__ uint32_t cnt[WAVE];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), w = tid / WAVE;
    const int C = (int)ctl->C, k0 = blockIdx.x * WAVE;
    if (ctl->bad || C > SMP_SMALL || k0 >= C) return;  // uniform
    const unsigned long long mine = keys[min(k0 + lane, C - 1)];
    if (tid < WAVE) cnt[tid] = 0;
    const int per = (C + NW - 1) / NW, lo = min(w * per, C), hi = min(lo + per, C);
    __syncthreads();
    uint32_t n = 0;
    for (int b = lo; b < hi; b += WAVE) {
        const unsigned long long o = b + lane < hi ? keys[b + lane] : ~0ull;  // ~0: below no key
        const int live = min(WAVE, hi - b);
        for (int i = 0; i < live; i += 16) {  // (lanes past live hold ~0)
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const uint32_t klo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)o, i + j);
                const uint32_t khi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(o >> 32), i + j);
                n += (((unsigned long long)khi << 32) | klo) < mine ? 1u : 0u;
            }
        }
    }
    atomicAdd(&cnt[lane], n);
    __syncthreads();
    if (tid < WAVE && k0 + lane < C) {
        sq[cnt[lane]] = smp_key_q(mine);
        sid[cnt[lane]] = (uint32_t)mine;
    }
}

// The last launch of a call with at most SMP_SMALL candidates: cutoff, the
// candidates' sum and the draw.  More candidates: ctl->large for the host.
__global__ __launch_bounds__(1024) void k_smp_final(const float *__restrict__ sq, const uint32_t *__restrict__ sid,
                                                    int V, double top_p, double u, SmpCtl *ctl) {
    __shared__ PwTree t;
    __shared__ OrdLds ord;
    const int tid = threadIdx.x, C = (int)ctl->C;
    if (ctl->bad) {
        if (tid == 0) ctl->status = SMP_ST_INPUT;
        return;
    }
    if (C > SMP_SMALL) {
        if (tid == 0) ctl->large = 1;
        return;
    }
    float s;
    int cut = ord_block<float, false>(sq, 1.0f, C, s, [=](float r) { return (double)r >= top_p; }, ord, nullptr);
    if (cut < 0) {
        if (C != V) {  // the selection bound guarantees a crossing inside a strict prefix
            if (tid == 0) ctl->status = SMP_ST_BOUND;
            return;
        }
        cut = V;  // searchsorted past the end: every token is a candidate
    } else {
        cut += 1;
    }
    const float s2 = 0.0f + block_pw_sum(sq, cut, t);
    const int pos = ord_draw(sq, cut, s2, u, ord);
    if (tid == 0) {
        ctl->cut = cut;
        ctl->token = (int)sid[pos];
        ctl->status = SMP_ST_OK;
    }
}

// ------------------------------------------------ more than 8192 candidates
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
    if (ctl->bad) {  // (the sort ran on what the bad logits gave)
        if (threadIdx.x == 0) ctl->status = SMP_ST_INPUT;
        return;
    }
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
    const float s2 = smp_total(sums, (cut + NP_BUFSIZE - 1) / NP_BUFSIZE);
    const int pos = ord_draw(sq, cut, s2, u, ord);
    if (threadIdx.x == 0) {
        ctl->token = (int)sid[pos];
        ctl->status = SMP_ST_OK;
    }
}

// ------------------------------------------------ launchers
static unsigned smp_grid(long n, long per) { return (unsigned)std::max<long>(1, std::min<long>(256, (n + per - 1) / per)); }

// p and the buffer sums; then q with or without the candidate selection
static void launch_probs(const SmpBufs &b, const float *logits, int V, float T, double top_p, bool select,
                         hipStream_t st) {
    const unsigned nb = smp_grid(V, SMP_T * 4);
    const int nchunks = (V + NP_BUFSIZE - 1) / NP_BUFSIZE;
    TG_LAUNCH(k_smp_max, dim3(nb), dim3(SMP_T), 0, st, logits, V, b.pmax, b.pbad, b.hcnt, b.hmass, b.ctl);
    TG_LAUNCH(k_smp_exp_chunks, dim3(nchunks), dim3(1024), 0, st, logits, V, b.pmax, b.pbad, (int)nb, T, b.p, b.sums,
              b.ctl);
    if (select)
        TG_LAUNCH(k_smp_norm_select, dim3((unsigned)((V + SL_T * SL_R - 1) / (SL_T * SL_R))), dim3(SL_T), 0, st, b.p,
                  V, b.sums, nchunks, top_p, b.ctl, b.q, b.hcnt, b.hmass);
    else
        TG_LAUNCH(k_smp_norm, dim3(smp_grid(V, SMP_T * 2)), dim3(SMP_T), 0, st, b.p, V, b.sums, nchunks, b.ctl, b.q);
}

hipError_t launch_sample_main(const SmpBufs &b, const float *logits, int V, float T, double top_p, double u,
                              hipStream_t st) {
    if (V <= 0 || V > SMP_VMAX) return hipErrorInvalidValue;
    launch_probs(b, logits, V, T, top_p, true, st);
    TG_LAUNCH(k_smp_compact, dim3((unsigned)((V + SL_T * SL_R - 1) / (SL_T * SL_R))), dim3(SL_T), 0, st, b.q, V,
              b.ctl, b.keys);
    TG_LAUNCH(k_smp_rank, dim3((unsigned)((std::min(V, SMP_SMALL) + WAVE - 1) / WAVE)), dim3(1024), 0, st, b.keys,
              b.ctl, b.sq, b.sid);
    TG_LAUNCH(k_smp_final, dim3(1), dim3(1024), 0, st, b.sq, b.sid, V, top_p, u, b.ctl);
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
    TG_LAUNCH(k_smp_chunks, dim3(nchunks), dim3(1024), 0, st, b.sq, b.ctl, b.sums);
    TG_LAUNCH(k_smp_draw, dim3(1), dim3(1024), 0, st, b.sq, b.sid, b.sums, u, b.ctl);
    return hipGetLastError();
}

hipError_t launch_sample_all(const SmpBufs &b, const float *logits, int V, float T, double top_p, double u,
                             hipStream_t st) {
    if (V <= 0 || V > SMP_VMAX) return hipErrorInvalidValue;
    launch_probs(b, logits, V, T, top_p, false, st);
    return launch_sample_large(b, V, top_p, u, st);
}

}  // namespace tg
