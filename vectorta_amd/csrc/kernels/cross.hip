// Double-ALMA crossover backtest reduction for gfx950.
//
// For every (fast, slow) pair of ALMA parameter sets the position is
// pos_t = sign(ALMA_fast[t] - ALMA_slow[t]) from the first bar w where both
// are valid, and the per-pair statistics are
//   trades   = #{t > w : pos_t != pos_{t-1}}
//   n_long   = #{t >= w : pos_t = +1},  n_short = #{t >= w : pos_t = -1}
//   checksum = sum_t pos_t * (t + 1)                  (exact, int64)
//   pnl      = sum_{t <= T-2} pos_t * (x_{t+1} - x_t) (f64)
// The 58,300 x 200,000 position matrix is never materialised.
//
// The rows of the distinct ALMA parameter sets are computed here in f64 with
// the oracle's exact operation order (cross_rows_f64: 4-wide grouped dot,
// then * inv_norm, no contraction, weights from the host with glibc exp), so
// they are bit-identical to the f64 rows and every sign -- exact ties
// included -- equals the oracle's without any guard band.

// cross_pairs_f64 works on 32-bar words.  Per pair and bar it forms the f64
// difference and shifts its sign bit into a word (v_alignbit); an exact tie is
// the only difference of these finite rows with a zero high half (the rows hold
// no -0), so a running minimum of the high halves
// tells whether a word holds one.  Transitions are the set bits of the word
// xor its own shift, and all statistics are accumulated per transition r from
// position p to q: with s = p - q, net sum of pos += s r, 2 checksum +=
// s r (r + 1) and pnl += p (x[r] - x[last transition]); the differences of f32
// prices are exact in f64 and so are their sums (all are multiples of the
// smallest price's ulp), which makes the pnl equal to the bar-by-bar f64 sum.
// Words holding a tie run bar by bar.
//
// Work split: a wave takes 16 fast x 16 slow rows, four pairs (2 x 2) per
// lane, over one time segment.  The 32 rows' words are staged in LDS (row
// stride 34 doubles: the 8 rows read at one bar fall on distinct banks) and
// each value read feeds two pairs.  Each segment reads the position
// before it from the rows, so the segments are independent; cross_reduce sums
// them in segment order.  From eight segments on all tiles of a segment run on
// one XCD (dispatch is round-robin over 8), whose L2 then serves the segment's
// rows to every tile; fewer are spread over all (1,457,500 pairs x 3,000 bars in
// two segments: 682 us, 2,304 on two XCDs).
//
// Bound: VALU issue (88% of the issue slots): 2.5 instructions per pair and bar
// (subtract, shift, half a minimum), 0.4 for the words' sums and 0.5 for the
// transitions, which neighbouring pairs make at the same bars.  58,300 pairs
// x 200k bars: 1.37-1.5 ms, where a branch on every bar of the f64 sign, its
// rows read per pair, took 3.64.  Four fast rows per lane (237 VGPRs, two
// waves per SIMD, or spills at three) measured 1.74-2.4 ms, per-pair
// transition loops, each waiting for its own price, 1.69.
#include "vta_common.h"

struct cross_args {
    double *rows;               // [nrows][ldr] f64 ALMA rows
    const float *prices;        // [T]
    const double *w64;          // [nrows][pmax] f64 batch weights, not normalised
    const double *inv64;        // [nrows] 1 / sum(w)
    const int32_t *row_period;  // [nrows]
    const int32_t *fast_row;    // [nfast] -> row
    const int32_t *slow_row;    // [nslow] -> row
    int32_t *part_n;            // [nseg][3][npairs]: trades, bars long, bars short
    long long *part_ck;         // [nseg][npairs]
    double *part_pnl;           // [nseg][npairs]
    long long *out_i;           // [npairs][4]
    double *out_pnl;            // [npairs]
    int T;
    int fv;
    int nfast;
    int nslow;
    int nseg;
    int seg_len;
    int pmax;
    int ntiles_s;
    int ntiles;                 // 16 x 16-pair tiles
    int ldr;                    // row stride of `rows` (T rounded up to whole words)
    uint32_t rows_bytes;        // size of `rows` (below 4 GiB: cross_pairs_f64)
    int pad_;
};

#define CR_CH 32              // bars per word
#define CR_LD (CR_CH + 2)     // LDS row stride, doubles
#define CR_FN 2               // fast rows per lane
#define CR_SN 2               // slow rows per lane
#define CR_WPE 4              // waves per SIMD the registers are held to
#define CR_F (8 * CR_FN)      // fast rows per wave
#define CR_S (8 * CR_SN)      // slow rows per wave
#define RW_NB 8               // consecutive bars per lane of the row kernel
#define RW_T (256 * RW_NB)    // bars per row workgroup
#define RW_PMAX 296

// f64 ALMA rows in the oracle's order (alma.rs:1505-1527): for output t,
// sum over 4-tap groups g = (x0 w0 + x1 w1) + x2 w2 + x3 w3, sum += g, then
// the tail taps one at a time, out = sum * inv_norm.  NaN before fv + p - 1.
// Bound: f64 VALU (32 multiplies and 32 adds, none fused, per eight outputs
// and four taps; 89% of the instructions issued).  290 rows x 200k bars:
// 0.60-0.68 ms; 0.84 with the weights and every group's eleven prices read
// from LDS.
// grid.x = bar tiles of RW_T, grid.y = rows; lane l computes bars
// t0 + RW_NB l .. t0 + RW_NB (l + 1) - 1.
extern "C" __global__ __launch_bounds__(256) void cross_rows_f64(cross_args a) {
#pragma clang fp contract(off)
    // one pad double per eight: lane l's bars start at 9 l, so the lanes' reads
    // of one tap spread over all banks (8 l would put them on two)
    __shared__ double xs[(RW_T + RW_PMAX) / 8 * 9 + 9];
    const int tid = threadIdx.x;
    const int r = blockIdx.y;
    const int p = a.row_period[r];
    const int T = a.T;
    const int t0 = blockIdx.x * RW_T;
    const int xlo = t0 - p + 1;
    for (int i = tid; i < RW_T + p - 1; i += 256) {
        const int idx = xlo + i;
        xs[i + (i >> 3)] = (idx >= 0 && idx < T) ? (double)a.prices[idx] : 0.0;
    }
    __syncthreads();
    const double inv = a.inv64[r];
    const int warm = a.fv + p - 1;
    double *row = a.rows + (size_t)r * a.ldr;
    const double *ws = a.w64 + (size_t)r * a.pmax;   // wave-uniform: scalar loads
    // lane = RW_NB consecutive bars tb .. tb + RW_NB - 1: a 4-tap group of all
    // of them needs the RW_NB + 3 prices x(k) .., of which the last group left
    // all but four in registers, and 4 weights; each output keeps its own
    // operation order
    const int tb = RW_NB * tid;
    const double *x = xs + 9 * tid;         // x(m) = x[m + m / 8] = price[t0 + tb + m - p + 1]
    double acc[RW_NB];
#pragma unroll
    for (int i = 0; i < RW_NB; ++i) acc[i] = 0.0;
    double v[RW_NB + 7];
    auto group = [&](const double *w, int o) {
        const double w0 = w[0], w1 = w[1], w2 = w[2], w3 = w[3];
#pragma unroll
        for (int i = 0; i < RW_NB; ++i) {
            double g = v[o + i] * w0 + v[o + i + 1] * w1;
            g = g + v[o + i + 2] * w2;
            g = g + v[o + i + 3] * w3;
            acc[i] += g;
        }
    };
#pragma unroll
    for (int j = 0; j < RW_NB - 1; ++j) v[j] = x[j];
    int k = 0;
    for (; k + 8 <= p; k += 8, x += 9) {
#pragma unroll
        for (int j = RW_NB - 1; j < RW_NB + 7; ++j) v[j] = x[j + (j >> 3)];
        group(ws + k, 0);
        group(ws + k + 4, 4);
#pragma unroll
        for (int j = 0; j < RW_NB - 1; ++j) v[j] = v[j + 8];
    }
    // v[0 .. RW_NB - 2] hold x(0) .. of the advanced pointer
#pragma unroll
    for (int j = RW_NB - 1; j < RW_NB + 6; ++j) v[j] = x[j + (j >> 3)];
    if (p & 4) {
        group(ws + k, 0);
        k += 4;
#pragma unroll
        for (int j = 0; j < RW_NB + 2; ++j) v[j] = v[j + 4];
    }
#pragma unroll
    for (int d = 0; d < 3; ++d)
        if (k + d < p) {
            const double w = ws[k + d];
#pragma unroll
            for (int i = 0; i < RW_NB; ++i) acc[i] += v[i + d] * w;
        }
#pragma unroll
    for (int i = 0; i < RW_NB; ++i) {
        const int t = t0 + tb + i;
        // + 0.0: no row holds -0 (cross_pairs_f64 tells ties by +0 differences)
        if (t < T)
            row[t] = t >= warm ? acc[i] * inv + 0.0 : __builtin_bit_cast(double, 0x7ff8000000000000ull);
    }
}

// Statistics of one pair over one segment of words w = 0, 1, ...  A bar holds
// n = 1 - pos (0 long, 1 flat, 2 short), so that whole words add with a
// popcount: n2 = sum of n, z = flat bars, s2 = sum over the words of n2 after
// the word (which gives sum of w n = W n2 - s2 at the end) and b2 = sum of n b
// over the bars b of their words, added up from the transitions.
struct CrossRun {
    int at = 0;                  // open position: 0 long, 1 short, 2 flat
    int tr = 0;                  // transitions
    int n2 = 0, z = 0, b2 = 0;
    uint32_t s2 = 0;             // < 2^32: segments hold at most 2^18 bars
    double xa = 0.0;             // price at the open run's first bar
    double pnl = 0.0;
};

typedef double cross_d2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ int cross_at(double d) { return d > 0.0 ? 0 : (d < 0.0 ? 1 : 2); }
__device__ __forceinline__ double cross_pos(int at) { return at == 0 ? 1.0 : (at == 1 ? -1.0 : 0.0); }

// r (r + 1) / 2: the sum of t + 1 over [0, r)
__device__ __forceinline__ long long tri(int r) { return ((long long)r * ((long long)r + 1)) >> 1; }

// grid.x = 8 x ceil(nseg / 8) x ntiles (nseg x ntiles below eight segments),
// block = one wave.  WIDE: the rows take
// 4 GiB or more, so a lane's row offsets need 64 bits (else a scalar base and
// 32-bit lane offsets, which keep 24 registers and the address arithmetic
// out of the word loop).
template <bool WIDE>
__device__ __forceinline__ void cross_pairs(const cross_args &a) {
    __shared__ __align__(16) double lr[(CR_F + CR_S) * CR_LD];   // fast rows, then slow
    __shared__ double lx[CR_CH];                 // the word's prices
    const int lane = threadIdx.x;
    const bool by8 = a.nseg >= 8;                // (fewer would leave XCDs idle)
    const int in = by8 ? blockIdx.x >> 3 : blockIdx.x;
    const int seg = by8 ? (in / a.ntiles) * 8 + (blockIdx.x & 7) : in / a.ntiles;
    if (seg >= a.nseg) return;
    const int tile = in % a.ntiles;
    const int f0 = tile / a.ntiles_s * CR_F, s0 = tile % a.ntiles_s * CR_S;
    const int fg = lane >> 3, sg = lane & 7;
    const int T = a.T;
    const size_t ldr = (size_t)a.ldr;
    const int seg0 = seg * a.seg_len;
    const int seg1 = min(T, seg0 + a.seg_len);

    // pair (i, j) of a lane: fast row f0 + fg + 8 i, slow row s0 + sg + 8 j
    CrossRun run[CR_FN][CR_SN];
    int warm[CR_FN][CR_SN];                      // first bar counted; seg1: none
    bool odd = false;                            // a row that may hold NaN or Inf
    int first = seg1, last = 0;
#pragma unroll
    for (int i = 0; i < CR_FN; ++i)
#pragma unroll
        for (int j = 0; j < CR_SN; ++j) {
            const int f = f0 + fg + 8 * i, s = s0 + sg + 8 * j;
            const int rf = a.fast_row[min(f, a.nfast - 1)], rs = a.slow_row[min(s, a.nslow - 1)];
            const int w = a.fv + max(a.row_period[rf], a.row_period[rs]) - 1;
            const int b0 = max(seg0, w);
            // identical rows: always 0
            const bool walk = f < a.nfast && s < a.nslow && rf != rs && b0 < seg1;
            warm[i][j] = walk ? b0 : seg1;
            if (walk) {
                // at b0 = w the run opens; past it the bar before tells the
                // position, and a change at b0 itself is found by the walk
                const int ts = b0 > w ? b0 - 1 : b0;
                run[i][j].at = cross_at(a.rows[rf * ldr + ts] - a.rows[rs * ldr + ts]);
                run[i][j].xa = a.prices[b0];
                first = min(first, b0);
                last = max(last, b0);
                odd = odd || !vta_isfinite_d(a.inv64[rf]) || !vta_isfinite_d(a.inv64[rs]);
            }
        }
    for (int o = 32; o > 0; o >>= 1) {
        first = min(first, __shfl_xor(first, o));
        last = max(last, __shfl_xor(last, o));
    }
    first = __builtin_amdgcn_readfirstlane(first) & ~(CR_CH - 1);
    last = __builtin_amdgcn_readfirstlane(last);

    // staging: lane loads 16 bytes of rows lane / 16 + 4 k at bars 2 (lane & 15)
    const int tc = 2 * (lane & 15), tr4 = lane >> 4;
    uint32_t roff[(CR_F + CR_S) / 4];            // bytes, or the row
#pragma unroll
    for (int k = 0; k < (CR_F + CR_S) / 4; ++k) {
        const int r = tr4 + 4 * k;
        roff[k] = r < CR_F ? a.fast_row[min(f0 + r, a.nfast - 1)]
                           : a.slow_row[min(s0 + r - CR_F, a.nslow - 1)];
        if (!WIDE) roff[k] = (roff[k] * (uint32_t)a.ldr + (uint32_t)tc) * 8u;
    }
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(
        a.rows, (short)0, WIDE ? 0 : (int)a.rows_bytes, 0x00027000);
    for (int c0 = first; c0 < seg1; c0 += CR_CH) {
        cross_d2 g[(CR_F + CR_S) / 4];
#pragma unroll
        for (int k = 0; k < (CR_F + CR_S) / 4; ++k)
            g[k] = WIDE ? *reinterpret_cast<const cross_d2 *>(a.rows + roff[k] * ldr + c0 + tc)
                        : __builtin_bit_cast(cross_d2, __builtin_amdgcn_raw_buffer_load_b128(
                                                           rsrc, (int)roff[k], c0 * 8, 0));
        const float px = a.prices[min(c0 + (lane & 31), T - 1)];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k = 0; k < (CR_F + CR_S) / 4; ++k)
            *reinterpret_cast<cross_d2 *>(lr + (tr4 + 4 * k) * CR_LD + tc) = g[k];
        if (lane < CR_CH) lx[lane] = px;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

        // bar c0 + b at bit 31 - b: set where fast < slow
        uint32_t m[CR_FN][CR_SN];
        uint32_t tie[CR_FN][CR_SN];              // 0: the word may hold a tie
        // words that hold a pair's first bar or the series' end, or a row
        // that is not finite, run bar by bar
        const bool inner = c0 >= last && c0 + CR_CH <= seg1 && !odd;
#pragma unroll
        for (int i = 0; i < CR_FN; ++i)
#pragma unroll
            for (int j = 0; j < CR_SN; ++j) {
                m[i][j] = 0u;
                tie[i][j] = inner && run[i][j].at != 2 ? 0xffffffffu : 0u;
            }
        const double *pf = lr + fg * CR_LD, *ps = lr + (CR_F + sg) * CR_LD;
#pragma unroll 2
        for (int b = 0; b < CR_CH; b += 2) {
            cross_d2 vf[CR_FN], vs[CR_SN];
#pragma unroll
            for (int i = 0; i < CR_FN; ++i)
                vf[i] = *reinterpret_cast<const cross_d2 *>(pf + 8 * i * CR_LD + b);
#pragma unroll
            for (int j = 0; j < CR_SN; ++j)
                vs[j] = *reinterpret_cast<const cross_d2 *>(ps + 8 * j * CR_LD + b);
#pragma unroll
            for (int i = 0; i < CR_FN; ++i)
#pragma unroll
                for (int j = 0; j < CR_SN; ++j) {
                    const uint32_t h0 = __double2hiint(vf[i].x - vs[j].x);
                    const uint32_t h1 = __double2hiint(vf[i].y - vs[j].y);
                    m[i][j] = __builtin_amdgcn_alignbit(m[i][j], h0, 31);
                    m[i][j] = __builtin_amdgcn_alignbit(m[i][j], h1, 31);
                    tie[i][j] = min(min(tie[i][j], h0), h1);
                }
        }
        const int hi = min(seg1 - c0, CR_CH);
        // transitions of the words without ties: where the position differs
        // from the bar before
        uint32_t x[CR_FN][CR_SN], any = 0u;
        int sgn[CR_FN][CR_SN];                   // position before the next transition
#pragma unroll
        for (int i = 0; i < CR_FN; ++i)
#pragma unroll
            for (int j = 0; j < CR_SN; ++j) {
                CrossRun &q = run[i][j];
                const uint32_t mm = m[i][j];
                x[i][j] = 0u;
                sgn[i][j] = 1 - 2 * q.at;
                if (tie[i][j] != 0u) {
                    x[i][j] = mm ^ __builtin_amdgcn_alignbit((uint32_t)q.at, mm, 1);
                    q.tr += __popc(x[i][j]);
                    q.n2 += 2 * __popc(mm);
                    q.at = (int)(mm & 1u);
                    q.b2 += q.at * (CR_CH * (CR_CH - 1));
                    any |= x[i][j];
                } else {
                    for (int b = max(warm[i][j] - c0, 0); b < hi; ++b) {
                        const int at = cross_at(pf[8 * i * CR_LD + b] - ps[8 * j * CR_LD + b]);
                        const int n = at == 0 ? 0 : 3 - at;
                        q.n2 += n;
                        q.z += at >> 1;
                        q.b2 += n * b;
                        if (at != q.at) {
                            q.tr += 1;
                            q.pnl = fma(cross_pos(q.at), lx[b] - q.xa, q.pnl);
                            q.xa = lx[b];
                            q.at = at;
                        }
                    }
                }
                q.s2 += (uint32_t)q.n2;
            }
        // the lane's pairs take their next transitions together, so that the
        // price reads overlap; one with none left adds zeros
        while (any != 0u) {
            any = 0u;
#pragma unroll
            for (int i = 0; i < CR_FN; ++i)
#pragma unroll
                for (int j = 0; j < CR_SN; ++j) {
                    CrossRun &q = run[i][j];
                    const bool on = x[i][j] != 0u;
                    const int b = __builtin_clz(x[i][j] | 1u);   // 31 when none is left
                    const int sg1 = on ? sgn[i][j] : 0;
                    const double xt = lx[b];
                    q.pnl = fma((double)sg1, xt - q.xa, q.pnl);
                    q.xa = on ? xt : q.xa;
                    // a short run [b, b') holds n = 2: b' (b' - 1) - b (b - 1)
                    q.b2 -= sg1 * (b * (b - 1));
                    sgn[i][j] = -sgn[i][j];
                    x[i][j] &= 0x7fffffffu >> b;
                    any |= x[i][j];
                }
        }
    }
    const size_t npairs = (size_t)a.nfast * a.nslow;
    const double xe = a.prices[min(seg1, T - 1)];
    const long long words = first < seg1 ? (seg1 - first + CR_CH - 1) / CR_CH : 0;
#pragma unroll
    for (int i = 0; i < CR_FN; ++i)
#pragma unroll
        for (int j = 0; j < CR_SN; ++j) {
            const int f = f0 + fg + 8 * i, s = s0 + sg + 8 * j;
            if (f >= a.nfast || s >= a.nslow) continue;
            const bool walk = warm[i][j] < seg1;
            const CrossRun &q = run[i][j];
            const int bars = walk ? seg1 - warm[i][j] : 0;
            const int nshort = (q.n2 - q.z) >> 1;
            // sum of n (t + 1), t = first + 32 w + b
            const long long sn = (long long)(first + 1) * q.n2 +
                                 CR_CH * (words * (long long)q.n2 - (long long)q.s2) + (long long)q.b2;
            const size_t pair = (size_t)f * a.nslow + s;
            int32_t *n = a.part_n + (size_t)seg * 3 * npairs + pair;
            n[0] = walk ? q.tr : 0;
            n[npairs] = walk ? bars - q.z - nshort : 0;
            n[2 * npairs] = walk ? nshort : 0;
            const size_t o = (size_t)seg * npairs + pair;
            a.part_ck[o] = walk ? tri(seg1) - tri(warm[i][j]) - sn : 0;
            a.part_pnl[o] =
                walk ? fma(cross_pos(q.at), xe - q.xa, q.pnl) : 0.0;
        }
}

extern "C" __global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(CR_WPE)))
void cross_pairs_f64(cross_args a) { cross_pairs<false>(a); }
extern "C" __global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(CR_WPE)))
void cross_pairs_f64_wide(cross_args a) { cross_pairs<true>(a); }

// Sum of the segment partials: 64 pairs per block, its four waves take a
// quarter of the segments each (one lane per pair alone left too few loads
// in flight: 72 against 14 us at 40 segments), added in segment order.
extern "C" __global__ __launch_bounds__(256) void cross_reduce(cross_args a) {
    __shared__ long long si[3][4][64];
    __shared__ double sp[3][64];
    const size_t npairs = (size_t)a.nfast * a.nslow;
    const int lane = threadIdx.x & 63, part = threadIdx.x >> 6;
    const size_t p = (size_t)blockIdx.x * 64 + lane;
    const bool active = p < npairs;
    long long s[4] = {0, 0, 0, 0};
    double pn = 0.0;
    const int each = (a.nseg + 3) / 4;
    const int g1 = min(a.nseg, (part + 1) * each);
    if (active) {
#pragma unroll 4
        for (int g = part * each; g < g1; ++g) {
            const int32_t *n = a.part_n + (size_t)g * 3 * npairs + p;
            const size_t o = (size_t)g * npairs + p;
            s[0] += n[0];
            s[1] += n[npairs];
            s[2] += n[2 * npairs];
            s[3] += a.part_ck[o];
            pn += a.part_pnl[o];
        }
    }
    if (part > 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) si[part - 1][i][lane] = s[i];
        sp[part - 1][lane] = pn;
    }
    __syncthreads();
    if (part > 0 || !active) return;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] += si[q][i][lane];
        pn += sp[q][lane];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) a.out_i[p * 4 + i] = s[i];
    a.out_pnl[p] = pn;
}
