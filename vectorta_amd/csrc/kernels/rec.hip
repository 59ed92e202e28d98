// Wilder / exponential recurrences for gfx950: EMA, RSI, ATR, ADX and the fused
// EMA+RSI+ATR many-series launch.
//
// Each lane runs one stream (a combo of a one-series batch, or one series of
// a time-major matrix) through an f64 engine that restates the reference's
// scalar arithmetic in the same order:
//   EMA  src/indicators/moving_averages/ema.rs:430-468
//   RSI  src/indicators/rsi.rs:327-414
//   ATR  src/indicators/atr.rs:329-460
//   ADX  src/indicators/adx.rs:299-422
//   SMMA src/indicators/moving_averages/smma.rs:243-271
//   Wilders src/indicators/moving_averages/wilders.rs:262-320
// so a lane that starts exactly at first_valid reproduces the oracle's f64
// values and only rounds them to f32 on output.
//
// Time parallelism: the series is cut into chunks of L bars, one wave per
// (64 streams, chunk).  A wave whose chunk starts far enough after the
// warm-up begins K bars early with an approximate state and discards those
// outputs ("burn-in").  All four recurrences contract the state error by
// beta = 1 - 1/p (EMA: 1 - 2/(p+1)) per bar, so after K >= 20 / -ln(beta)
// bars (ADX, two coupled stages: 32 / -ln(beta)) the error is below
// e^-20 ~ 2.1e-9 of the state: ~30x under f32 rounding of the output and four
// orders under the 1e-5 parity bound.  This holds only when
// every bar after first_valid is finite (non-finite bars stop EMA decay and
// poison ATR forever), so each stream carries a "clean" flag; an unclean
// stream always starts exactly at first_valid.
//
// One-series batches use an exact chunked scan instead when the series is
// clean (see "chunked scan" below): no lane replays bars outside its chunk, so
// the chunk length is chosen for waves in flight alone.
#include "vta_common.h"

struct rec_args {
    const float *x;          // close / prices
    const float *h;          // high (ATR, ADX)
    const float *l;          // low  (ATR, ADX)
    const int32_t *periods;  // batch: per combo; many-series: [0] only
    const int32_t *fvs;      // many-series: per series
    const int32_t *clean;    // many-series: per series; batch: scan_flags; NULL: not clean
    const int32_t *fvs2;     // fused kernel: per-series first_valid of (high, low, close)
    float *out0;
    float *out1;
    float *out2;
    double *carry;           // batch scan: [chunk][state][64 x groups] chunk-end states, then
                             // [span][state][64 x groups] the spans'
    const double *terms;     // batch scan: per-bar terms from bar t0 on (scan_term_at)
    const double *state_in;  // batch scan: [state][64 x groups] before bar t0, or NULL
    double *state_out;       // batch scan: the same after bar t1 - 1, or NULL
    const float *alphas;     // EMA / Wilders: caller's smoothing factor (batch: per combo,
                             // many-series: [0]); NULL derives it from the period
    int T;                   // bars
    int nlanes;              // combos (batch) or series (many-series)
    int chunk;               // bars per chunk
    int p1, p2, p3;          // fused kernel periods (EMA, RSI, ATR)
    int fv;                  // batch: first_valid
    int nch, groups;         // batch: chunks, groups of 64 combos
    int span;                // batch scan: chunks per span, 0 without spans
    int t0, t1;              // batch scan: the bars of this launch
    int tstride;
    int scan;                // batch: 0 burn-in / exact lanes, else the scan (ADX: stage 1 or 2)
    int epoch;               // batch: of the call, 0: counted on the device (scan_flags)
    int last;                // batch: the call's last output pass
    int pad_;
};

// Words of a one-series batch's flags, and of a pack's after its jobs'.  A flag
// is set where it holds the call's epoch, so that no word needs clearing.  The
// host counts the epochs of calls that it launches (from 1).  Those of a
// captured call, whose arguments are the same at every replay, are counted on
// the device, with flags of their own (0.3 us more on an 18 us call): the
// launches before the output pass take SF_LAST + 1; scan_states (scan_prepare
// where there is none) leaves it in SF_EPOCH, where the output pass reads it,
// and the call's last output pass copies it to SF_LAST: no launch reads a word
// that it writes.  (A repeated epoch can only read a clean series as unclean,
// which then runs exactly from first_valid.)
enum scan_flags { SF_BAD, SF_ODD, SF_EPOCH, SF_LAST };

#define REC_NAN __builtin_bit_cast(double, 0x7ff8000000000000ull)

__device__ __forceinline__ bool fin(double v) { return vta_isfinite_d(v); }

// Burn-in length in nats of state decay: the carried error of a burnt-in
// start is below e^-20 ~ 2.1e-9 of the state, ~30x under the f32 rounding of
// an output and four orders under the 1e-5 parity bound (ADX, whose two
// coupled stages compound the error, uses 32).
#define REC_NATS 20.0

__device__ __forceinline__ int burn_bars(double beta, double nats) {
    if (!(beta > 0.0)) return 1;
    double k = nats / -log(beta);
    if (k > 1.0e8) return 100000000;
    return max(1, (int)ceil(k));
}

// Bars t of [c0, c1) with t >= from.
__device__ __forceinline__ int bars_from(int c0, int c1, int from) {
    return max(0, c1 - max(c0, from));
}

// ---------------------------------------------------------------- engines

struct EmaEng {
    static constexpr bool kSeedScan = false;
    double alpha, beta, prev;
    int p, fv, vc;
    __device__ void setup(int p_, int fv_) {
        p = p_; fv = fv_;
        alpha = 2.0 / ((double)p + 1.0);
        beta = 1.0 - alpha;
    }
    __device__ void set_alpha(double a_) { alpha = a_; beta = 1.0 - a_; }
    __device__ int kb() const { return burn_bars(beta, REC_NATS); }
    __device__ int exact_start() const { return fv; }
    __device__ int burn_ok_from() const { return fv + p; }   // b >= this may burn in
    // exact start at bar fv
    __device__ double begin_exact(double x) { prev = x; vc = 1; return prev; }
    __device__ void begin_burn(double x) { prev = fin(x) ? x : 0.0; vc = p; }
    __device__ double step(int t, double x) {
        if (t < fv + p) {                       // running-mean warm-up (ema.rs:441-452)
            if (fin(x)) {
                vc += 1;
                double v = (double)vc;
                prev = ((v - 1.0) * prev + x) / v;
            }
        } else if (fin(x)) {
            prev = fma(beta, prev, alpha * x);  // ema.rs:458-466
        }
        return prev;
    }
    __device__ double out_before_start(int t) const { return REC_NAN; }
    static constexpr int kPre = 0;
    // steps t < seed_end() after the start are the warm-up accumulation only
    __device__ int seed_end() const { return fv + p; }
    __device__ double seed_step(int t, double x) {
        if (fin(x)) {
            vc += 1;
            double v = (double)vc;
            prev = ((v - 1.0) * prev + x) / v;
        }
        return prev;
    }
    // the step for t >= burn_ok_from() (no warm-up branches)
    __device__ double steady(double x) {
        if (fin(x)) prev = fma(beta, prev, alpha * x);
        return prev;
    }
};

// num / den for den > 0: an f32 reciprocal estimate refined by one f64 Newton
// step (relative error ~1e-14 instead of the IEEE division sequence; the
// outputs are f32).
__device__ __forceinline__ double rec_ratio(double num, double den) {
    if (!(den > 1e-30 && den < 1e30)) return num / den;   // outside the f32 estimate's range
    double r = (double)__builtin_amdgcn_rcpf((float)den);
    r = fma(fma(-den, r, 1.0), r, r);
    return num * r;
}

// RSI output 100 ag / (ag + al) (50 when the denominator is 0), formed in
// f32 from the f64 averages: both rounded to f32, their f32 sum, a
// reciprocal estimate refined by one Newton step and two f32 products --
// within ~6 ulp of f32 (~4e-7 relative; the output is f32, the parity bound
// 1e-5).  A sum outside [1e-30, 1e30] takes the f64 quotient (and 50 for a
// zero denominator).  The ratio is an output only; the state stays f64.
__device__ __forceinline__ float rsi_ratio_f32(double ag, double al) {
    const float a = (float)ag, b = (float)al;
    const float den = a + b;
    if (!(den > 1e-30f && den < 1e30f)) {
        const double dd = ag + al;
        return dd == 0.0 ? 50.0f : (float)(100.0 * ag / dd);
    }
    float r = __builtin_amdgcn_rcpf(den);
    r = fmaf(fmaf(-den, r, 1.0f), r, r);
    return (100.0f * a) * r;
}

// DX = 100 |+DM - -DM| / (+DM + -DM) for den > 0, divided in f32 (reciprocal
// estimate and one Newton step, <= ~2 ulp of f32); outside the estimate's
// range the f64 quotient.  Each DX enters the ADX as a weighted mean, so its
// ~1e-7 relative error is not amplified.
__device__ __forceinline__ double dx_ratio(double num, double den) {
    if (!(den > 1e-30 && den < 1e30)) return num / den;
    const float d = (float)den;
    float r = __builtin_amdgcn_rcpf(d);
    r = fmaf(fmaf(-d, r, 1.0f), r, r);
    return (double)((float)num * r);
}

struct RsiEng {
    static constexpr bool kSeedScan = true;
    double inv_p, beta, ag, al, px;
    int p, fv;
    bool poisoned;
    __device__ void setup(int p_, int fv_) {
        p = p_; fv = fv_;
        inv_p = 1.0 / (double)p;
        beta = 1.0 - inv_p;
        poisoned = false;
    }
    __device__ int kb() const { return burn_bars(beta, REC_NATS); }
    __device__ int exact_start() const { return fv; }
    __device__ int burn_ok_from() const { return fv + p + 1; }
    __device__ double begin_exact(double x) { px = x; ag = 0.0; al = 0.0; return REC_NAN; }
    __device__ void begin_burn(double x) { px = x; ag = 0.0; al = 0.0; }
    // the seed window (fv, fv+p] has a non-finite delta -> NaN forever (rsi.rs:340-361)
    __device__ void seed_scan(int t, double x) {
        if (t > fv && t <= fv + p && !fin(x - px)) poisoned = true;
        px = x;
    }
    __device__ double step(int t, double x) {
        double d = x - px;
        px = x;
        if (t <= fv + p) {
            if (!poisoned) {
                if (!fin(d)) poisoned = true;
                else if (d > 0.0) ag += d;
                else if (d < 0.0) al -= d;
            }
            if (t < fv + p) return REC_NAN;
            if (poisoned) { ag = REC_NAN; al = REC_NAN; return REC_NAN; }
            ag *= inv_p;
            al *= inv_p;
        } else {
            double g = d > 0.0 ? d : 0.0;
            double lo = d < 0.0 ? -d : 0.0;
            ag = fma(ag, beta, inv_p * g);
            al = fma(al, beta, inv_p * lo);
        }
        if (poisoned) return REC_NAN;
        return (double)rsi_ratio_f32(ag, al);
    }
    static constexpr int kPre = 0;
    __device__ int seed_end() const { return fv + p; }
    __device__ double seed_step(int t, double x) {
        double d = x - px;
        px = x;
        if (!poisoned) {
            if (!fin(d)) poisoned = true;
            else if (d > 0.0) ag += d;
            else if (d < 0.0) al -= d;
        }
        return REC_NAN;
    }
    __device__ double steady(double x) {
        double d = x - px;
        px = x;
        double g = d > 0.0 ? d : 0.0;
        double lo = d < 0.0 ? -d : 0.0;
        ag = fma(ag, beta, inv_p * g);
        al = fma(al, beta, inv_p * lo);
        if (poisoned) return REC_NAN;
        return (double)rsi_ratio_f32(ag, al);
    }
};

__device__ __forceinline__ double true_range(double hi, double lo, double pc) {
    double tr = hi - lo;
    double hc = fabs(hi - pc);
    if (hc > tr) tr = hc;
    double lc = fabs(lo - pc);
    if (lc > tr) tr = lc;
    return tr;
}

struct AtrEng {
    static constexpr bool kSeedScan = false;
    double alpha, sum, rma, pc;
    int p, fv;
    __device__ void setup(int p_, int fv_) {
        p = p_; fv = fv_;
        alpha = 1.0 / (double)p;
    }
    __device__ int kb() const { return burn_bars(1.0 - alpha, REC_NATS); }
    __device__ int exact_start() const { return fv; }
    __device__ int burn_ok_from() const { return fv + p; }
    __device__ double begin_exact(double h, double l, double c) {
        sum = h - l;
        pc = c;
        if (p == 1) { rma = sum / (double)p; return rma; }
        return REC_NAN;
    }
    __device__ void begin_burn(double h, double l, double c) { rma = h - l; pc = c; }
    __device__ double step(int t, double h, double l, double c) {
        double tr = true_range(h, l, pc);
        pc = c;
        if (t < fv + p - 1) { sum += tr; return REC_NAN; }
        if (t == fv + p - 1) { sum += tr; rma = sum / (double)p; return rma; }
        rma = fma(-alpha, rma, rma) + alpha * tr;  // atr.rs:393
        return rma;
    }
    static constexpr int kPre = 1;
    __device__ int seed_end() const { return fv + p - 1; }
    __device__ double seed_step(int t, double h, double l, double c) {
        sum += true_range(h, l, pc);
        pc = c;
        return REC_NAN;
    }
    __device__ double steady(double h, double l, double c) {
        double tr = true_range(h, l, pc);
        pc = c;
        rma = fma(-alpha, rma, rma) + alpha * tr;
        return rma;
    }
    // per-bar term shared by every combo: the true range of bar t
    static __device__ void pre(double h, double l, double, double, double, double pc, double *o) {
        o[0] = true_range(h, l, pc);
    }
    __device__ void set_prev(double, double, double c) { pc = c; }
    __device__ double steady_pre(const double *o) {
        rma = fma(-alpha, rma, rma) + alpha * o[0];
        return rma;
    }
};

// ATR fed by a precomputed true-range series (atr_wrapper.rs:626-700,
// atr_batch_device_with_tr): seed = mean of tr[fv .. fv+p) at fv+p-1, then
// the Wilder update of atr.rs:393 on tr.
struct AtrTrEng {
    static constexpr bool kSeedScan = false;
    double alpha, sum, rma;
    int p, fv;
    __device__ void setup(int p_, int fv_) {
        p = p_; fv = fv_;
        alpha = 1.0 / (double)p;
    }
    __device__ int kb() const { return burn_bars(1.0 - alpha, REC_NATS); }
    __device__ int exact_start() const { return fv; }
    __device__ int burn_ok_from() const { return fv + p; }
    __device__ double begin_exact(double tr) {
        sum = tr;
        if (p == 1) { rma = sum; return rma; }
        return REC_NAN;
    }
    __device__ void begin_burn(double tr) { rma = tr; }
    __device__ double step(int t, double tr) {
        if (t < fv + p - 1) { sum += tr; return REC_NAN; }
        if (t == fv + p - 1) { sum += tr; rma = sum / (double)p; return rma; }
        rma = fma(-alpha, rma, rma) + alpha * tr;
        return rma;
    }
    __device__ double out_before_start(int t) const { return REC_NAN; }
    static constexpr int kPre = 0;
    __device__ int seed_end() const { return fv + p - 1; }
    __device__ double seed_step(int t, double tr) {
        sum += tr;
        return REC_NAN;
    }
    __device__ double steady(double tr) {
        rma = fma(-alpha, rma, rma) + alpha * tr;
        return rma;
    }
};

struct AdxEng {
    static constexpr bool kSeedScan = false;
    double rp, omr, pm1, atr, pds, mds, dx_sum, adx, ph, pl, pc;
    int p, fv, dx_count;
    __device__ void setup(int p_, int fv_) {
        p = p_; fv = fv_;
        double pf = (double)p;
        rp = 1.0 / pf;
        omr = 1.0 - rp;
        pm1 = pf - 1.0;
    }
    __device__ int kb() const { return burn_bars(omr, 32.0); }
    __device__ int exact_start() const { return fv; }
    __device__ int burn_ok_from() const { return fv + 2 * p; }
    __device__ double begin_exact(double h, double l, double c) {
        atr = 0.0; pds = 0.0; mds = 0.0; dx_sum = 0.0; adx = 0.0; dx_count = 0;
        ph = h; pl = l; pc = c;
        return REC_NAN;
    }
    __device__ void begin_burn(double h, double l, double c) {
        atr = 0.0; pds = 0.0; mds = 0.0; adx = 0.0; dx_sum = 0.0; dx_count = p;
        ph = h; pl = l; pc = c;
    }
    __device__ double step(int t, double ch, double cl, double cc) {
        double hl = ch - cl;
        double hpc = fabs(ch - pc);
        double lpc = fabs(cl - pc);
        double tr = fmax(fmax(hl, hpc), lpc);
        double up = ch - ph;
        double down = pl - cl;
        ph = ch; pl = cl; pc = cc;
        int i = t - fv;   // index within the slice starting at first_valid
        if (i <= p) {     // adx.rs:327-348 seed sums
            if (up > down && up > 0.0) pds += up;
            if (down > up && down > 0.0) mds += down;
            atr += tr;
            if (i < p) return REC_NAN;
            double pdi = 0.0, mdi = 0.0;
            if (atr != 0.0) { pdi = (pds / atr) * 100.0; mdi = (mds / atr) * 100.0; }
            double sdi = pdi + mdi;
            dx_sum = sdi != 0.0 ? (fabs(pdi - mdi) / sdi) * 100.0 : 0.0;
            dx_count = 1;
            return REC_NAN;
        }
        double pdm = (up > down && up > 0.0) ? up : 0.0;
        double mdm = (down > up && down > 0.0) ? down : 0.0;
        atr = atr * omr + tr;
        pds = pds * omr + pdm;
        mds = mds * omr + mdm;
        // DX = 100 |DI+ - DI-| / (DI+ + DI-) with DI = 100 DM / ATR: the ATR
        // cancels, leaving one ratio (zero when ATR or DM+ + DM- is zero, as
        // adx.rs:370-390 gives)
        const double sdm = pds + mds;
        double dx = (atr != 0.0 && sdm != 0.0) ? dx_ratio(100.0 * fabs(pds - mds), sdm) : 0.0;
        if (dx_count < p) {
            dx_sum += dx;
            dx_count += 1;
            if (dx_count == p) { adx = dx_sum * rp; return adx; }
            return REC_NAN;
        }
        adx = (adx * pm1 + dx) * rp;
        return adx;
    }
    static constexpr int kPre = 3;
    __device__ int seed_end() const { return fv + p; }
    __device__ double seed_step(int t, double ch, double cl, double cc) {
        double hl = ch - cl;
        double hpc = fabs(ch - pc);
        double lpc = fabs(cl - pc);
        double tr = fmax(fmax(hl, hpc), lpc);
        double up = ch - ph;
        double down = pl - cl;
        ph = ch; pl = cl; pc = cc;
        if (up > down && up > 0.0) pds += up;
        if (down > up && down > 0.0) mds += down;
        atr += tr;
        return REC_NAN;
    }
    __device__ double steady(double ch, double cl, double cc) {
        double hl = ch - cl;
        double hpc = fabs(ch - pc);
        double lpc = fabs(cl - pc);
        double tr = fmax(fmax(hl, hpc), lpc);
        double up = ch - ph;
        double down = pl - cl;
        ph = ch; pl = cl; pc = cc;
        double pdm = (up > down && up > 0.0) ? up : 0.0;
        double mdm = (down > up && down > 0.0) ? down : 0.0;
        atr = atr * omr + tr;
        pds = pds * omr + pdm;
        mds = mds * omr + mdm;
        const double sdm = pds + mds;
        double dx = (atr != 0.0 && sdm != 0.0) ? dx_ratio(100.0 * fabs(pds - mds), sdm) : 0.0;
        adx = (adx * pm1 + dx) * rp;
        return adx;
    }
    // per-bar terms shared by every combo: the true range, +DM and -DM of bar t
    static __device__ void pre(double ch, double cl, double, double ph_, double pl_, double pc_,
                               double *o) {
        double hl = ch - cl;
        double hpc = fabs(ch - pc_);
        double lpc = fabs(cl - pc_);
        o[0] = fmax(fmax(hl, hpc), lpc);
        double up = ch - ph_;
        double down = pl_ - cl;
        o[1] = (up > down && up > 0.0) ? up : 0.0;
        o[2] = (down > up && down > 0.0) ? down : 0.0;
    }
    __device__ void set_prev(double h, double l, double c) { ph = h; pl = l; pc = c; }
    __device__ double steady_pre(const double *o) {
        atr = atr * omr + o[0];
        pds = pds * omr + o[1];
        mds = mds * omr + o[2];
        const double sdm = pds + mds;
        double dx = (atr != 0.0 && sdm != 0.0) ? dx_ratio(100.0 * fabs(pds - mds), sdm) : 0.0;
        adx = (adx * pm1 + dx) * rp;
        return adx;
    }
};

// SMMA (smma.rs:243-271): the mean of the first p bars at fv+p-1, then
// prev = (prev*(p-1) + x) / p (here times 1/p).  p = 1 copies the input.
struct SmmaEng {
    static constexpr bool kSeedScan = false;
    double pm1, rp, prev, sum;
    int p, fv;
    __device__ void setup(int p_, int fv_) {
        p = p_; fv = fv_;
        pm1 = (double)p - 1.0;
        rp = 1.0 / (double)p;
    }
    __device__ int kb() const { return burn_bars(1.0 - rp, REC_NATS); }
    __device__ int exact_start() const { return fv; }
    __device__ int burn_ok_from() const { return fv + p; }
    __device__ double begin_exact(double x) {
        sum = x;
        prev = x;
        if (p == 1) return x;
        return REC_NAN;
    }
    __device__ void begin_burn(double x) { prev = x; }
    __device__ double step(int t, double x) {
        if (p == 1) { prev = x; return x; }
        const int ws = fv + p - 1;
        if (t < ws) { sum += x; return REC_NAN; }
        if (t == ws) { sum += x; prev = sum / (double)p; return prev; }
        prev = (prev * pm1 + x) * rp;
        return prev;
    }
    __device__ double out_before_start(int t) const { return REC_NAN; }
    static constexpr int kPre = 0;
    __device__ int seed_end() const { return p == 1 ? fv : fv + p - 1; }
    __device__ double seed_step(int t, double x) {
        sum += x;
        return REC_NAN;
    }
    __device__ double steady(double x) {
        if (p == 1) { prev = x; return x; }
        prev = (prev * pm1 + x) * rp;
        return prev;
    }
};

// Wilders (wilders.rs:262-320): seed summed in groups of four,
// sum += ((x0 + x1) + x2) + x3, y = sum * (1/p) at fv+p-1, then
// y = fma(x - y, 1/p, y).  p = 1 copies after the seed bar.
struct WildersEng {
    static constexpr bool kSeedScan = false;
    double al, y, sum, g;
    int p, fv;
    __device__ void setup(int p_, int fv_) {
        p = p_; fv = fv_;
        al = 1.0 / (double)p;
    }
    __device__ void set_alpha(double a_) { al = a_; }
    __device__ int kb() const { return burn_bars(1.0 - al, REC_NATS); }
    __device__ int exact_start() const { return fv; }
    __device__ int burn_ok_from() const { return fv + p; }
    __device__ double seed_bar(int k, double x) {       // k = t - fv < p
        if ((k & 3) == 0) g = x; else g += x;
        if ((k & 3) == 3 || k == p - 1) sum += g;
        if (k == p - 1) { y = sum * al; return y; }
        return REC_NAN;
    }
    __device__ double begin_exact(double x) { sum = 0.0; return seed_bar(0, x); }
    __device__ void begin_burn(double x) { y = x; }
    __device__ double step(int t, double x) {
        const int k = t - fv;
        if (k < p) return seed_bar(k, x);
        if (p == 1) { y = x; return x; }
        y = fma(x - y, al, y);
        return y;
    }
    __device__ double out_before_start(int t) const { return REC_NAN; }
    static constexpr int kPre = 0;
    __device__ int seed_end() const { return fv + p - 1; }
    __device__ double seed_step(int t, double x) { return seed_bar(t - fv, x); }
    __device__ double steady(double x) {
        if (p == 1) { y = x; return x; }
        y = fma(x - y, al, y);
        return y;
    }
};

// ---------------------------------------------------------------- chunk planning

// A caller-supplied smoothing factor (the reference's d_alphas / alpha
// arguments of the EMA and Wilders device forms) replaces the one the engine
// derives from the period; the other engines have none.
template <class E>
__device__ __forceinline__ void apply_alpha(E &e, const float *alphas, int i) {
    if constexpr (__is_same(E, EmaEng) || __is_same(E, WildersEng)) {
        if (alphas) e.set_alpha((double)alphas[i]);
    }
}

// Bar at which a lane starts (exact or burn-in) for chunk [c0, c1).
template <class E>
__device__ __forceinline__ int lane_start(const E &e, int c0, bool clean, bool *burn) {
    int es = e.exact_start();
    if (clean) {
        int b = c0 - e.kb();
        if (b >= e.burn_ok_from() && b > es) { *burn = true; return b; }
    }
    *burn = false;
    return es;
}

// Wave-wide minimum, returned as a scalar (readfirstlane) so loops bounded by
// it keep their induction variables and row addresses in SGPRs.
__device__ __forceinline__ int wave_min(int v) {
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o));
    return __builtin_amdgcn_readfirstlane(v);
}

// ---------------------------------------------------------------- many series (time-major)
//
// grid.x: groups of 64 series, grid.y: chunks.  Lane = series; every load and
// store is one coalesced row segment of the [T][N] matrix.
template <class E, int NIN>
__device__ __forceinline__ void drive_ms(const rec_args &a, int p, float *out) {
    const int lane = threadIdx.x & 63;
    const int s = blockIdx.x * 64 + lane;
    const bool active = s < a.nlanes;
    const int N = a.nlanes;
    const int c0 = blockIdx.y * a.chunk;
    const int c1 = min(c0 + a.chunk, a.T);
    const int fv = active ? a.fvs[s] : a.T;
    const bool clean = active ? (a.clean != nullptr && a.clean[s] != 0) : true;
    E e;
    e.setup(p, fv);
    apply_alpha(e, a.alphas, 0);
    bool burn = false;
    int start = active ? lane_start(e, c0, clean, &burn) : a.T;
    if (start > a.T) start = a.T;
    const int t_begin = wave_min(min(start, c0));
    const int lo = active ? min(start, c0) : a.T - 1;
    const int sc = min(s, N - 1);
    // blocks of 8 bars: the block's loads (rows clamped into [lo, T-1]) are
    // issued before its sequential updates; a block in which every lane is
    // past its start and its warm-up takes the engine's steady update only
    for (int tb = t_begin; tb < c1; tb += 8) {
        double xv[8], hv[8], lv[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const long loff = (long)min(max(tb + k, lo), a.T - 1) * N + sc;
            xv[k] = (double)a.x[loff];
            if (NIN == 3) {
                hv[k] = (double)a.h[loff];
                lv[k] = (double)a.l[loff];
            }
        }
        const bool lean = tb + 8 <= c1 && __all(!active || (start < tb && tb >= e.burn_ok_from()));
        if (lean) {
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                double y;
                if constexpr (NIN == 1) y = e.steady(xv[k]);
                else y = e.steady(hv[k], lv[k], xv[k]);
                if (active && tb + k >= c0) out[(size_t)(tb + k) * N + s] = (float)y;
            }
            continue;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int t = tb + k;
            if (t >= c1) break;
            double y = REC_NAN;
            if (active) {
                if (t == start) {
                    if constexpr (NIN == 1) {
                        if (burn) e.begin_burn(xv[k]); else y = e.begin_exact(xv[k]);
                    } else {
                        if (burn) e.begin_burn(hv[k], lv[k], xv[k]);
                        else y = e.begin_exact(hv[k], lv[k], xv[k]);
                    }
                } else if (t > start) {
                    if constexpr (NIN == 1) y = e.step(t, xv[k]); else y = e.step(t, hv[k], lv[k], xv[k]);
                }
                if (t >= c0) out[(size_t)t * N + s] = (float)y;
            }
        }
    }
}

// RSI burn-in needs the seed-window NaN check, done by a short scan first.
__device__ __forceinline__ void drive_ms_rsi(const rec_args &a, int p, float *out) {
    const int lane = threadIdx.x & 63;
    const int s = blockIdx.x * 64 + lane;
    const bool active = s < a.nlanes;
    const int N = a.nlanes;
    const int c0 = blockIdx.y * a.chunk;
    const int c1 = min(c0 + a.chunk, a.T);
    const int fv = active ? a.fvs[s] : a.T;
    const bool clean = active ? (a.clean != nullptr && a.clean[s] != 0) : true;
    RsiEng e;
    e.setup(p, fv);
    bool burn = false;
    int start = active ? lane_start(e, c0, clean, &burn) : a.T;
    if (burn) {
        e.px = (double)a.x[(size_t)fv * N + s];
        for (int t = fv + 1; t <= min(fv + p, a.T - 1); ++t) e.seed_scan(t, (double)a.x[(size_t)t * N + s]);
    }
    const int t_begin = wave_min(min(start, c0));
    for (int t = t_begin; t < c1; ++t) {
        const size_t off = (size_t)t * N + s;
        const double x = (double)a.x[(long)min(max(t, active ? min(start, c0) : a.T - 1),
                                               a.T - 1) * N + min(s, N - 1)];
        double y = REC_NAN;
        if (active) {
            if (t == start) {
                if (burn) e.begin_burn(x); else y = e.begin_exact(x);
            } else if (t > start) {
                y = e.step(t, x);
            }
            if (t >= c0) out[off] = (float)y;
        }
    }
}

extern "C" __global__ __launch_bounds__(64) void ema_ms1p_f32(rec_args a) {
    drive_ms<EmaEng, 1>(a, a.periods[0], a.out0);
}
extern "C" __global__ __launch_bounds__(64) void rsi_ms1p_f32(rec_args a) {
    drive_ms_rsi(a, a.periods[0], a.out0);
}
extern "C" __global__ __launch_bounds__(64) void atr_ms1p_f32(rec_args a) {
    drive_ms<AtrEng, 3>(a, a.periods[0], a.out0);
}
extern "C" __global__ __launch_bounds__(64) void smma_ms1p_f32(rec_args a) {
    drive_ms<SmmaEng, 1>(a, a.periods[0], a.out0);
}
extern "C" __global__ __launch_bounds__(64) void wilders_ms1p_f32(rec_args a) {
    drive_ms<WildersEng, 1>(a, a.periods[0], a.out0);
}
extern "C" __global__ __launch_bounds__(64) void adx_ms1p_f32(rec_args a) {
    drive_ms<AdxEng, 3>(a, a.periods[0], a.out0);
}

// ---------------------------------------------------------------- fused EMA + RSI + ATR
//
// One pass over close/high/low [T][N]: EMA(p1) and RSI(p2) of close and
// ATR(p3) of (high, low, close), three time-major outputs.
//
// Every lane has a bar `steady` from which its three engines are in pure
// recurrence.  Each bar, lanes at or past it run the lean update (three
// recurrences, no phase checks, the RSI ratio divided in f32 via rcp + one
// Newton step: <= ~2 ulp of f32, far inside the 1e-5 bound); lanes still in a
// warm-up run the general engines.  When every lane of the wave is steady the
// general path is skipped entirely, so a series start costs its own lane ~p
// general bars.  Loads of the next U rows are issued before the current U
// rows are consumed (register double buffering); addresses are clamped so
// the loads are unconditional and stay in flight.  U = 8 keeps the kernel at
// 167 VGPRs (3 waves per SIMD); U = 16 (185 VGPRs, 2 waves) was 1.5% slower
// on 4,096 x 50,000, U = 32 (286 VGPRs) holds one wave.
#define FUSED_U 8


extern "C" __global__ __launch_bounds__(64) void ms_ema_rsi_atr_f32(rec_args a) {
    const int lane = threadIdx.x & 63;
    const int s = blockIdx.x * 64 + lane;
    const bool active = s < a.nlanes;
    const int N = a.nlanes;
    const int c0 = blockIdx.y * a.chunk;
    const int c1 = min(c0 + a.chunk, a.T);
    const int fv = active ? a.fvs[s] : a.T;          // first non-NaN close
    const int fv3 = active ? a.fvs2[s] : a.T;        // first bar with high, low, close
    const bool clean = active ? (a.clean != nullptr && a.clean[s] != 0) : true;
    const bool live = active && fv < c1;             // has an output in this chunk
    EmaEng ee; RsiEng re; AtrEng ae;
    ee.setup(a.p1, fv); re.setup(a.p2, fv); ae.setup(a.p3, fv3);
    bool be = false, br = false, ba = false;
    int se = live ? lane_start(ee, c0, clean, &be) : a.T;
    int sr = live ? lane_start(re, c0, clean, &br) : a.T;
    int sa = live ? lane_start(ae, c0, clean, &ba) : a.T;
    if (br) {
        re.px = (double)a.x[(size_t)fv * N + s];
        for (int t = fv + 1; t <= min(fv + a.p2, a.T - 1); ++t)
            re.seed_scan(t, (double)a.x[(size_t)t * N + s]);
    }
    int steady = a.T;
    if (live && clean) {
        steady = max(be ? se + 1 : fv + a.p1, br ? sr + 1 : fv + a.p2 + 1);
        steady = max(steady, ba ? sa + 1 : fv3 + a.p3);
    }
    const int smin = live ? min(min(se, sr), min(sa, c0)) : c0;
    const int t_begin = wave_min(smin);
    // bars before a lane's first engine start need no work at all
    const int lane_first = live ? min(min(se, sr), sa) : a.T;
    const bool rsi_nan_fixed = re.poisoned;
    const int sc = min(s, N - 1);
    // Row addresses are wave-uniform (scalar base + 32-bit lane offset).

    float bc[FUSED_U], bh[FUSED_U], bl[FUSED_U];
    float nc[FUSED_U], nh[FUSED_U], nl[FUSED_U];
#pragma unroll
    for (int u = 0; u < FUSED_U; ++u) {
        const size_t rb = (size_t)min(t_begin + u, a.T - 1) * (size_t)N;
        bc[u] = (a.x + rb)[sc];
        bh[u] = (a.h + rb)[sc];
        bl[u] = (a.l + rb)[sc];
    }
    for (int t0 = t_begin; t0 < c1; t0 += FUSED_U) {
#pragma unroll
        for (int u = 0; u < FUSED_U; ++u) {
            const size_t rb = (size_t)min(t0 + FUSED_U + u, a.T - 1) * (size_t)N;
            nc[u] = (a.x + rb)[sc];
            nh[u] = (a.h + rb)[sc];
            nl[u] = (a.l + rb)[sc];
        }
        // wave-uniform: does any lane have warm-up bars inside this block?
        const bool mixed = __any(live && lane_first < t0 + FUSED_U && steady > t0);
        if (!mixed) {
            // every live lane is steady for the whole block, or has not started
            // (its state is rebuilt when it starts, so updating it is harmless)
#pragma unroll
            for (int u = 0; u < FUSED_U; ++u) {
                const int t = t0 + u;
                const double x = bc[u], hh = bh[u], ll = bl[u];
                ee.prev = fma(ee.beta, ee.prev, ee.alpha * x);          // ema.rs:462
                const double d = x - re.px;
                re.px = x;
                re.ag = fma(re.ag, re.beta, re.inv_p * (d > 0.0 ? d : 0.0));  // rsi.rs:377
                re.al = fma(re.al, re.beta, re.inv_p * (d < 0.0 ? -d : 0.0));
                const double tr = true_range(hh, ll, ae.pc);
                ae.pc = x;
                ae.rma = fma(-ae.alpha, ae.rma, ae.rma) + ae.alpha * tr;      // atr.rs:393
                const bool ok = t >= steady;
                const float o0 = ok ? (float)ee.prev : VTA_QNAN_F32;
                const float o1 = (ok && !rsi_nan_fixed) ? rsi_ratio_f32(re.ag, re.al)
                                                        : VTA_QNAN_F32;
                const float o2 = ok ? (float)ae.rma : VTA_QNAN_F32;
                if (t >= c0 && t < c1 && active) {
                    const size_t rb = (size_t)t * (size_t)N;
                    (a.out0 + rb)[s] = o0;
                    (a.out1 + rb)[s] = o1;
                    (a.out2 + rb)[s] = o2;
                }
            }
        } else {
#pragma unroll
        for (int u = 0; u < FUSED_U; ++u) {
            const int t = t0 + u;
            if (t >= c1) break;
            const double x = bc[u], hh = bh[u], ll = bl[u];
            float o0 = VTA_QNAN_F32, o1 = VTA_QNAN_F32, o2 = VTA_QNAN_F32;
            if (t >= steady) {
                // lean steady-state update (clean, started lanes only)
                ee.prev = fma(ee.beta, ee.prev, ee.alpha * x);          // ema.rs:462
                const double d = x - re.px;
                re.px = x;
                re.ag = fma(re.ag, re.beta, re.inv_p * (d > 0.0 ? d : 0.0));  // rsi.rs:377
                re.al = fma(re.al, re.beta, re.inv_p * (d < 0.0 ? -d : 0.0));
                const double tr = true_range(hh, ll, ae.pc);
                ae.pc = x;
                ae.rma = fma(-ae.alpha, ae.rma, ae.rma) + ae.alpha * tr;      // atr.rs:393
                o0 = (float)ee.prev;
                o1 = rsi_nan_fixed ? VTA_QNAN_F32 : rsi_ratio_f32(re.ag, re.al);
                o2 = (float)ae.rma;
            } else if (t >= lane_first) {
                double y0 = REC_NAN, y1 = REC_NAN, y2 = REC_NAN;
                if (t == se) { if (be) ee.begin_burn(x); else y0 = ee.begin_exact(x); }
                else if (t > se) y0 = ee.step(t, x);
                if (t == sr) { if (br) re.begin_burn(x); else y1 = re.begin_exact(x); }
                else if (t > sr) y1 = re.step(t, x);
                if (t == sa) { if (ba) ae.begin_burn(hh, ll, x); else y2 = ae.begin_exact(hh, ll, x); }
                else if (t > sa) y2 = ae.step(t, hh, ll, x);
                o0 = (float)y0;
                o1 = (float)y1;
                o2 = (float)y2;
            }
            if (active && t >= c0) {
                const size_t off = (size_t)t * N + s;
                a.out0[off] = o0;
                a.out1[off] = o1;
                a.out2[off] = o2;
            }
        }
        }
#pragma unroll
        for (int u = 0; u < FUSED_U; ++u) { bc[u] = nc[u]; bh[u] = nh[u]; bl[u] = nl[u]; }
    }
}

// ---------------------------------------------------------------- one series, many params
//
// Lane = combo.  What one block of a one-series batch works on: the series,
// the combos' periods and outputs, the chunking, and which combo group and
// chunk this block is.
struct batch_view {
    const float *x, *h, *l;
    const int32_t *periods;
    const float *alphas;     // per combo, or NULL (see apply_alpha)
    double *carry;           // see rec_args
    const double *terms, *state_in;
    double *state_out;
    int T, nlanes, chunk, nch, groups, span, fv, t0, t1, tstride, scan, group;
    int kb, k;               // the block's first chunk, this wave's
    int32_t epoch;           // see scan_flags
    bool clean, odd, coop;
};

// A block is REC_WPB waves: with that many combo groups, one chunk of as many
// groups, whose waves then read the same terms (one miss of the scalar cache
// for four); else consecutive chunks of one group, which share the work of
// folding the chunks before them (`coop`).
#define REC_WPB 4
__device__ __forceinline__ int block_wave() {
    return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}
__device__ __forceinline__ void block_chunk(batch_view &v, int flat) {
    v.coop = v.groups < REC_WPB;
    if (v.coop) {
        const int per = (v.nch + REC_WPB - 1) / REC_WPB;
        v.group = flat / per;
        v.kb = flat % per * REC_WPB;
        v.k = v.kb + block_wave();
    } else {
        v.group = flat / v.nch * REC_WPB + block_wave();
        v.kb = v.k = flat % v.nch;
    }
}
// Whether the wave has a chunk at all.
__device__ __forceinline__ bool wave_idle(const batch_view &v) {
    return v.k >= v.nch || v.group >= v.groups;
}

// The view of a wave of a direct launch (OUT: the output pass): the blocks of a
// group in order.
template <bool OUT>
__device__ __forceinline__ batch_view view_of(const rec_args &a) {
    batch_view v;
    v.x = a.x; v.h = a.h; v.l = a.l;
    v.periods = a.periods;
    v.alphas = a.alphas;
    v.carry = a.carry;
    v.terms = a.terms;
    v.state_in = a.state_in;
    v.state_out = a.state_out;
    v.T = a.T;
    v.nlanes = a.nlanes;
    v.chunk = a.chunk;
    v.nch = a.nch;
    v.groups = a.groups;
    v.span = a.span;
    v.fv = a.fv;
    v.t0 = a.t0;
    v.t1 = a.t1;
    v.tstride = a.tstride;
    v.scan = a.scan;
    block_chunk(v, blockIdx.x);
    v.clean = v.odd = false;
    v.epoch = 0;
    if (a.clean) {
        v.epoch = a.epoch ? a.epoch : OUT ? a.clean[SF_EPOCH] : a.clean[SF_LAST] + 1;
        v.clean = a.clean[SF_BAD] != v.epoch;
        v.odd = a.clean[SF_ODD] == v.epoch;
    }
    return v;
}

// LDS of a wave, dynamic (batch_lds_bytes, rec.cpp): the bars or the per-bar
// terms formed from them, and the 64-row output staging of drive_batch; the
// scan's output pass has its own staging in the same bytes (at most 10 KiB, so
// that four blocks of four waves fit a CU).
#define REC_STAGE 33         // floats per staged row of drive_batch (32 bars + 1)
#define REC_ROW 36           // floats per row staged by scan_output (16-byte rows)
template <class E>
__device__ __forceinline__ double *wave_lds() {
    constexpr int drive = (E::kPre > 1 ? E::kPre * 512 : 3 * 256) + 64 * REC_STAGE * 4;
    constexpr int scan = 64 * REC_ROW * 4;
    extern __shared__ __align__(16) double rec_lds[];
    return rec_lds + block_wave() * ((drive > scan ? drive : scan) / 8);
}

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Exact and burn-in lanes: the wave stages 64 bars of the series in LDS (one
// coalesced load, then broadcast reads) and 64 rows x 32 bars of output.  An
// unclean series runs exactly from first_valid.
template <class E, int NIN>
__device__ __forceinline__ void drive_batch(const batch_view &a, float *out) {
    // per-bar terms every combo shares (E::kPre of them, f64): lane j computes
    // them for bar tb + j, so the steady loop reads them instead of
    // recomputing them in every lane
    constexpr int NPRE = E::kPre;
    double *pv = wave_lds<E>();                                    // [NPRE][64], or
    float *xs = reinterpret_cast<float *>(pv);                     // [3][64]
    float *ob = xs + (NPRE > 1 ? NPRE * 128 : 3 * 64);             // [64][REC_STAGE]
    const int lane = threadIdx.x & 63;
    const int c = a.group * 64 + lane;
    const bool active = c < a.nlanes;
    const int T = a.T;
    const int c0 = a.k * a.chunk;
    const int c1 = min(c0 + a.chunk, T);
    const int fv = a.fv;
    const int p = active ? a.periods[c] : 1;
    E e;
    e.setup(p, fv);
    if (active) apply_alpha(e, a.alphas, c);
    bool burn = false;
    const int start = active ? lane_start(e, c0, a.clean, &burn) : T;
    if constexpr (E::kSeedScan) {
        // RSI burn-in: the seed window's NaN rule still has to be seen
        if (burn) {
            e.px = (double)a.x[fv];
            for (int t = fv + 1; t <= min(fv + p, T - 1); ++t) e.seed_scan(t, (double)a.x[t]);
        }
    }
    // rows of bars tb + 32 hh .. + 31, each store two rows x 32 consecutive
    // bars (lane & 31 = bar, lane >> 5 = row parity)
    const int nrow = min(64, a.nlanes - a.group * 64);
    auto flush_half = [&](int tb, int hh) {
        wave_lds_sync();
        const int t = tb + 32 * hh + (lane & 31);
        if (tb + 32 * hh + 32 > c0) {
            const bool ok = t >= c0 && t < c1;
#pragma unroll 4
            for (int i = 0; i < 32; ++i) {
                const int r = 2 * i + (lane >> 5);
                if (ok && r < nrow)
                    out[(size_t)(a.group * 64 + r) * T + t] = ob[r * REC_STAGE + (lane & 31)];
            }
        }
        wave_lds_sync();
    };
    auto emit = [&](int tb, int j, double y) {
        ob[lane * REC_STAGE + (j & 31)] = (float)y;
        if ((j & 31) == 31) flush_half(tb, j >> 5);
    };
    const int t_begin = wave_min(min(start, c0)) & ~63;
    // bars of the next block are loaded into registers while the current one
    // is processed (with the bar before each, for the per-bar terms)
    float nx0, nx1 = 0.0f, nx2 = 0.0f, np0 = 0.0f, np1 = 0.0f, np2 = 0.0f;
    auto load_next = [&](int tb0) {
        const long t = min(tb0 + lane, T - 1);
        nx0 = a.x[t];
        if (NIN == 3) {
            nx1 = a.h[t];
            nx2 = a.l[t];
        }
        if constexpr (NPRE > 0) {
            const long tp = max(t - 1, 0L);
            np0 = a.x[tp];
            if (NIN == 3) {
                np1 = a.h[tp];
                np2 = a.l[tp];
            }
        }
    };
    load_next(t_begin);
    for (int tb = t_begin; tb < c1; tb += 64) {
        // lean path: a full block in which every lane is past its start and
        // its warm-up -- only the engine's steady update
        const bool lean = tb + 64 <= c1 && __all(!active || (start < tb && tb >= e.burn_ok_from()));
        const float lx0 = __shfl(nx0, 63), lx1 = __shfl(nx1, 63), lx2 = __shfl(nx2, 63);
        if (NPRE > 0 && lean) {
            double o[NPRE > 0 ? NPRE : 1];
            if constexpr (NPRE > 0)
                E::pre((double)nx1, (double)nx2, (double)nx0, (double)np1, (double)np2,
                       (double)np0, o);
#pragma unroll
            for (int i = 0; i < NPRE; ++i) pv[i * 64 + lane] = o[i];
        } else {
            xs[lane] = nx0;
            if (NIN == 3) {
                xs[64 + lane] = nx1;
                xs[128 + lane] = nx2;
            }
        }
        wave_lds_sync();
        load_next(tb + 64);
        if (lean) {
          if constexpr (NPRE > 0) {
#pragma unroll 4
            for (int j = 0; j < 64; ++j) {
                double o[NPRE];
#pragma unroll
                for (int i = 0; i < NPRE; ++i) o[i] = pv[i * 64 + j];
                emit(tb, j, e.steady_pre(o));
            }
            e.set_prev((double)lx1, (double)lx2, (double)lx0);
          } else {
#pragma unroll 2
            for (int j = 0; j < 64; j += 4) {
                const float4 x4 = *reinterpret_cast<const float4 *>(&xs[j]);
                emit(tb, j, e.steady(x4.x));
                emit(tb, j + 1, e.steady(x4.y));
                emit(tb, j + 2, e.steady(x4.z));
                emit(tb, j + 3, e.steady(x4.w));
            }
          }
        } else if (tb + 64 <= c1 && __all(!active || (start < tb && tb + 64 <= e.seed_end()))) {
            // every lane still accumulating its warm-up seed for the whole block
#pragma unroll 2
            for (int j = 0; j < 64; j += 4) {
                const float4 x4 = *reinterpret_cast<const float4 *>(&xs[j]);
                if constexpr (NIN == 1) {
                    emit(tb, j, e.seed_step(tb + j, x4.x));
                    emit(tb, j + 1, e.seed_step(tb + j + 1, x4.y));
                    emit(tb, j + 2, e.seed_step(tb + j + 2, x4.z));
                    emit(tb, j + 3, e.seed_step(tb + j + 3, x4.w));
                } else {
                    const float4 h4 = *reinterpret_cast<const float4 *>(&xs[64 + j]);
                    const float4 l4 = *reinterpret_cast<const float4 *>(&xs[128 + j]);
                    emit(tb, j, e.seed_step(tb + j, h4.x, l4.x, x4.x));
                    emit(tb, j + 1, e.seed_step(tb + j + 1, h4.y, l4.y, x4.y));
                    emit(tb, j + 2, e.seed_step(tb + j + 2, h4.z, l4.z, x4.z));
                    emit(tb, j + 3, e.seed_step(tb + j + 3, h4.w, l4.w, x4.w));
                }
            }
        } else
        for (int j = 0; j < 64; ++j) {
            const int t = tb + j;
            double y = REC_NAN;
            if (active && t < c1) {
                const double x = xs[j];
                if (t == start) {
                    if constexpr (NIN == 1) {
                        if (burn) e.begin_burn(x); else y = e.begin_exact(x);
                    } else {
                        if (burn) e.begin_burn(xs[64 + j], xs[128 + j], x);
                        else y = e.begin_exact(xs[64 + j], xs[128 + j], x);
                    }
                } else if (t > start) {
                    if constexpr (NIN == 1) y = e.step(t, x);
                    else y = e.step(t, xs[64 + j], xs[128 + j], x);
                }
            }
            emit(tb, j, y);
        }
        wave_lds_sync();
    }
}

// ---------------------------------------------------------------- chunked scan
//
// A clean series (every bar from first_valid on finite) in chunks of whole
// 64-bar blocks.  Up to a per-combo bar sw the state is the plain sum of the
// bars' terms, after it s = beta s + w f: with the averages kept as sums
// (p times Wilder's average; RSI's and DX's ratios cancel the factor) every
// indicator is s = (t > sw ? beta : 1) s + f, an affine map of the state, and
// the terms f are the same for every combo.  So
//   scan_prepare   forms the terms once per bar in f64 (EMA, SMMA, Wilders the
//                  close, RSI 100 x the gain and the absolute change, ATR the true
//                  range, ADX +DM + -DM, +DM - -DM and the true range: the
//                  ratios' own numerators and denominators), zero before
//                  first_valid,
//   scan_states    runs each chunk from a zero state: one fma per state, bar
//                  and combo, the term a scalar operand,
//   scan_output    folds the chunks before its own in order, s_k = g_k s_{k-1}
//                  + b_k with g_k the product of the chunk's multipliers,
//                  runs its chunk from that exact state and writes it;
//   scan_spans     between them (long scans) folds every `span` chunks into
//                  one map first, so that a wave folds at most the spans and
//                  one span's chunks.
// ADX's second stage (the sum, then the smoothing of DX) is a scan of its own
// over DX: scan_output without stores (scan = 2) gives its chunk states.
// The terms come through the scalar cache: the combos of a wave share them, so
// the vector unit only does the combos' own work, no block stages bars in LDS
// and a warm-up bar costs two selects more than another.  Terms of more
// than the context's buffer holds run in segments [t0, t1), the states passed
// on in state_in / state_out.
//
// Whole calls before (bars staged in LDS and widened in every lane, a launch
// with one wave per combo folding the chunks) and now:
//   1,250 EMA / RSI / ADX x 200k bars (1.0 GB)   282 / 366 / 709 -> 239 / 266 / 448 us
//   33 RSI x 10,007 bars                         59 -> 18 us
//   40 RSI series of up to 50k bars, 74 MB       124 -> 71 us
// The first two are near the rate such rows are written at (~5.2 TB/s, 193
// us); ADX is bound by its two divisions and two f64 rounds per output.

typedef const __attribute__((address_space(4))) double scan_term;

// Per-combo constants of the scan.
struct scan_lane {
    double beta;             // multiplier past sw
    double w;                // weight of a term past sw (EMA alpha, else 1)
    double kap;              // factor on the state at sw (EMA 1 / p, else 1)
    double scale, scale0;    // output = scale s past sw, scale0 s at sw
    int sw;                  // last bar of the plain sum
    int first;               // first bar with an output
    int sw2;                 // ADX: last bar of the DX sum
};

template <class E>
__device__ __forceinline__ scan_lane scan_params(const batch_view &a, int c, bool active) {
    scan_lane q;
    const int p = active ? a.periods[c] : 1;
    const double pf = (double)p;
    q.w = q.kap = q.scale = q.scale0 = 1.0;
    q.sw = a.fv + p - 1;
    q.first = q.sw;
    q.sw2 = 0;
    if constexpr (__is_same(E, EmaEng)) {
        q.w = active && a.alphas ? (double)a.alphas[c] : 2.0 / (pf + 1.0);
        q.beta = 1.0 - q.w;
        q.kap = 1.0 / pf;
        q.first = a.fv;
    } else if constexpr (__is_same(E, WildersEng)) {
        const double al = active && a.alphas ? (double)a.alphas[c] : 1.0 / pf;
        q.beta = p == 1 ? 0.0 : 1.0 - al;        // p = 1 copies after its first bar
        q.scale = p == 1 ? 1.0 : al;
        q.scale0 = al;
    } else if constexpr (__is_same(E, SmmaEng)) {
        q.scale = q.scale0 = 1.0 / pf;
        q.beta = (pf - 1.0) * q.scale;
    } else {
        const double rp = 1.0 / pf;
        q.beta = 1.0 - rp;
        q.scale = q.scale0 = rp;
        if constexpr (__is_same(E, RsiEng)) {
            q.sw = q.first = a.fv + p;
        } else if constexpr (__is_same(E, AdxEng)) {
            q.sw = a.fv + p;
            q.sw2 = a.fv + 2 * p - 1;
            q.first = p == 1 ? a.fv + 2 : q.sw2;
            q.scale = 100.0 * rp;
        }
    }
    return q;
}

template <class E> struct scan_dims {                // terms and first-stage states
    static constexpr int N = __is_same(E, AdxEng) ? 3 : (__is_same(E, RsiEng) ? 2 : 1);
    static constexpr int S = __is_same(E, AdxEng) ? 4 : N;
};

// Wave-wide maximum, as a scalar.
__device__ __forceinline__ int wave_max(int v) { return -wave_min(-v); }

// Where term i of an indicator with n of them is for bar r of the buffer:
// [tstride][2] pairs for two or three terms, then the third's [tstride].
__host__ __device__ __forceinline__ size_t scan_term_at(int n, int i, int tstride, long r) {
    return n == 1 ? (size_t)r : i < 2 ? 2 * (size_t)r + i : 2 * (size_t)tstride + r;
}

// Terms i of bars t, t + 1, ... (every second value for i < 2 of a pair).
template <class E>
__device__ __forceinline__ scan_term *scan_at(const batch_view &a, int i, int t) {
    return (scan_term *)(a.terms + scan_term_at(scan_dims<E>::N, i, a.tstride, t - a.t0));
}

// The N terms of U bars from bar t on.
template <class E, int N, int U>
__device__ __forceinline__ void scan_fetch(const batch_view &a, int t, double (&f)[U][N]) {
    constexpr int step = scan_dims<E>::N == 1 ? 1 : 2;
    scan_term *p = scan_at<E>(a, 0, t);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int i = 0; i < (N < 2 ? N : 2); ++i) f[u][i] = p[u * step + i];
    if constexpr (N > 2) {
        scan_term *q = scan_at<E>(a, 2, t);
#pragma unroll
        for (int u = 0; u < U; ++u) f[u][2] = q[u];
    }
}

// Brings the lines of the terms of bars [c0, c1) into the L2, all at once:
// scalar loads run one or two lines ahead of their use only, and the terms,
// written by another kernel, are in no L2 yet (the passes waited ~1,500 cycles
// on every eight bars).  `keep` takes the values, so that the loads are made.
template <class E>
__device__ __forceinline__ void scan_touch(const batch_view &a, int c0, int c1, double &keep) {
    // (the third term, of odd series only, is left to the scalar loads)
    constexpr int step = scan_dims<E>::N == 1 ? 1 : 2;
    const double *p = a.terms + (size_t)step * (c0 - a.t0);
    for (int r = 16 * (int)(threadIdx.x & 63); r < step * (c1 - c0); r += 64 * 16) {
        const double v = p[r];
        asm volatile("" : "+v"(keep) : "v"(v));
    }
}

// s = beta s + f with the term as a scalar operand (the compiler would move it
// to vector registers first, two more instructions per term).
__device__ __forceinline__ void scan_step(double &s, double beta, double f) {
    double r;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(beta), "v"(s), "s"(f));
    s = r;
}

// beta^n, n >= 0.
__device__ __forceinline__ double scan_pow(double beta, int n) {
    double r = 1.0;
    for (; __any(n > 0); n >>= 1) {
        if (n & 1) r *= beta;
        beta *= beta;
    }
    return r;
}

// One scan of a wave's combos: plain sums up to bar sw (at most `last` over
// the wave), times kap there, then beta.
struct scan_sum {
    double beta, kap;
    int sw, last;
};

// Folds chunks [j, j1) of `chunk` bars onto M states, their loads eight at a
// time ahead of the chain; gg (may be NULL): times their multipliers.  Past the
// chunk that holds the wave's last sum every multiplier is beta^chunk; up
// to it a chunk's is 1, that of its sum's last bar, or beta^chunk by combo.
// `zero`: the states are zero, so the first multiplier does not matter.
template <int M>
__device__ __forceinline__ void scan_chain(const batch_view &a, const scan_sum &q, int chunk,
                                           const double *b, size_t step, size_t cp, int j, int j1,
                                           bool zero, double *s, double *gg) {
    if (j >= j1) return;
    const double gl = scan_pow(q.beta, chunk);
    const int jl = q.last < a.t0 ? -1 : (q.last - a.t0) / chunk;
    double v[M][8];
    auto fetch = [&](int at) {
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int i = 0; i < M; ++i) v[i][u] = b[(size_t)min(at + u, j1 - 1) * step + i * cp];
    };
    if (j <= jl && !(zero && !gg && j == jl)) {
        const int r = q.sw - a.t0;                   // < 0: before this segment
        const int jm = r < 0 ? -1 : r / chunk;
        const double gm = q.kap * scan_pow(q.beta, r < 0 ? 0 : chunk - 1 - r % chunk);
        for (const int m = min(j1, jl + 1); j < m; ++j) {
            const double g = j > jm ? gl : (j == jm ? gm : 1.0);
            if (gg) *gg *= g;
#pragma unroll
            for (int i = 0; i < M; ++i) s[i] = fma(g, s[i], b[(size_t)j * step + i * cp]);
        }
    }
    for (; j < j1; j += 8) {
        fetch(j);
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (j + u < j1) {
                if (gg) *gg *= gl;
#pragma unroll
                for (int i = 0; i < M; ++i) s[i] = fma(gl, s[i], v[i][u]);
            }
    }
}

// The exact states [i0, i0 + M) of combo c at the start of the wave's chunk
// (sum up to bar sw, then beta): the segment's incoming state, the spans, then
// the chunks, in a cooperative block each wave a share of the chunks before
// the block as one affine map (lds: 64 (M + 1) doubles per wave; every wave of
// the block calls it).  NEXT: and in `next` those at the start of the chunk
// after it (if there is one), by the operations of that chunk's own fold.
template <int M, bool NEXT>
__device__ __forceinline__ void scan_start(const batch_view &a, const scan_sum &q, int S, int i0,
                                           int c, double *s, double *next, double *lds) {
    const size_t cp = (size_t)a.groups * 64, step = (size_t)S * cp;
    const double *b = a.carry + (size_t)i0 * cp + c;
    const bool idle = wave_idle(a), zero = a.state_in == nullptr;
#pragma unroll
    for (int i = 0; i < M; ++i)
        s[i] = !zero && !idle ? a.state_in[(size_t)(i0 + i) * cp + c] : 0.0;
    int j = 0;
    if (a.span && !idle) {
        const int n = a.k / a.span;
        scan_chain<M>(a, q, a.chunk * a.span, b + (size_t)a.nch * step, step, cp, 0, n, zero, s,
                      nullptr);
        j = n * a.span;
    }
    double after[M];                                 // NEXT: the states after the spans
    if (NEXT)
#pragma unroll
        for (int i = 0; i < M; ++i) after[i] = s[i];
    // onto `after`, where chunk k opens a span: the span before it
    auto span_before = [&](int k) {
        const int n = k / a.span - 1;
        scan_chain<M>(a, q, a.chunk * a.span, b + (size_t)a.nch * step, step, cp, n, n + 1,
                      zero && n == 0, after, nullptr);
    };
    if (!a.coop) {
        if (idle) return;
        const bool more = NEXT && a.k + 1 < a.nch;
        double bk[M];                                // (loaded ahead of the chain)
        if (more)
#pragma unroll
            for (int i = 0; i < M; ++i) bk[i] = b[(size_t)a.k * step + i * cp];
        scan_chain<M>(a, q, a.chunk, b, step, cp, j, a.k, zero && j == 0, s, nullptr);
        if (more) {
            if (a.span && (a.k + 1) % a.span == 0) {
                span_before(a.k + 1);
#pragma unroll
                for (int i = 0; i < M; ++i) next[i] = after[i];
            } else {
                // the step of scan_chain over chunk k
                const int r = q.sw - a.t0, jm = r < 0 ? -1 : r / a.chunk;
                const int jl = q.last < a.t0 ? -1 : (q.last - a.t0) / a.chunk;
                double g = scan_pow(q.beta, a.chunk);
                if (a.k <= jl && !(zero && a.k == 0 && jl == 0) && a.k <= jm)
                    g = a.k == jm ? q.kap * scan_pow(q.beta, a.chunk - 1 - r % a.chunk) : 1.0;
#pragma unroll
                for (int i = 0; i < M; ++i) next[i] = fma(g, s[i], bk[i]);
            }
        }
        return;
    }
    const int lane = threadIdx.x & 63, w = a.k - a.kb;
    double m[M], gg = 1.0;
#pragma unroll
    for (int i = 0; i < M; ++i) m[i] = 0.0;
    // (an idle wave's share counts too; a span holds whole blocks)
    const int j0 = a.span ? a.kb / a.span * a.span : 0, all = a.kb - j0;
    scan_chain<M>(a, q, a.chunk, b, step, cp, j0 + all * w / REC_WPB,
                  j0 + all * (w + 1) / REC_WPB, false, m, &gg);
    double v[M][REC_WPB - 1];                        // the chunks of the block before this one
#pragma unroll
    for (int u = 0; u < REC_WPB - 1; ++u)
#pragma unroll
        for (int i = 0; i < M; ++i)
            v[i][u] = b[(size_t)min(a.kb + u, a.nch - 1) * step + i * cp];
    double *to = lds + w * 64 * (M + 1) + lane;
    to[0] = gg;
#pragma unroll
    for (int i = 0; i < M; ++i) to[64 * (i + 1)] = m[i];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < REC_WPB; ++q) {
        const double *from = lds + q * 64 * (M + 1) + lane;
#pragma unroll
        for (int i = 0; i < M; ++i) s[i] = fma(from[0], s[i], from[64 * (i + 1)]);
    }
    const int r = q.sw - a.t0, jm = r < 0 ? -1 : r / a.chunk;
    const double gl = scan_pow(q.beta, a.chunk);
    const double gm = q.kap * scan_pow(q.beta, r < 0 ? 0 : a.chunk - 1 - r % a.chunk);
#pragma unroll
    for (int u = 0; u < REC_WPB - 1; ++u)
        if (u < w) {
            const double g = a.kb + u > jm ? gl : (a.kb + u == jm ? gm : 1.0);
#pragma unroll
            for (int i = 0; i < M; ++i) s[i] = fma(g, s[i], v[i][u]);
        }
    __syncthreads();
    if constexpr (NEXT) {
        // from the next wave; the last wave's is the first of the next block,
        // which the block folds as that one does
#pragma unroll
        for (int i = 0; i < M; ++i) lds[((w + REC_WPB - 1) % REC_WPB) * 64 * (M + 1) + lane + 64 * i] = s[i];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < M; ++i) next[i] = lds[w * 64 * (M + 1) + lane + 64 * i];
        __syncthreads();
        const int kb = a.kb + REC_WPB;
        if (kb >= a.nch) return;
        const int j0 = a.span ? kb / a.span * a.span : 0, all = kb - j0;
        if (a.span && j0 == kb) span_before(kb);
        double m[M], gg = 1.0;
#pragma unroll
        for (int i = 0; i < M; ++i) m[i] = 0.0;
        scan_chain<M>(a, q, a.chunk, b, step, cp, j0 + all * w / REC_WPB,
                      j0 + all * (w + 1) / REC_WPB, false, m, &gg);
        to[0] = gg;
#pragma unroll
        for (int i = 0; i < M; ++i) to[64 * (i + 1)] = m[i];
        __syncthreads();
        if (w == REC_WPB - 1) {
#pragma unroll
            for (int i = 0; i < M; ++i) next[i] = after[i];
#pragma unroll
            for (int v = 0; v < REC_WPB; ++v) {
                const double *from = lds + v * 64 * (M + 1) + lane;
#pragma unroll
                for (int i = 0; i < M; ++i) next[i] = fma(from[0], next[i], from[64 * (i + 1)]);
            }
        }
        __syncthreads();
    }
}

// Pass 1: the chunk's states from zero, for G groups [a.group, a.group + G) per
// wave: each term read then feeds G lanes' combos (the scalar cache hands out
// a line every ~16 cycles, more than one group's fma of it takes: 1,250 EMAs x
// 200k bars took 36 us at one group per wave, 27 at four).  ODD (ADX only):
// the true range is summed too (see scan_prepare).
template <class E, bool ODD, int G>
__device__ __forceinline__ void scan_states(const batch_view &a) {
    constexpr int N = __is_same(E, AdxEng) && !ODD ? 2 : scan_dims<E>::N;
    constexpr int S = scan_dims<E>::S;
    constexpr bool EMA = __is_same(E, EmaEng);
    const int lane = threadIdx.x & 63;
    const int c0 = a.t0 + a.k * a.chunk, c1 = c0 + a.chunk;
    double keep = 0.0;
    scan_touch<E>(a, c0, c1, keep);
    scan_lane q[G];
    double s[G][N];
    int smax = 0;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int c = (a.group + g) * 64 + lane;
        q[g] = scan_params<E>(a, c, c < a.nlanes);
        smax = max(smax, q[g].sw);
#pragma unroll
        for (int i = 0; i < N; ++i) s[g][i] = 0.0;
    }
    smax = wave_max(smax);
    int t = c0;
    const bool mixed = t <= smax;                    // a sum in this chunk
    // eight bars' terms at a time, the next eight on their way (a scalar load
    // per bar would be waited for per bar)
    double f[8][N];
    if (mixed) {
        scan_fetch<E, N, 8>(a, t, f);
        for (const int m = EMA ? c1 : min(c1, (smax + 8) & ~7); t < m; t += 8) {
            double n[8][N];
            scan_fetch<E, N, 8>(a, min(t + 8, c1 - 8), n);
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const bool past = t + u > q[g].sw;
                    const double b = past ? q[g].beta : 1.0;
#pragma unroll
                    for (int i = 0; i < N; ++i) {
                        s[g][i] = fma(b, s[g][i], EMA && past ? q[g].w * f[u][i] : f[u][i]);
                        if (EMA && t + u == q[g].sw) s[g][i] *= q[g].kap;
                    }
                }
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int i = 0; i < N; ++i) f[u][i] = n[u][i];
        }
    }
    auto steps = [&](const double (&from)[8][N]) {
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int i = 0; i < N; ++i) scan_step(s[g][i], q[g].beta, from[u][i]);
    };
    if (t < c1) scan_fetch<E, N, 8>(a, t, f);
    for (; t + 8 < c1; t += 8) {
        double n[8][N];
        scan_fetch<E, N, 8>(a, t + 8, n);
        steps(f);
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int i = 0; i < N; ++i) f[u][i] = n[u][i];
    }
    if (t < c1) steps(f);
#pragma unroll
    for (int g = 0; g < G; ++g) {
        if (a.group + g >= a.groups) continue;
        double *o = a.carry + (size_t)a.k * S * a.groups * 64 + (a.group + g) * 64 + lane;
#pragma unroll
        for (int i = 0; i < N; ++i)
            o[(size_t)i * a.groups * 64] = EMA && !mixed ? s[g][i] * q[g].w : s[g][i];
    }
}

// State i of one group's whole span q from zero: one wave per group, span and
// state (block.y).
template <class E>
__device__ __forceinline__ void scan_spans(const batch_view &a, int q, int i) {
    constexpr int S = scan_dims<E>::S;
    const int c = a.group * 64 + (threadIdx.x & 63);
    const size_t cp = (size_t)a.groups * 64, step = (size_t)S * cp;
    const scan_lane p = scan_params<E>(a, c, c < a.nlanes);
    const int sw = a.scan == 2 ? p.sw2 : p.sw;
    const scan_sum sum{p.beta, p.kap, sw, wave_max(sw)};
    double *b = a.carry + (size_t)i * cp + c;
    double s[1] = {0.0};
    scan_chain<1>(a, sum, a.chunk, b, step, cp, q * a.span, (q + 1) * a.span, true, s, nullptr);
    b[(size_t)(a.nch + q) * step] = s[0];
}

// RSI from the sums of 100 times the gain and of the absolute change, DX / 100 from the DM difference
// and sum, in f32 as rsi_ratio_f32 and dx_ratio form them (50 and 0 for a zero
// denominator).
__device__ __forceinline__ float scan_rsi(double gain, double all) {
    const float den = (float)all;
    if (!(den > 1e-30f && den < 1e30f))
        return all == 0.0 ? 50.0f : (float)(gain / all);
    float r = __builtin_amdgcn_rcpf(den);
    r = fmaf(fmaf(-den, r, 1.0f), r, r);
    return (float)gain * r;
}
__device__ __forceinline__ float scan_dx(double diff, double all) {
    return all != 0.0 ? (float)dx_ratio(fabs(diff), all) : 0.0f;
}

// A chunk from its exact start state: the outputs (EMIT), or ADX's second
// stage from zero for its scan.  Blocks of 32 bars past every sum run the
// plain updates, eight terms at a time; the others select per bar.
//
// RAG (rows that do not all start on a 128-byte line; kernels of their own,
// *_batch_lines_f32, or short calls would fetch the longer code): a wave keeps its
// last two tiles of 32 bars and stores whole lines only, those that start in its
// chunk; for the last of them it runs one tile into the next chunk, from that
// chunk's own start state, so that the rows' bits are those of tiles.  Stored
// tile by tile, each line of such rows is written in two parts some
// microseconds apart, more of them open at once than the L2 holds: 1,250 EMA x
// 180,001 bars 466 us, 255 with whole lines (180,000 bars: 221).  The next
// chunk's start takes 3% where a wave folds alone, 6% where the block does; its
// running state would do, but for the last bits.
template <class E, bool ODD, bool EMIT, bool RAG = false>
__device__ __forceinline__ void scan_output(const batch_view &a, float *out) {
    constexpr bool EMA = __is_same(E, EmaEng), RSI = __is_same(E, RsiEng),
                   ADX = __is_same(E, AdxEng);
    constexpr int N = ADX && !ODD ? 2 : scan_dims<E>::N;
    constexpr int S = scan_dims<E>::S;
    extern __shared__ __align__(16) double rec_lds[];
    float *ob = nullptr;                             // [64][REC_ROW], RAG [64][64]
    if (RAG) ob = reinterpret_cast<float *>(rec_lds) + block_wave() * 64 * 64;
    else if (EMIT) ob = reinterpret_cast<float *>(wave_lds<E>());
    const int lane = threadIdx.x & 63;
    const int c = a.group * 64 + lane;
    const size_t cp = (size_t)a.groups * 64;
    const int c0 = a.t0 + a.k * a.chunk, c1 = min(c0 + a.chunk, a.t1);
    double keep = 0.0;
    if (!wave_idle(a)) scan_touch<E>(a, c0, c1, keep);
    const scan_lane q = scan_params<E>(a, c, c < a.nlanes);
    double s[N], dxs = 0.0;                          // dxs: ADX's second stage
    double sn[N], dxn = 0.0;                         // the next chunk's (RAG)
    scan_start<N, RAG>(a, scan_sum{q.beta, q.kap, q.sw, wave_max(q.sw)}, S, 0, c, s, sn, rec_lds);
    const int last = wave_max(ADX ? max(q.sw2, q.first) : q.sw);
    if (ADX && EMIT)
        scan_start<1, RAG>(a, scan_sum{q.beta, 1.0, q.sw2, last}, S, S - 1, c, &dxs, &dxn, rec_lds);
    if (wave_idle(a) || (!EMIT && a.k + 1 >= a.nch)) return;
    const int nrow = min(64, a.nlanes - a.group * 64);
    float *row0 = out + (size_t)(a.group * 64 + (lane >> 3)) * a.T + 4 * (lane & 7);
    const float *src = ob + (lane >> 3) * REC_ROW + 4 * (lane & 7);
    const bool end = c1 == a.t1;
    // RAG: bars 4 j of row r sit at columns 4 j ^ 4 (r mod 16) of its two tiles
    // (a wave's float4 writes then fall on all banks)
    auto place = [&](int tb, int b) -> float4 * {
        return reinterpret_cast<float4 *>(
            RAG ? ob + lane * 64 + (((tb & 32) + b) ^ (4 * (lane & 15))) : ob + lane * REC_ROW + b);
    };
    // ... and stores, of each row, the line that bar tb lies in: the tile
    // before tb and the one at tb hold it
    auto lines = [&](int tb) {
        const int lim = min(end ? c1 : c1 + 32, a.t1);
        const uint32_t base = (uint32_t)(reinterpret_cast<uintptr_t>(out) >> 2);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int r = 8 * i + (lane >> 3);
            const uint32_t at = base + (uint32_t)(a.group * 64 + r) * (uint32_t)a.T + (uint32_t)tb;
            const int line = tb - (int)(at & 31);
            const int t = line + 4 * (lane & 7), x = 4 * (r & 15);
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = ob[r * 64 + (((t + u) & 63) ^ x)];
            // the line is this chunk's if it starts in it; a first chunk also
            // takes the part of the one before that lies in it
            const bool own = line >= c0 ? line < c1 : c0 == a.t0;
            if (r >= nrow || !own) continue;
            float *o = out + (size_t)(a.group * 64 + r) * a.T;
            if (line >= c0 && line + 32 <= lim) {
                *reinterpret_cast<vta_row4 *>(o + t) = vta_row4{v[0], v[1], v[2], v[3]};
            } else {
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (t + u >= c0 && t + u < lim) o[t + u] = v[u];
            }
        }
    };
    int tb = c0;
    for (; tb < (RAG && !end ? c1 + 32 : c1); tb += 32) {
        if (RAG && tb == c1) {
#pragma unroll
            for (int i = 0; i < N; ++i) s[i] = sn[i];
            dxs = dxn;
        }
        if (tb > last) {
#pragma unroll
            for (int b = 0; b < 32; b += 4) {
                double f[4][N];
                scan_fetch<E, N, 4>(a, tb + b, f);
                {
                    float y[4];
                    if constexpr (RSI || ADX) {
                        // four bars' denominators are checked together against
                        // the f32 reciprocal's range; outside it, the f64 forms
                        double u0[4], u1[4];         // denominators and numerators
                        bool some = true;            // no zero range sum (ODD)
                        float num[4], den[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
#pragma unroll
                            for (int i = 0; i < N; ++i) scan_step(s[i], q.beta, f[u][i]);
                            u0[u] = RSI ? s[1] : s[0];
                            u1[u] = RSI ? s[0] : s[1];
                            // a zero range sum makes DX zero
                            if (ODD) u0[u] = s[N - 1] != 0.0 ? u0[u] : 0.0;
                            if (ODD) some = some && s[N - 1] != 0.0;
                            num[u] = fabsf((float)u1[u]);
                            den[u] = (float)u0[u];
                        }
                        // (as integers: none is negative, and a NaN is above all)
                        uint32_t lo = 0xffffffffu, hi = 0u;
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const uint32_t d = __builtin_bit_cast(uint32_t, den[u]);
                            lo = min(lo, d);
                            hi = max(hi, d);
                        }
                        const bool fast = lo > __builtin_bit_cast(uint32_t, 1e-30f) &&
                                          hi < __builtin_bit_cast(uint32_t, 1e30f) && some;
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            float r = __builtin_amdgcn_rcpf(den[u]);
                            r = fmaf(fmaf(-den[u], r, 1.0f), r, r);
                            y[u] = num[u] * r;
                        }
                        if (!fast) {
#pragma unroll
                            for (int u = 0; u < 4; ++u)
                                y[u] = RSI ? scan_rsi(u1[u], u0[u]) : scan_dx(u1[u], u0[u]);
                        }
                        if constexpr (ADX) {
#pragma unroll
                            for (int u = 0; u < 4; ++u) {
                                dxs = fma(q.beta, dxs, (double)y[u]);
                                y[u] = (float)(dxs * q.scale);
                            }
                        }
                    } else {
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            if (EMA) s[0] = fma(q.beta, s[0], q.w * f[u][0]);
                            else scan_step(s[0], q.beta, f[u][0]);
                            y[u] = (float)(EMA ? s[0] : s[0] * q.scale);
                        }
                    }
                    if (EMIT)
                        *place(tb, b) = make_float4(y[0], y[1], y[2], y[3]);
                }
            }
        } else {
            // EMA's running mean divides by the bars so far, the same for
            // every combo: lane j forms the reciprocal for bar tb + j
            double inv = 0.0;
            if (EMA) inv = 1.0 / (double)(tb + (lane & 31) - a.fv + 1);
            double f[4][N];
            scan_fetch<E, N, 4>(a, tb, f);
            for (int b = 0; b < 32; b += 4) {
                double n[4][N];                      // the next four bars' terms
                scan_fetch<E, N, 4>(a, tb + min(b + 4, 28), n);
                float y[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int t = tb + b + u;
                    const bool past = t > q.sw;
                    const double g = past ? q.beta : 1.0;
#pragma unroll
                    for (int i = 0; i < N; ++i) {
                        s[i] = fma(g, s[i], EMA && past ? q.w * f[u][i] : f[u][i]);
                        if (EMA && t == q.sw) s[i] *= q.kap;
                    }
                    double v;
                    if constexpr (EMA) {
                        const double iv = __shfl(inv, b + u);   // every lane takes part
                        v = t < q.sw ? s[0] * iv : s[0];
                    } else if constexpr (RSI) {
                        v = (double)scan_rsi(s[0], s[1]);
                    } else if constexpr (ADX) {
                        const bool some = !ODD || s[N - 1] != 0.0;
                        const double dx = (double)scan_dx(s[1], some ? s[0] : 0.0);
                        dxs = fma(t > q.sw2 ? q.beta : 1.0, dxs, t >= q.sw ? dx : 0.0);
                        v = dxs * q.scale;
                    } else {
                        v = s[0] * (t == q.sw ? q.scale0 : q.scale);
                    }
                    y[u] = t >= q.first ? (float)v : VTA_QNAN_F32;
                }
                if (EMIT)
                    *place(tb, b) = make_float4(y[0], y[1], y[2], y[3]);
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int i = 0; i < N; ++i) f[u][i] = n[u][i];
            }
        }
        if (EMIT) {
            // eight rows x 128 bytes per store
            wave_lds_sync();
            if (RAG) {
                lines(tb);
            } else if (tb + 32 <= c1) {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (8 * i + (lane >> 3) < nrow)
                        *reinterpret_cast<vta_row4 *>(row0 + (size_t)(8 * i) * a.T + tb) =
                            *reinterpret_cast<const vta_row4 *>(src + 8 * i * REC_ROW);
            } else {
                for (int i = 0; i < 8; ++i)
                    for (int u = 0; u < 4; ++u)
                        if (8 * i + (lane >> 3) < nrow && tb + 4 * (lane & 7) + u < c1)
                            row0[(size_t)(8 * i) * a.T + tb + u] = src[8 * i * REC_ROW + u];
            }
            wave_lds_sync();
        }
    }
    if (RAG && end) lines(tb);
    if (EMIT) {
        if (a.state_out && a.k == a.nch - 1) {
#pragma unroll
            for (int i = 0; i < N; ++i) a.state_out[(size_t)i * cp + c] = s[i];
            if (ADX) a.state_out[(size_t)(S - 1) * cp + c] = dxs;
        }
    } else {
        a.carry[((size_t)a.k * S + S - 1) * cp + c] = dxs;
    }
}

// The passes of a block: scan_states (all chunks but the last), ADX's second
// stage, the output pass (an unclean series: one exact chunk in the first
// block of each group).
template <class E>
__device__ __forceinline__ void scan_pass1(batch_view a) {
    if (!a.clean) return;
    const bool odd = __is_same(E, AdxEng) && a.odd;
    if (a.coop) {
        if (a.k + 1 >= a.nch) return;
        if (odd) scan_states<E, true, 1>(a);
        else scan_states<E, false, 1>(a);
    } else {
        // four groups per wave: the first quarter of the blocks take all chunks
        // (a whole run of them, so that every XCD has its share) but those
        // with a sum in them, whose steps are long: the next blocks take
        // these, one group per wave
        const int w = a.group % REC_WPB, quarter = (a.nch + REC_WPB - 1) / REC_WPB;
        a.group -= w;
        int sw = 0;
        for (int g = 0; g < REC_WPB; ++g) {
            const int c = (a.group + g) * 64 + (int)(threadIdx.x & 63);
            sw = max(sw, scan_params<E>(a, c, c < a.nlanes).sw);
        }
        sw = wave_max(sw);
        int sums = sw < a.t0 ? 0 : (sw - a.t0) / a.chunk + 1;
        if (quarter + sums > a.nch) sums = 0;        // (too few blocks for that)
        if (a.k >= quarter) {
            a.k -= quarter;
            a.group += w;
            if (a.k >= sums || a.k + 1 >= a.nch || a.group >= a.groups) return;
            if (odd) scan_states<E, true, 1>(a);
            else scan_states<E, false, 1>(a);
            return;
        }
        a.k = REC_WPB * a.k + w;
        if (a.k < sums || a.k + 1 >= a.nch) return;
        if (odd) scan_states<E, true, REC_WPB>(a);
        else scan_states<E, false, REC_WPB>(a);
    }
}
__device__ __forceinline__ void scan_pass2(const batch_view &a) {
    if (!a.clean || a.nch < 2) return;               // (a one-chunk job has no carry)
    if (a.odd) scan_output<AdxEng, true, false>(a, nullptr);
    else scan_output<AdxEng, false, false>(a, nullptr);
}
template <class E, int NIN, bool RAG>
__device__ __forceinline__ void batch_pass(batch_view a, float *out) {
    if (a.scan == 0) {
        if (!wave_idle(a)) drive_batch<E, NIN>(a, out);
    } else if (!a.clean) {
        if (wave_idle(a) || a.k != 0 || a.t0 != 0) return;
        a.chunk = a.T;
        drive_batch<E, NIN>(a, out);
    } else if (__is_same(E, AdxEng) && a.odd) {
        scan_output<E, true, true, RAG>(a, out);
    } else {
        scan_output<E, false, true, RAG>(a, out);
    }
}
template <class E>
__device__ __forceinline__ void span_pass(batch_view &a, int flat) {
    if (!a.clean) return;
    const int per = (a.nch - 1) / a.span;            // spans read by later chunks
    const int i = a.scan == 2 ? scan_dims<E>::S - 1 : (int)blockIdx.y;
    if (__is_same(E, AdxEng) && i == 2 && !a.odd) return;
    a.group = flat / per;
    scan_spans<E>(a, flat % per, i);
}

// ---------------------------------------------------------------- packed batches
//
// Many one-series batches of one indicator in one launch per scan pass: job j
// is a series (its own length, first_valid and output) with its own period
// table.  A pass is a 1-D grid over every job's blocks (a combo group and
// REC_WPB chunks, or the other way round), job j owning those from block0 on;
// the span folds are a 1-D grid likewise, from span0 on.  A block finds its
// job by binary search over block0 (span0), then runs exactly
// the block of that job's direct launch, so a job's outputs are bit-identical
// alone and packed.  A job that its own call runs in segments has an entry for
// each, and the passes run for all first segments, then for all second ones.
struct rec_job {
    const float *x, *h, *l;
    const int32_t *periods;
    float *out;
    double *carry;           // this job's [chunk][state][64 x groups] and spans
    double *terms;           // this job's [term][tstride]
    int T, nlanes, fv, chunk, nch, groups, block0, span0, tstride, span;
};
// Beside the table's entry, in a pack with segments: the entry's bars and job
// (whose flags are its), the states as in rec_args.
struct rec_seg {
    const double *state_in;
    double *state_out;
    int t0, t1, job, pad_;
};

struct rec_pack_args {
    const rec_job *jobs;
    const rec_seg *segs;
    int32_t *flags;          // per job: SF_BAD and SF_ODD
    int32_t *call;           // SF_EPOCH and SF_LAST
    int n_jobs;
    int scan;
    int epoch;               // as in rec_args
    int last;
};

// The last job whose first block (span) is <= flat; jobs are in order.
__device__ __forceinline__ int pack_find(const rec_pack_args &p, int flat, bool spans) {
    int lo = 0, hi = p.n_jobs - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        const int first = spans ? p.jobs[mid].span0 : p.jobs[mid].block0;
        if (first <= flat) lo = mid; else hi = mid - 1;
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

// (SEG: a pack with segments.  In others entry j is all of job j: what segments
// need beyond that took 2 of the 71 us of 40 RSI series)
template <bool SEG, bool OUT>
__device__ __forceinline__ batch_view pack_view(const rec_pack_args &p, int j) {
    const rec_job &jb = p.jobs[j];
    batch_view v;
    v.x = jb.x; v.h = jb.h; v.l = jb.l;
    v.periods = jb.periods;
    v.alphas = nullptr;
    v.carry = jb.carry;
    v.terms = jb.terms;
    v.state_in = SEG ? p.segs[j].state_in : nullptr;
    v.state_out = SEG ? p.segs[j].state_out : nullptr;
    v.T = jb.T;
    v.nlanes = jb.nlanes;
    v.chunk = __builtin_amdgcn_readfirstlane(jb.chunk);
    v.nch = __builtin_amdgcn_readfirstlane(jb.nch);
    v.groups = __builtin_amdgcn_readfirstlane(jb.groups);
    v.span = __builtin_amdgcn_readfirstlane(jb.span);
    v.fv = jb.fv;
    v.t0 = SEG ? __builtin_amdgcn_readfirstlane(p.segs[j].t0) : 0;
    v.t1 = __builtin_amdgcn_readfirstlane(SEG ? p.segs[j].t1 : jb.T);
    v.tstride = jb.tstride;
    v.scan = v.nch > 1 || v.t0 > 0 ? p.scan : 0;     // one chunk: exact lanes
    const int f = SEG ? __builtin_amdgcn_readfirstlane(p.segs[j].job) : j;
    v.epoch = p.epoch ? p.epoch : OUT ? p.call[0] : p.call[1] + 1;
    v.clean = p.flags[2 * f] != v.epoch;
    v.odd = p.flags[2 * f + 1] == v.epoch;
    v.group = v.kb = v.k = 0;
    v.coop = false;
    return v;
}

template <bool SEG, bool OUT>
__device__ __forceinline__ batch_view pack_block(const rec_pack_args &p, float **out) {
    const int flat = blockIdx.x;
    const int j = pack_find(p, flat, false);
    batch_view v = pack_view<SEG, OUT>(p, j);
    block_chunk(v, flat - __builtin_amdgcn_readfirstlane(p.jobs[j].block0));
    *out = p.jobs[j].out;
    return v;
}

// (a job without spans owns no block here: the next job starts at its span0)
template <class E, bool SEG>
__device__ __forceinline__ void packed_spans(const rec_pack_args &p) {
    const int flat = blockIdx.x;
    const int j = pack_find(p, flat, true);
    batch_view v = pack_view<SEG, false>(p, j);
    span_pass<E>(v, flat - __builtin_amdgcn_readfirstlane(p.jobs[j].span0));
}

// The word that scan_flags asks of scan_states and of a call's last output pass
// (at their ends: a uniform load after a store goes through the vector cache).
__device__ __forceinline__ void leave_epoch(const batch_view &v, const int32_t *word) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *const_cast<int32_t *>(word) = v.epoch;
}

// Waves per SIMD of the direct output passes, what their LDS allows: scheduled
// for more they take longer (33 RSI x 10,007 bars 18.2 us, 17.8 so; 1,250 ADX x
// 200,000 457 and 452).  Packed, it is the other way round (27 ADX jobs 43.5 us,
// 44.2 so).
#define REC_WPE __attribute__((amdgpu_waves_per_eu(4, 4)))
#define REC_OUTPUT(KERNEL, ENG, NIN, RAG)                                                    \
    extern "C" __global__ __launch_bounds__(256) REC_WPE void KERNEL(rec_args a) {           \
        const batch_view v = view_of<true>(a);                                               \
        batch_pass<ENG, NIN, RAG>(v, a.out0);                                                \
        if (!a.epoch && a.last && a.clean) leave_epoch(v, a.clean + SF_LAST);                \
    }
#define REC_BATCH(NAME, ENG, NIN)                                                            \
    extern "C" __global__ __launch_bounds__(256) void NAME##_scan_states(rec_args a) {       \
        const batch_view v = view_of<false>(a);                                              \
        scan_pass1<ENG>(v);                                                                  \
        if (!a.epoch) leave_epoch(v, a.clean + SF_EPOCH);                                    \
    }                                                                                        \
    extern "C" __global__ __launch_bounds__(64) void NAME##_scan_spans(rec_args a) {         \
        batch_view v = view_of<false>(a);                                                    \
        span_pass<ENG>(v, blockIdx.x);                                                       \
    }                                                                                        \
    REC_OUTPUT(NAME##_batch_f32, ENG, NIN, false)                                            \
    REC_OUTPUT(NAME##_batch_lines_f32, ENG, NIN, true)
#define REC_PACKED_(NAME, ENG, NIN, SEG, X)                                                  \
    extern "C" __global__ __launch_bounds__(256) void NAME##_packed_states##X(               \
        rec_pack_args p) {                                                                   \
        float *out;                                                                          \
        const batch_view v = pack_block<SEG, false>(p, &out);                                \
        scan_pass1<ENG>(v);                                                                  \
        if (!p.epoch) leave_epoch(v, p.call);                                                \
    }                                                                                        \
    extern "C" __global__ __launch_bounds__(64) void NAME##_packed_spans##X(rec_pack_args p) {\
        packed_spans<ENG, SEG>(p);                                                           \
    }                                                                                        \
    extern "C" __global__ __launch_bounds__(256) void NAME##_packed_f32##X(rec_pack_args p) { \
        float *out;                                                                          \
        const batch_view v = pack_block<SEG, true>(p, &out);                                 \
        batch_pass<ENG, NIN, false>(v, out);                                                 \
        if (!p.epoch && p.last) leave_epoch(v, p.call + 1);                                  \
    }
#define REC_PACKED(NAME, ENG, NIN)                                                           \
    REC_PACKED_(NAME, ENG, NIN, false, )                                                     \
    REC_PACKED_(NAME, ENG, NIN, true, _seg)
REC_BATCH(ema, EmaEng, 1)
REC_BATCH(rsi, RsiEng, 1)
REC_BATCH(atr, AtrEng, 3)
REC_BATCH(adx, AdxEng, 3)
REC_BATCH(smma, SmmaEng, 1)
REC_BATCH(wilders, WildersEng, 1)
REC_BATCH(atr_tr, AtrTrEng, 1)
REC_PACKED(ema, EmaEng, 1)
REC_PACKED(rsi, RsiEng, 1)
REC_PACKED(atr, AtrEng, 3)
REC_PACKED(adx, AdxEng, 3)
REC_PACKED(smma, SmmaEng, 1)
REC_PACKED(wilders, WildersEng, 1)
extern "C" __global__ __launch_bounds__(256) void adx_scan_stage2(rec_args a) {
    scan_pass2(view_of<false>(a));
}
extern "C" __global__ __launch_bounds__(256) void adx_packed_stage2(rec_pack_args p) {
    float *out;
    scan_pass2(pack_block<false, false>(p, &out));
}
extern "C" __global__ __launch_bounds__(256) void adx_packed_stage2_seg(rec_pack_args p) {
    float *out;
    scan_pass2(pack_block<true, false>(p, &out));
}

// The per-bar terms of one series at bar t (kind: 0 the close, 1 RSI, 2 ATR,
// 3 ADX), zero outside (RSI, ADX: the first delta is at first_valid + 1)
// [first_valid, T), and whether its inputs are not finite, or odd: a
// directional move above the true range (a previous close outside its
// high..low).  Without an odd bar +DM and -DM never exceed the true range
// they are summed beside, so a zero range sum has a zero DM sum and the
// DX rule for it (adx.rs:370-390) needs no range sum; with one the range is
// summed too.
struct scan_bar { bool bad, odd; };
__device__ __forceinline__ scan_bar scan_bar_terms(const float *x, const float *h, const float *l,
                                                   int T, int fv, int kind, long t, double *f) {
    f[0] = f[1] = f[2] = 0.0;
    scan_bar r{false, false};
    if (t < fv || t >= T) return r;
    const double c = x[t], hi = h ? (double)h[t] : 0.0, lo = l ? (double)l[t] : 0.0;
    r.bad = !fin(c) || !fin(hi) || !fin(lo);
    if (kind == 0) {
        f[0] = c;
    } else if (t == fv) {
        if (kind == 2) f[0] = hi - lo;
    } else if (kind == 1) {
        const double d = c - (double)x[t - 1];
        f[0] = d > 0.0 ? 100.0 * d : 0.0;
        f[1] = fabs(d);
    } else if (kind == 2) {
        f[0] = true_range(hi, lo, (double)x[t - 1]);
    } else {
        double o[3];
        AdxEng::pre(hi, lo, c, (double)h[t - 1], (double)l[t - 1], (double)x[t - 1], o);
        f[0] = o[1] + o[2];      // (one of them is zero)
        f[1] = o[1] - o[2];
        f[2] = o[0];
        r.odd = o[1] > o[0] || o[2] > o[0];
    }
    return r;
}

// The one launch before a device-resident one-series batch: the terms of bars
// [t0, t1) (t1 up to a whole 64-bar block past the series; none when terms is
// NULL), the flags of a bar at or after first_valid that is not finite or is
// odd, and the call's epoch (scan_flags); and,
// with warms, vta_check_warms' check of the reference's warm indices against
// first_valid + period - 1 (a mismatch stores 1 in *err).  Grid: enough threads
// for the bars checked or formed from bar `from` on, and for n.
extern "C" __global__ __launch_bounds__(256) void scan_prepare(
    const float *__restrict__ x, const float *__restrict__ h, const float *__restrict__ l, int T,
    int first_valid, int kind, int nterms, int from, int t0, int t1, int tstride,
    double *__restrict__ terms, int call_epoch, int32_t *__restrict__ flags,
    const int32_t *__restrict__ periods, const int32_t *__restrict__ warms, int n,
    int32_t *__restrict__ err) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    const long t = (long)from + i;
    double f[3];
    const scan_bar r = scan_bar_terms(x, h, l, T, first_valid, kind, t, f);
    if (terms && t >= t0 && t < t1)
        for (int q = 0; q < nterms; ++q) terms[scan_term_at(nterms, q, tstride, t - t0)] = f[q];
    const bool alone = !call_epoch && !terms && i == 0;   // (no pass before the output's)
    if (r.bad || r.odd || alone) {
        const int32_t epoch = call_epoch ? call_epoch : flags[SF_LAST] + 1;
        if (r.bad) flags[SF_BAD] = epoch;
        if (r.odd) flags[SF_ODD] = epoch;
        if (alone) flags[SF_EPOCH] = epoch;
    }
    if (warms && i < n && (long long)warms[i] != (long long)first_valid + periods[i] - 1)
        err[0] = 1;
}

// The same for every job of a pack: grid (blocks, jobs).
extern "C" __global__ __launch_bounds__(256) void packed_prepare(
    const rec_job *jobs, int32_t *flags, int kind, int nterms, int call_epoch, int32_t *call) {
    const rec_job &jb = jobs[blockIdx.y];
    const int end = jb.nch > 1 ? jb.tstride : jb.T;  // a one-chunk job has no terms
    bool bad = false, odd = false;
    for (long t = (long)blockIdx.x * 256 + threadIdx.x; t < end; t += (long)gridDim.x * 256) {
        double f[3];
        const scan_bar r = scan_bar_terms(jb.x, jb.h, jb.l, jb.T, jb.fv, kind, t, f);
        if (jb.nch > 1)
            for (int q = 0; q < nterms; ++q)
                jb.terms[scan_term_at(nterms, q, jb.tstride, t)] = f[q];
        bad = bad || r.bad;
        odd = odd || r.odd;
    }
    if (bad || odd) {
        const int32_t epoch = call_epoch ? call_epoch : call[1] + 1;
        if (bad) flags[2 * blockIdx.y] = epoch;
        if (odd) flags[2 * blockIdx.y + 1] = epoch;
    }
}

// The same for the entries of a level of a pack with segments: grid (blocks,
// entries).
extern "C" __global__ __launch_bounds__(256) void packed_prepare_seg(
    const rec_job *jobs, const rec_seg *segs, int32_t *flags, int kind, int nterms, int call_epoch,
    int32_t *call) {
    const rec_job &jb = jobs[blockIdx.y];
    const int t0 = segs[blockIdx.y].t0, job = segs[blockIdx.y].job;
    const bool scan = jb.nch > 1 || t0 > 0;
    const int bars = scan ? jb.tstride : jb.T;
    bool bad = false, odd = false;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < bars; i += (long)gridDim.x * 256) {
        double f[3];
        const scan_bar r = scan_bar_terms(jb.x, jb.h, jb.l, jb.T, jb.fv, kind, t0 + i, f);
        if (scan)
            for (int q = 0; q < nterms; ++q)
                jb.terms[scan_term_at(nterms, q, jb.tstride, i)] = f[q];
        bad = bad || r.bad;
        odd = odd || r.odd;
    }
    if (bad || odd) {
        const int32_t epoch = call_epoch ? call_epoch : call[1] + 1;
        if (bad) flags[2 * job] = epoch;
        if (odd) flags[2 * job + 1] = epoch;
    }
}

// True range of one series (tr_from_hlc_f32 in the reference): 0 before
// first_valid, high - low at first_valid, then max(h - l, |h - c[t-1]|,
// |l - c[t-1]|), evaluated in f64 (exact for f32 inputs) and rounded once.
extern "C" __global__ __launch_bounds__(256) void tr_from_hlc_f32(
    const float *__restrict__ h, const float *__restrict__ l, const float *__restrict__ c, int T,
    int first_valid, float *__restrict__ tr) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= T) return;
    float v = 0.0f;
    if (t == first_valid) v = (float)((double)h[t] - (double)l[t]);
    else if (t > first_valid) v = (float)true_range(h[t], l[t], c[t - 1]);
    tr[t] = v;
}

// ---------------------------------------------------------------- preparation
//
// Per time-major series: first_valid and the clean flag (every input finite
// at every bar from first_valid on).  One lane per series walks its column;
// each row is one coalesced load across lanes.
//   mode 0: x only (EMA, RSI)
//   mode 1: first bar with high, low and x all non-NaN (ATR, atr.rs:197-207)
//   mode 2: max of the per-input first non-NaN bars (ADX, adx.rs:190-198)
//   mode 3: fv = first non-NaN x, fv2 = mode-1 bar, clean over all inputs
//           from fv on (fused EMA/RSI/ATR)
//   mode 4: fv = first non-NaN x; clean[s] receives the first bar at or after
//           fv whose x is not finite (T if none), for the windowed averages
extern "C" __global__ __launch_bounds__(64) void ms_prepare_meta(
    const float *__restrict__ x, const float *__restrict__ h, const float *__restrict__ l,
    int T, int N, int mode, int32_t *__restrict__ fvs, int32_t *__restrict__ fvs2,
    int32_t *__restrict__ clean) {
    const int s = blockIdx.x * 64 + (threadIdx.x & 63);
    if (s >= N) return;
    const bool hl = mode == 1 || mode == 2 || mode == 3;
    int fx = T, fh = T, fl = T, f3 = T;
    for (int t = 0; t < T; ++t) {
        const size_t off = (size_t)t * N + s;
        const bool nx = !isnan(x[off]);
        const bool nh = hl ? !isnan(h[off]) : true;
        const bool nl = hl ? !isnan(l[off]) : true;
        if (fx == T && nx) fx = t;
        if (fh == T && nh) fh = t;
        if (fl == T && nl) fl = t;
        if (f3 == T && nx && nh && nl) f3 = t;
        if (fx < T && f3 < T && fh < T && fl < T) break;
    }
    int f = mode == 0 ? fx : mode == 1 ? f3 : mode == 2 ? max(fx, max(fh, fl)) : fx;
    int zf = T;
    for (int t = f; t < T; ++t) {
        const size_t off = (size_t)t * N + s;
        const bool ok = vta_isfinite(x[off]) &&
                        (!hl || (vta_isfinite(h[off]) && vta_isfinite(l[off])));
        if (!ok) {
            zf = t;
            break;
        }
    }
    fvs[s] = f;
    if (fvs2) fvs2[s] = f3;
    clean[s] = mode == 4 ? zf : (zf == T ? 1 : 0);
}

// Per series s of a time-major [T][N] matrix, from the caller's first_valid
// (clamped into [0, T]): clean[s] = 1 when every bar from it on is finite
// (the recurrences' device forms), or, with want_index, the first non-finite
// bar (T if none; the finite-window averages' device forms).
__device__ __forceinline__ void ms_scan_from_fv(const float *__restrict__ x, int T, int N,
                                                const int32_t *__restrict__ fvs,
                                                int32_t *__restrict__ out, bool want_index) {
    const int s = blockIdx.x * 64 + (threadIdx.x & 63);
    if (s >= N) return;
    const int f = min(max((int)fvs[s], 0), T);
    int zf = T;
    for (int t = f; t < T; ++t) {
        if (!vta_isfinite(x[(size_t)t * N + s])) {
            zf = t;
            break;
        }
    }
    out[s] = want_index ? zf : (zf == T ? 1 : 0);
}
extern "C" __global__ __launch_bounds__(64) void ms_clean_from_first_valids(
    const float *__restrict__ x, int T, int N, const int32_t *__restrict__ fvs,
    int32_t *__restrict__ clean) {
    ms_scan_from_fv(x, T, N, fvs, clean, false);
}
extern "C" __global__ __launch_bounds__(64) void ms_first_nonfinite_from_first_valids(
    const float *__restrict__ x, int T, int N, const int32_t *__restrict__ fvs,
    int32_t *__restrict__ z) {
    ms_scan_from_fv(x, T, N, fvs, z, true);
}

// The reference's device forms of SMMA, SWMA and Wilders take per-combo warm
// indices that its host code sets to first_valid + period - 1; the kernels
// here derive the warm-up from the period, so the indices are checked: a
// mismatch stores 1 in *err (the context reports it at its next synchronize).
// first_valid < 0 derives first_valid from combo 0 (SWMA passes none) and
// stores it in *fv_out; a derived value outside [0, T - max_period] is an
// error too, and T (no output bar) is stored instead.
extern "C" __global__ __launch_bounds__(256) void vta_check_warms(
    const int32_t *__restrict__ periods, const int32_t *__restrict__ warms, int n, int T,
    int first_valid, int max_period, int32_t *__restrict__ fv_out, int32_t *__restrict__ err) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    long long fv = first_valid;
    bool bad = false;
    if (first_valid < 0) {
        fv = (long long)warms[0] - (long long)periods[0] + 1;
        const bool ok = fv >= 0 && fv <= (long long)T - (long long)max_period;
        if (c == 0 && fv_out) *fv_out = ok ? (int32_t)fv : T;
        bad = !ok;
    }
    if (c < n && (long long)warms[c] != fv + (long long)periods[c] - 1) bad = true;
    if (bad) err[0] = 1;
}

extern "C" __global__ __launch_bounds__(256) void vta_fill_i32(int32_t *__restrict__ p, int n,
                                                                int v) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = v;
}
