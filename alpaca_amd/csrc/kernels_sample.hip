// Token sampling on the device: Sampler.sample(logits:) (Sources/AlpacaCore/
// Runtime/Sampler.swift:57-93) for a draw u in [0, 1) supplied by the caller's
// RNG, so a step's logits never leave HBM.
//
// The reference: temperature 0 is the arg-max (lowest index on ties; NaN is an
// error).  Otherwise NaN is an error; top-k keeps the k largest logits (ties to
// the lower index); p_i = exp((l_i - top) / t) in double; top-p keeps the
// shortest prefix whose cumulative p/sum reaches top_p; the draw walks the kept
// probabilities in order until their running sum exceeds u * sum.  Candidates
// are in logit-descending, index-ascending order when top-k or top-p applies,
// in index order otherwise.
//
// What bounds a draw is a chain of short steps, not the 200 KB of logits, so
// the steps are few, the passes over all logits run on a workgroup per 1024 of
// them, and none walks an array on one thread longer than the reference's own
// order of sums requires.
//   * plain temperature (no top-k, top-p = 1): runs of 1024 logits are summed
//     by a workgroup each; their sums, in order, name the run that holds the
//     draw, and one workgroup walks it.  The sums are associated by run rather
//     than strictly left to right, so the token can differ from a strictly
//     sequential sum only when u * sum falls within about 1e-16 (relative) of
//     a boundary between two tokens.  A token whose probability is zero is never
//     drawn, at such a boundary either.
//   * top-k and/or top-p: one workgroup of 1024 threads takes candidates in the
//     reference's order in windows of up to 1024, each the next smallest (key,
//     index) pairs after the previous window.  The first window is gathered by
//     all CUs: the logits that reach a threshold which enough of the maxima of
//     64 reach.  Later ones (a flat distribution under top-p) lie between the
//     last value and a threshold found by counting: a step doubles or halves
//     the distance below the last value until enough logits qualify, on up to
//     48 logits a thread held in registers, one barrier a step (a radix
//     select's four passes of LDS histograms collide on the few exponents that
//     logits have).  Where no threshold separates at most 1024 (ties), a radix
//     select with the boundary's ties in index order takes the window.  The
//     window is sorted in registers, one element a thread.  One thread each
//     accumulates, in exactly the reference's order, the running sum of p (its
//     value at the last kept candidate is the kept total, and the draw is a
//     search in it) and the top-p cumulative of p/sum; the quotients are formed
//     in parallel.  Without top-k the total for top-p is the runs' sum over
//     all logits (same caveat as above).
// A draw of 49,152 normal logits (scale 3) through ahip_session_sample, host
// call to token, us: top-k 40 and top-p 0.95 159 -> 40, plain temperature 117 ->
// 34; through ahip_op_sample, which uploads them, top-p 0.9 327 -> 136, top-p
// 0.98 at temperature 1.3 (18,000 candidates) 6,940 -> 1,020.
#include "common.h"

#include <algorithm>

#include <limits.h>

namespace {

constexpr int kST = 1024;  // threads
constexpr int kWin = 1024;  // candidates per window
constexpr int kRun = 1024;  // logits per workgroup of sample_parts_kernel

struct SampleArgs {
    const float* logits;
    int n;
    float temperature;
    int top_k;
    float top_p;
    double u;
    int32_t* out;       // [1] token
    int* status;        // [1] 0 ok, 1 NaN in the logits
    uint32_t* cand_idx;  // [n] scratch: candidate indices in order
    double* cand_p;      // [n] scratch: running sums of their probabilities
    // scratch of sample_parts_kernel and sample_gather_kernel
    double* part;        // [runs][3]: per 1024 logits the max, the sum (all) and whether a NaN was seen
    float* sub;          // [64 runs / 4]: the max of each 64 logits
    uint64_t* list;      // [kWin]: the first window's composites, unsorted
    int* count;          // [1] their number; past kWin (or 0): no list
    int all;             // without top-k: every logit's probability counts
    int want;            // candidates the first window aims at
};

// Ascending in this key = logit descending; -0 and +0 share a key (they compare equal).
__device__ __forceinline__ uint32_t order_key(float l) {
    if (l == 0.0f) l = 0.0f;
    const uint32_t u = __float_as_uint(l);
    const uint32_t asc = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    return ~asc;
}
__device__ __forceinline__ float key_value(uint32_t key) {
    const uint32_t asc = ~key;
    return __uint_as_float((asc & 0x80000000u) ? (asc & 0x7FFFFFFFu) : ~asc);
}
__device__ __forceinline__ uint64_t composite(uint32_t key, uint32_t idx) { return ((uint64_t)key << 32) | idx; }

__device__ __forceinline__ double prob(float l, double top, double t) { return exp(((double)l - top) / t); }

__device__ __forceinline__ double readlane_d(double v, int l) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, l), hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), l);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// One pass over the logits, a run of 1024 per workgroup: its max and whether it
// holds a NaN, the max of each 64, and without top-k, where every logit counts,
// the sum of exp((l - max) / t).  One CU alone reads 200 KB from memory in 8 us,
// and the 64-bit exponentials are about 150 instructions a logit.
__global__ __launch_bounds__(256) void sample_parts_kernel(SampleArgs a) {
    __shared__ float s_f[4];
    __shared__ int s_nan[4];
    __shared__ double s_d[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i0 = blockIdx.x * kRun + threadIdx.x;
    if (blockIdx.x == 0 && threadIdx.x == 0) *a.count = 0;
    float l[4];
    bool nan_seen = false;
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < 4; j++) l[j] = a.logits[min(i0 + 256 * j, a.n - 1)];  // (a repeated last one leaves the max)
#pragma unroll
    for (int j = 0; j < 4; j++) {
        nan_seen |= l[j] != l[j];
        const float m = wave_max(l[j]);
        if (lane == 0) a.sub[blockIdx.x * (kRun / 64) + 4 * j + wave] = m;
        mx = fmaxf(mx, m);
    }
    const bool wave_nan = __builtin_amdgcn_ballot_w64(nan_seen) != 0;
    if (lane == 0) {
        s_f[wave] = mx;
        s_nan[wave] = wave_nan;
    }
    __syncthreads();
    mx = fmaxf(fmaxf(s_f[0], s_f[1]), fmaxf(s_f[2], s_f[3]));
    if (a.temperature == 0.0f && gridDim.x == 1) {  // the arg-max of one run needs no second launch
        __shared__ int s_at;
        if (threadIdx.x == 0) s_at = INT_MAX;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (i0 + 256 * j < a.n && l[j] == mx) atomicMin(&s_at, i0 + 256 * j);
        __syncthreads();
        if (threadIdx.x == 0) {
            const bool any = s_nan[0] | s_nan[1] | s_nan[2] | s_nan[3];
            *a.status = any ? 1 : 0;
            *a.out = any ? -1 : s_at;
        }
        return;
    }
    const double top = (double)mx, t = (double)a.temperature;
    double s = 0.0;
    if (a.all) {
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (i0 + 256 * j < a.n) s += prob(l[j], top, t);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    }
    if (lane == 0) s_d[wave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double* o = a.part + 3 * (int64_t)blockIdx.x;
        o[0] = top;
        o[1] = (s_d[0] + s_d[1]) + (s_d[2] + s_d[3]);
        o[2] = (s_nan[0] | s_nan[1] | s_nan[2] | s_nan[3]) ? 1.0 : 0.0;
    }
}

// The first window's candidates, a run of 1024 logits per workgroup: those at
// least as large as a threshold that `want` of the 64-logit maxima reach (each
// of those contributes one at least, and few contribute two), appended to the
// list in any order.  Every workgroup finds the threshold alike, by bisection
// over the maxima.  A list longer than kWin is not used.
__global__ __launch_bounds__(256) void sample_gather_kernel(SampleArgs a) {
    constexpr int kSub = 8;  // maxima a thread holds (131,072 logits); more are read again
    __shared__ int s_cnt[2][4];
    __shared__ float s_mm[2][4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i0 = blockIdx.x * kRun + threadIdx.x;
    const int subs = gridDim.x * (kRun / 64);
    float l[4], m[kSub];
#pragma unroll
    for (int j = 0; j < 4; j++) l[j] = a.logits[min(i0 + 256 * j, a.n - 1)];
    const float kNone = __uint_as_float(0x7FC00000u);
    float lo = INFINITY, hi = -INFINITY;
#pragma unroll
    for (int k = 0; k < kSub; k++) m[k] = a.sub[min((int)threadIdx.x + 256 * k, subs - 1)];
#pragma unroll
    for (int k = 0; k < kSub; k++) {
        if ((int)threadIdx.x + 256 * k >= subs) m[k] = kNone;
        lo = fminf(lo, m[k]);
        hi = fmaxf(hi, m[k]);
    }
    for (int k = threadIdx.x + 256 * kSub; k < subs; k += 256) {
        lo = fminf(lo, a.sub[k]);
        hi = fmaxf(hi, a.sub[k]);
    }
    lo = -wave_max(-lo);
    hi = wave_max(hi);
    if (lane == 0) {
        s_mm[0][wave] = lo;
        s_mm[1][wave] = hi;
    }
    __syncthreads();
    lo = fminf(fminf(s_mm[0][0], s_mm[0][1]), fminf(s_mm[0][2], s_mm[0][3]));
    hi = fmaxf(fmaxf(s_mm[1][0], s_mm[1][1]), fmaxf(s_mm[1][2], s_mm[1][3]));
    // lo: reached by every maximum; hi: by fewer than want
    for (int step = 0; step < 24; step++) {
        const float mid = 0.5f * lo + 0.5f * hi;
        if (!(mid > lo) || !(mid < hi)) break;  // (also where either is infinite)
        int c = 0;
#pragma unroll
        for (int k = 0; k < kSub; k++) c += __popcll(__builtin_amdgcn_ballot_w64(m[k] >= mid));
        for (int k0 = 256 * kSub; k0 < subs; k0 += 256) {
            const int k = k0 + threadIdx.x;
            c += __popcll(__builtin_amdgcn_ballot_w64(k < subs && a.sub[min(k, subs - 1)] >= mid));
        }
        if (lane == 0) s_cnt[step & 1][wave] = c;
        __syncthreads();
        c = (s_cnt[step & 1][0] + s_cnt[step & 1][1]) + (s_cnt[step & 1][2] + s_cnt[step & 1][3]);
        if (c >= a.want) lo = mid;
        else hi = mid;
        if (c >= a.want && c <= a.want + a.want / 8) break;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int i = i0 + 256 * j;
        const bool in = i < a.n && l[j] >= lo;
        const uint64_t mask = __builtin_amdgcn_ballot_w64(in);
        if (!mask) continue;
        int at = 0;
        if (lane == 0) at = atomicAdd(a.count, __popcll(mask));
        at = __builtin_amdgcn_readfirstlane(at) + __popcll(mask & ((1ull << lane) - 1));
        if (in && at < kWin) a.list[at] = composite(order_key(l[j]), (uint32_t)i);
    }
}

// A run's sum relative to the largest logit of all (a run of -inf adds nothing).
__device__ __forceinline__ double part_sum(const double* part, double top, double t) {
    return part[0] == -INFINITY ? 0.0 : part[1] * exp((part[0] - top) / t);
}

// The draw without top-k and top-p: the runs' sums in index order name the run
// that holds u * total, its logits (one a thread) the token.
__global__ __launch_bounds__(kRun) void sample_plain_kernel(SampleArgs a) {
    constexpr int NW = kRun / 64;
    __shared__ double s_sum[NW];
    __shared__ int s_token;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, runs = (a.n + kRun - 1) / kRun;
    const double t = (double)a.temperature;
    double top = -INFINITY;
    bool nan_seen = false;
    for (int r = lane; r < runs; r += 64) {  // (every wave alike)
        top = fmax(top, a.part[3 * r]);
        nan_seen |= a.part[3 * r + 2] != 0.0;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) top = fmax(top, __shfl_xor(top, o, 64));
    if (__builtin_amdgcn_ballot_w64(nan_seen)) {
        if (tid == 0) {
            *a.status = 1;
            *a.out = -1;
        }
        return;
    }
    // running sums of the runs, 64 at a time: this lane's run sum, then in order
    auto run_sum = [&](int r) { return r < runs ? part_sum(a.part + 3 * r, top, t) : 0.0; };
    double total = 0.0;
    for (int r0 = 0; r0 < runs; r0 += 64) {
        const double s = run_sum(r0 + lane);
        for (int c = 0; c < min(64, runs - r0); c++) total += readlane_d(s, c);
    }
    const double target = a.u * total;
    int token = a.n - 1;
    double acc = 0.0;
    bool done = false;  // (uniform over the workgroup: every wave computes the same sums)
    for (int r0 = 0; r0 < runs && !done; r0 += 64) {
        const double s = run_sum(r0 + lane);
        for (int c = 0; c < min(64, runs - r0) && !done; c++) {
            const double next = acc + readlane_d(s, c);
            if (target < next) {
                // this run's logits, one a thread: the waves' sums name the wave,
                // its running sums the lane; sums that rounding leaves short pass
                // on to the next token of a probability in the next wave or run
                const int i = (r0 + c) * kRun + tid;
                const double p = i < a.n ? prob(a.logits[i], top, t) : 0.0;
                double ws = p;
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) ws += __shfl_xor(ws, o, 64);
                __syncthreads();
                if (lane == 0) s_sum[wave] = ws;
                if (tid == 0) s_token = INT_MAX;
                __syncthreads();
                double before = acc;
                for (int w = 0; w < wave; w++) before += s_sum[w];
                if (s_sum[wave] > 0.0 && target < before + s_sum[wave]) {
                    double run = before;
                    for (int e = 0; e < 64; e++) {
                        const double pe = readlane_d(p, e);
                        run += pe;
                        if (target < run && pe > 0.0) {
                            const int at = (r0 + c) * kRun + wave * 64 + e;
                            if (lane == 0 && at < a.n) atomicMin(&s_token, at);
                            break;
                        }
                    }
                }
                __syncthreads();
                if (s_token != INT_MAX) {
                    token = s_token;
                    done = true;
                }
            }
            acc = next;
        }
    }
    // sums left short up to the end: the last token of a probability (none: the last)
    for (int r = total > 0.0 ? runs - 1 : -1; r >= 0 && !done; r--) {
        if (!(part_sum(a.part + 3 * r, top, t) > 0.0)) continue;  // (uniform)
        const int i = r * kRun + tid;
        __syncthreads();
        if (tid == 0) s_token = -1;
        __syncthreads();
        if (i < a.n && prob(a.logits[i], top, t) > 0.0) atomicMax(&s_token, i);
        __syncthreads();
        if (s_token >= 0) {
            token = s_token;
            done = true;
        }
    }
    if (tid == 0) {
        *a.status = 0;
        *a.out = token;
    }
}

}  // namespace

template <int NPT>
__global__ __launch_bounds__(kST) void sample_kernel(SampleArgs a) {
    constexpr int NW = kST / 64;
    __shared__ int s_int[8];
    __shared__ int s_cnt[2][NW];
    __shared__ uint32_t s_hist[256];
    __shared__ uint64_t s_win[kWin];   // window being gathered or sorted
    __shared__ double s_p[kWin];       // its probabilities
    __shared__ double s_q[kWin];       // their quotients by the total
    __shared__ double s_pre[kWin];     // running sums of the probabilities
    __shared__ uint32_t s_tie[kST];    // per-thread tie counts
    const int tid = threadIdx.x, lane = tid & 63, n = a.n;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const float* L = a.logits;

    // This wave's logits are [base, base + 64 R), lane by lane, the first NPT
    // rows of 64 in registers once a window needs them; past the end NaN, which
    // no comparison admits.
    const int R = (n + kST - 1) / kST, base = wave * R * 64;
    const float kNone = __uint_as_float(0x7FC00000u);
    float v[NPT];
    bool loaded = false;
    auto load = [&]() {
#pragma unroll
        for (int j = 0; j < NPT; j++) v[j] = L[min(base + j * 64 + lane, n - 1)];
#pragma unroll
        for (int j = 0; j < NPT; j++)
            if (j >= R || base + j * 64 + lane >= n) v[j] = kNone;
        loaded = true;
    };
    // f(logit, index) for this wave's logits [64 j0, 64 R) of its range, read
    // from memory (the L2), rows of 64 in step: what the registers do not hold,
    // and loops with bodies too large to unroll over them
    auto for_rows = [&](int j0, auto f) {
#pragma unroll 1
        for (; j0 < R; j0 += 8) {
            float w[8];
#pragma unroll
            for (int j = 0; j < 8; j++) w[j] = L[min(base + (j0 + j) * 64 + lane, n - 1)];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int i = base + (j0 + j) * 64 + lane;
                f(j0 + j < R && i < n ? w[j] : kNone, i);
            }
        }
    };

    // ---- NaN check and maximum, from the runs (every wave alike)
    const int runs = (n + kRun - 1) / kRun;
    float bm = -INFINITY;
    int first = INT_MAX;  // the first run that holds it
    bool nan_seen = false;
    for (int r = lane; r < runs; r += 64) {
        const float m = (float)a.part[3 * r];
        nan_seen |= a.part[3 * r + 2] != 0.0;
        if (m > bm || first == INT_MAX) {
            bm = m;
            first = r;
        }
    }
    wave_argmax(bm, first);
    if (__builtin_amdgcn_ballot_w64(nan_seen)) {
        if (tid == 0) {
            *a.status = 1;
            *a.out = -1;
        }
        return;
    }
    if (a.temperature == 0.0f) {  // Sampler.argmax: the lowest index of the largest
        if (tid == 0) s_int[0] = INT_MAX;
        __syncthreads();
        const int i = first * kRun + tid;
        if (i < n && L[i] == bm) atomicMin(&s_int[0], i);
        __syncthreads();
        if (tid == 0) {
            *a.status = 0;
            *a.out = s_int[0];
        }
        return;
    }
    const double top = (double)bm, t = (double)a.temperature;
    const int K = a.top_k > 0 ? min(a.top_k, n) : n;

    // ---- sorted candidates, produced window by window
    int produced = 0;      // candidates so far
    bool have_prev = false;
    uint64_t prev = 0;     // composite of the last candidate produced
    float width = 0.f;     // distance below the last value that the last window spanned
    int parity = 0;

    // How many logits past the candidates so far are at least thr (every thread
    // gets the count); thr is not above the last candidate's value.
    auto count_to = [&](float thr) {
        int c = 0;
#pragma unroll
        for (int j = 0; j < NPT; j++) c += __popcll(__builtin_amdgcn_ballot_w64(v[j] >= thr));
        for_rows(NPT, [&](float l, int) { c += __popcll(__builtin_amdgcn_ballot_w64(l >= thr)); });
        if (lane == 0) s_cnt[parity][wave] = c;
        __syncthreads();
        int sum = 0;
#pragma unroll
        for (int w = 0; w < NW; w++) sum += s_cnt[parity][w];
        parity ^= 1;  // the next count writes the other row, so one barrier a step is enough
        return sum - produced;
    };

    // The next candidates by threshold, at least min(want, left) of them where
    // that fits a window: their number, their composites unsorted in s_win; 0
    // where no threshold separates 1 to kWin of them.  A search in vain is 24
    // steps, so the ties with pv that are left are counted before it where the
    // last window was taken by radix select, which may have ended among more of
    // them than a window holds, and after six steps in vain.
    bool in_ties = false;  // the last window was taken by radix select
    auto threshold_window = [&](int want) -> int {
        if (!loaded) load();
        const int soft = min(kWin, max(64, 4 * want));  // a few more steps are cheaper than sorting many more
        const float pv = have_prev ? key_value((uint32_t)(prev >> 32)) : bm;
        if (!(pv < INFINITY)) return 0;  // (no distance below an infinity)
        const uint32_t pi = (uint32_t)prev;
        float lo = 0.f, hi = 0.f;  // distances known to admit too few, too many (0: none yet)
        float d = width > 0.f ? width : 0.5f;
        int best = 0;
        float best_thr = 0.f;
        for (int step = in_ties ? -1 : 0; step < 24; step++) {
            const bool ties = step == -1 || (step == 6 && !best);
            const float thr = ties ? pv : pv - d;
            const int c = count_to(thr);
            if (ties) {
                if (c > kWin) return 0;
                continue;
            }
            const bool fits = c >= 1 && c <= kWin;
            if (fits && (!best || (best < want ? c > best : c >= want && c < best))) {
                best = c;
                best_thr = thr;
                width = d;
            }
            if (fits && c >= want && c <= soft) break;
            if (c > soft) hi = d;
            else lo = d;
            if (thr == -INFINITY && c <= soft) break;  // every logit is in
            d = hi > 0.f ? 0.5f * (lo + hi) : 2.f * d;
            if (hi > 0.f && (d <= lo || d >= hi)) break;
        }
        if (!best) return 0;
        if (tid == 0) s_int[3] = 0;
        __syncthreads();
        for_rows(0, [&](float l, int i) {
            if (l >= best_thr && (!have_prev || l < pv || (l == pv && (uint32_t)i > pi))) {
                const int slot = atomicAdd(&s_int[3], 1);
                if (slot < kWin) s_win[slot] = composite(order_key(l), (uint32_t)i);
            }
        });
        __syncthreads();
        return best;
    };

    // The next m candidates (m <= kWin, m <= n - produced) by radix select over
    // the order key, the boundary's ties by index; composites unsorted in s_win.
    const int chunk = (n + kST - 1) / kST, c0 = min(n, tid * chunk), c1 = min(n, c0 + chunk);
    auto radix_window = [&](int m) {
        uint32_t prefix = 0, mask = 0;
        int need = m;
        for (int pass = 0; pass < 4; pass++) {
            const int shift = 24 - 8 * pass;
            for (int b = tid; b < 256; b += kST) s_hist[b] = 0;
            __syncthreads();
            for (int i = tid; i < n; i += kST) {
                const uint32_t key = order_key(L[i]);
                if (have_prev && composite(key, (uint32_t)i) <= prev) continue;
                if ((key & mask) != prefix) continue;
                atomicAdd(&s_hist[(key >> shift) & 255u], 1u);
            }
            __syncthreads();
            if (tid == 0) {
                int cum = 0, b = 0;
                for (; b < 255; b++) {
                    if (cum + (int)s_hist[b] >= need) break;
                    cum += (int)s_hist[b];
                }
                s_int[0] = b;
                s_int[1] = need - cum;
            }
            __syncthreads();
            prefix |= (uint32_t)s_int[0] << shift;
            mask |= 255u << shift;
            need = s_int[1];
            __syncthreads();
        }
        // `prefix` is the boundary key; take its `need` lowest-index members (after prev)
        const uint32_t bkey = prefix;
        uint32_t ties = 0;
        for (int i = c0; i < c1; i++) {
            const uint32_t key = order_key(L[i]);
            if (key == bkey && !(have_prev && composite(key, (uint32_t)i) <= prev)) ties++;
        }
        s_tie[tid] = ties;
        __syncthreads();
        if (tid == 0) {
            int cum = 0, k = 0;
            for (; k < kST; k++) {
                if (cum + (int)s_tie[k] >= need) break;
                cum += (int)s_tie[k];
            }
            // walk chunk k for the (need - cum)-th tied index
            int left = need - cum, bidx = -1;
            const int b0 = min(n, k * chunk), b1 = min(n, b0 + chunk);
            for (int i = b0; i < b1 && left > 0; i++) {
                const uint32_t key = order_key(L[i]);
                if (key == bkey && !(have_prev && composite(key, (uint32_t)i) <= prev) && --left == 0) bidx = i;
            }
            s_int[2] = bidx;
            s_int[3] = 0;  // gather counter
        }
        __syncthreads();
        const uint64_t bound = composite(bkey, (uint32_t)s_int[2]);
        for (int i = tid; i < n; i += kST) {
            const uint64_t c = composite(order_key(L[i]), (uint32_t)i);
            if ((have_prev && c <= prev) || c > bound) continue;
            const int slot = atomicAdd(&s_int[3], 1);
            if (slot < kWin) s_win[slot] = c;  // exactly m <= kWin pass: the passes count the same elements
        }
        __syncthreads();
    };

    // Appends the next candidates (at least one, `want` where a threshold
    // allows it) and returns their number: indices at cand_idx[produced...],
    // probabilities in s_p (zeros up to kWin).
    auto next_window = [&](int want) -> int {
        int c = 0;
        if (!have_prev && *a.count <= kWin) {  // the first window, gathered already
            c = min(*a.count, kWin);
            if (tid < c) s_win[tid] = a.list[tid];
            __syncthreads();
        }
        if (!c) c = threshold_window(min(min(want, kWin / 2), n - produced));
        in_ties = !c;
        if (!c) {
            c = min(kWin, n - produced);
            radix_window(c);
        }
        // bitonic sort, one composite a thread: strides below 64 inside the
        // wave, the others through LDS
        int size_max = 64;
        while (size_max < c) size_max <<= 1;
        uint64_t x = tid < c ? s_win[tid] : ~0ull;  // padding sorts last
        for (int size = 2; size <= size_max; size <<= 1)
            for (int stride = size >> 1; stride > 0; stride >>= 1) {
                uint64_t y;
                if (stride >= 64) {
                    __syncthreads();
                    s_win[tid] = x;
                    __syncthreads();
                    y = s_win[tid ^ stride];
                } else {
                    y = ((uint64_t)(uint32_t)__shfl_xor((int)(x >> 32), stride, 64) << 32) |
                        (uint32_t)__shfl_xor((int)(uint32_t)x, stride, 64);
                }
                const bool keep_min = ((tid & size) == 0) == ((tid & stride) == 0);
                x = keep_min ? (y < x ? y : x) : (y > x ? y : x);
            }
        double p = 0.0;
        if (tid < c) {
            a.cand_idx[produced + tid] = (uint32_t)x;
            p = prob(key_value((uint32_t)(x >> 32)), top, t);
        }
        s_p[tid] = p;
        __syncthreads();  // (also: every read of s_win by the sort is done)
        if (tid == c - 1) s_win[0] = x;
        __syncthreads();
        prev = s_win[0];
        have_prev = true;
        return c;
    };

    // One thread: running sums of s_p[0..c) onto s, left in s_pre (s_p is padded
    // with zeros to a multiple of 8); the next eight are read under the adds.
    auto running_sums = [&](double s, int c) {
        double q[8], nx[8];
#pragma unroll
        for (int e = 0; e < 8; e++) nx[e] = s_p[e];
        for (int i = 0; i < c; i += 8) {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                q[e] = nx[e];
                nx[e] = s_p[min(i + 8, kWin - 8) + e];
            }
#pragma unroll
            for (int e = 0; e < 8; e++) {
                s += q[e];
                q[e] = s;
            }
#pragma unroll
            for (int e = 0; e < 8; e++) s_pre[i + e] = q[e];
        }
    };
    // One thread: cum plus the quotients s_q[0..c) in order until it reaches
    // top_p: the number taken, or 0 if it is not reached.
    double cum = 0.0;
    auto top_p_prefix = [&](int c) -> int {
        double q[8], nx[8];
#pragma unroll
        for (int e = 0; e < 8; e++) nx[e] = s_q[e];
        for (int i = 0; i < c; i += 8) {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                q[e] = nx[e];
                nx[e] = s_q[min(i + 8, kWin - 8) + e];
            }
#pragma unroll
            for (int e = 0; e < 8; e++) {
                cum += q[e];
                q[e] = cum;
            }
            if (!(cum >= (double)a.top_p)) continue;  // the sums do not descend
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (i + e < c && q[e] >= (double)a.top_p) return i + e + 1;
        }
        return 0;
    };

    // The running sums of the candidates' probabilities go to cand_p; their
    // value at the last candidate of the prefix is its total.  With top-k the
    // top-p walk needs the total of all K first; without, the total comes from
    // the runs' sums and each window is walked as it is produced.
    const bool all = K == n;
    double total = 0.0, run = 0.0;
    if (all) {
        for (int r0 = 0; r0 < runs; r0 += 64) {
            const int r = r0 + lane;
            const double s = r < runs ? part_sum(a.part + 3 * r, top, t) : 0.0;
            for (int c = 0; c < min(64, runs - r0); c++) total += readlane_d(s, c);
        }
    }
    int keep = K;
    bool found = false, one_window = false;  // one_window: every candidate's p is still in s_p
    while (produced < K && !found) {
        const int c = min(next_window(all ? kWin / 2 : K - produced), K - produced);
        one_window = c == K;
        if (all) {
            s_q[tid] = s_p[tid] / total;
            __syncthreads();
        }
        // the two sums in order, by one thread each (of two waves)
        if (tid == 0) running_sums(run, c);
        if (all && tid == 64) s_int[4] = top_p_prefix(c);
        __syncthreads();
        if (tid < c) a.cand_p[produced + tid] = s_pre[tid];
        run = s_pre[c - 1];
        if (all) {
            found = s_int[4] != 0;
            if (found) keep = produced + s_int[4];
        }
        produced += c;
        __syncthreads();
    }
    if (!all && a.top_p < 1.0f) {
        total = run;
        for (int b = 0; b < K && !found; b += kWin) {
            const int c = min(kWin, K - b);
            double p = 0.0;
            if (tid < c) p = one_window ? s_p[tid] : prob(L[a.cand_idx[b + tid]], top, t);
            s_q[tid] = p / total;
            __syncthreads();
            if (tid == 64) s_int[4] = top_p_prefix(c);
            __syncthreads();
            found = s_int[4] != 0;
            if (found) keep = b + s_int[4];
            __syncthreads();
        }
    }

    // the draw: the first candidate whose running sum exceeds u * kept, else the last kept
    __syncthreads();
    if (tid == 0) s_int[5] = keep - 1;
    __syncthreads();
    const double target = a.u * a.cand_p[keep - 1];
    for (int b = 0; b < keep; b += kST) {
        const int i = b + tid;
        if (i < keep && target < a.cand_p[i]) {
            atomicMin(&s_int[5], i);
            break;
        }
    }
    __syncthreads();
    if (tid == 0) {
        *a.status = 0;
        *a.out = (int)a.cand_idx[s_int[5]];
    }
}

// cand_p [n], part [runs][3], list [kWin], sub [16 runs], count
size_t sample_scratch_bytes(int n) {
    const size_t runs = ((size_t)n + kRun - 1) / kRun;
    return (size_t)n * 8 + runs * 24 + kWin * 8 + runs * (kRun / 64) * 4 + 8;
}

hipError_t launch_sample(const float* logits, int n, float temperature, int top_k, float top_p, double u,
                         int32_t* out, int* status, uint32_t* cand_idx, double* cand_p, hipStream_t st) {
    if (n <= 0) return hipErrorInvalidValue;
    const int runs = (int)(((int64_t)n + kRun - 1) / kRun), K = top_k > 0 && top_k < n ? top_k : n;
    SampleArgs a{logits, n, temperature, top_k, top_p, u, out, status, cand_idx, cand_p};
    a.part = cand_p + n;
    a.list = (uint64_t*)(a.part + 3 * (size_t)runs);
    a.sub = (float*)(a.list + kWin);
    a.count = (int*)(a.sub + (size_t)runs * (kRun / 64));
    a.all = temperature != 0.0f && K == n;
    // the first window: all of a top-k that fits one, else enough for most nuclei
    // (the others go on window by window in sample_kernel)
    a.want = std::min(K, a.all ? kWin / 4 : kWin / 2);
    sample_parts_kernel<<<runs, 256, 0, st>>>(a);
    if (temperature == 0.0f && runs == 1) return hipGetLastError();
    if (a.all && !(top_p < 1.0f)) {
        sample_plain_kernel<<<1, kRun, 0, st>>>(a);
        return hipGetLastError();
    }
    if (temperature != 0.0f) sample_gather_kernel<<<runs, 256, 0, st>>>(a);
    // registers for up to 16 or 48 logits a thread (16,384 or 49,152 in all; 64
    // a thread would spill); 16 where the gathered list holds all of a top-k
    if (n <= 16 * kST || K <= a.want) sample_kernel<16><<<1, kST, 0, st>>>(a);
    else sample_kernel<48><<<1, kST, 0, st>>>(a);
    return hipGetLastError();
}
