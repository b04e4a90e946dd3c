// Timestral forecaster pieces that sit between the matrix-core launches (gfx950): the context
// preparation of forecastRaw, the causal per-patch statistics and patch features of predictBlock,
// the RoPE tables, the gates, the monotone quantile head, refineBlock's frames, the median
// feedback of blockDecode, and the final cap / symmetric average / clip.
//
// Reference: src/timestral/model.zig (predictBlock :220-432, runTransformer :434-482, StatsJob
// :712-750) and src/timestral/forecaster.zig (forecast :57-180, forecastRaw :303-421, blockDecode
// :423-563, refineBlock :582-662), for series of target variates with optional numeric past-only
// and known-future covariate rows (the window, the known rows' statistics and the role feedback).
//
// The sequential recurrences of the reference (the float64 Welford of every row, the fold of
// refineBlock) run one workgroup per row: what hangs on no earlier step (the loads, the divisions,
// the deviations) is spread over the threads, and only the chains of additions are walked by one
// lane, in the reference's order, so they give the reference's values; a row's state is kept
// between decode blocks and continued over the appended steps, which is the same sequence of
// operations as recomputing the grown row from its start.
#include "common.hpp"
#include "launch.hpp"

// Products and sums are rounded one at a time, as in the reference's scalar and vector code.
#pragma clang fp contract(off)

namespace tsfm {
namespace {

__device__ __forceinline__ double fmax_d(double a, double b) { return fmax(a, b); }

// forecastRaw's rows (src/timestral/forecaster.zig:321-379). Row r = g * vall + i of group g (g <
// batch: forward pass, else the mirrored pass of series g - batch, every value negated,
// forecast.zig:112-121); i < V targets (forward-filled, leading gaps 0), then n_past past-only
// and n_known known-future covariates (NaN = missing). Keep the last `keep` steps, left-pad to t;
// known rows also write their horizon values to kf/kfm (rows, hpad). Also the clip flag of each
// target input row (finish, :163-178).
// One workgroup per row: the forward fill of a step is the value of the last observed lane at or
// before it (a ballot and a shuffle), else that of an earlier wave or an earlier pass over the row. One
// thread per row walked every step behind its load (24 rows x 1500 steps: 557 us; now under 7 us).
constexpr int kCtxT = 512;
__global__ __launch_bounds__(kCtxT) void ts_context(const TsContextParams p) {
    const int r = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = r / p.vall, i = r % p.vall;
    const bool mirror = g >= p.batch;
    const int sidx = mirror ? g - p.batch : g;
    const float sign = mirror ? -1.f : 1.f;
    const int t0 = p.t0, keep = p.keep, t = p.t;
    float* c = p.ctx + (int64_t)r * p.cap_t;
    uint8_t* mk = p.mask + (int64_t)r * p.cap_t;
    for (int j = tid; j < t - keep; j += kCtxT) {
        c[j] = 0.f;
        mk[j] = 0;
    }
    if (i >= p.V) {
        const bool known = i >= p.V + p.n_past;
        const float* x = known ? p.known + ((int64_t)sidx * p.n_known + (i - p.V - p.n_past)) * (t0 + p.horizon)
                               : p.past + ((int64_t)sidx * p.n_past + (i - p.V)) * t0;
        for (int j = t0 - keep + tid; j < t0; j += kCtxT) {
            const float v = sign * x[j];
            const bool ob = !isnan(v);
            const int dst = (t - keep) + (j - (t0 - keep));
            c[dst] = ob ? v : 0.f;
            mk[dst] = ob ? 1 : 0;
        }
        if (known)
            for (int j = tid; j < p.hpad; j += kCtxT) {
                const float v = j < p.horizon ? sign * x[t0 + j] : 0.f;
                const bool ob = j < p.horizon && !isnan(v);
                p.kf[(int64_t)r * p.hpad + j] = ob ? v : 0.f;
                p.kfm[(int64_t)r * p.hpad + j] = ob ? 1 : 0;
            }
        return;
    }
    constexpr int NW = kCtxT / 64;
    __shared__ float wave_last[2][NW];  // by the pass's parity: the last observed value of each wave,
    __shared__ int wave_seen[2][NW];    // and whether it has one
    __shared__ int any_s, neg_s;
    const int src = sidx * p.V + i;
    const float* x = p.inputs + (int64_t)src * t0;
    const uint8_t* o = p.observed + (int64_t)src * t0;
    if (tid == 0) any_s = neg_s = 0;
    float last = 0.f;  // the last observed value before the pass (uniform over the workgroup)
    bool seen = false, any = false, neg = false;
    int par = 0;
    for (int j0 = 0; j0 < t0; j0 += kCtxT, par ^= 1) {
        const int j = j0 + tid;
        const float xj = j < t0 ? x[j] : 0.f, v = sign * xj;
        const bool ob = j < t0 && o[j] != 0;
        if (ob && isfinite(xj)) {
            any = true;
            neg = neg || !(xj >= 0.f);
        }
        const unsigned long long all = __ballot(ob), upto = all & (~0ull >> (63 - lane));
        const float fill = __shfl(v, upto ? 63 - __clzll(upto) : lane);
        if (lane == (all ? 63 - __clzll(all) : 0)) {
            wave_last[par][wave] = v;
            wave_seen[par][wave] = all != 0;
        }
        __syncthreads();  // (the other parity's arrays are free for the next pass)
        float before = last;
        bool sb = seen;
        for (int w = 0; w < NW; w++) {
            if (!wave_seen[par][w]) continue;
            if (w < wave) {
                before = wave_last[par][w];
                sb = true;
            }
            last = wave_last[par][w];
            seen = true;
        }
        if (j < t0 && j >= t0 - keep) {
            const int dst = (t - keep) + (j - (t0 - keep));
            c[dst] = upto ? fill : sb ? before : 0.f;
            mk[dst] = ob ? 1 : 0;
        }
    }
    if (mirror) return;
    __syncthreads();
    if (any) any_s = 1;
    if (neg) neg_s = 1;
    __syncthreads();
    if (tid == 0) p.nonneg[src] = any_s != 0 && neg_s == 0;
}

// predictBlock's window with covariates (model.zig:253-273): steps [t, t + blen) of every row are
// the block's known futures (known rows, from step `done` of kf) or blanks (targets and past-only
// rows; the targets' blanks become medians after the block).
__global__ void ts_window(float* ctx, uint8_t* mask, int cap_t, int t, int blen, const float* kf,
                          const uint8_t* kfm, int hpad, int done, int vall, int known_from, int rows) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)rows * blen) return;
    const int r = (int)(idx / blen), j = (int)(idx % blen);
    const bool known = r % vall >= known_from;
    ctx[(int64_t)r * cap_t + t + j] = known ? kf[(int64_t)r * hpad + done + j] : 0.f;
    mask[(int64_t)r * cap_t + t + j] = known ? kfm[(int64_t)r * hpad + done + j] : 0;
}

// Known-future rows' statistics (model.zig:283-310): float32 mean and population std of the
// observed steps of the whole window [0, w), at least min_scale; a row of only 0/1 values is
// neither shifted nor scaled and skips the asinh. Written over every patch of the row's loc and
// scale; other rows keep their causal statistics. One thread per row, the reference's order.
__global__ void ts_known_stats(const float* ctx, const uint8_t* mask, int cap_t, int w, int ps, int rows, int vall,
                               int known_from, float min_scale, float* loc, float* scale, int cap_p,
                               uint8_t* no_asinh) {
#pragma clang fp contract(off)
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    if (r % vall < known_from) {
        no_asinh[r] = 0;
        return;
    }
    const float* x = ctx + (int64_t)r * cap_t;
    const uint8_t* o = mask + (int64_t)r * cap_t;
    float cnt = 0.f, sum = 0.f;
    bool zero_one = true, any = false;
    for (int i = 0; i < w; i++)
        if (o[i]) {
            cnt += 1.f;
            sum += x[i];
            zero_one = zero_one && (x[i] == 0.f || x[i] == 1.f);
            any = true;
        }
    float kloc = sum / fmaxf(cnt, 1.f);
    float ss = 0.f;
    for (int i = 0; i < w; i++)
        if (o[i]) {
            const float dv = x[i] - kloc;
            ss += dv * dv;
        }
    float kscale = fmaxf(sqrtf(ss / fmaxf(cnt, 1.f)), min_scale);
    const bool binary = zero_one && any;
    if (binary) {
        kloc = 0.f;
        kscale = 1.f;
    }
    for (int pt = 0; pt < w / ps; pt++) {
        loc[(int64_t)r * cap_p + pt] = kloc;
        scale[(int64_t)r * cap_p + pt] = kscale;
    }
    no_asinh[r] = binary ? 1 : 0;
}

}  // namespace

hipError_t launch_ts_context(const TsContextParams& p, hipStream_t s) {
    if (p.rows <= 0) return hipSuccess;
    hipLaunchKernelGGL(ts_context, dim3((unsigned)p.rows), dim3(kCtxT), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_ts_window(float* ctx, uint8_t* mask, int cap_t, int t, int blen, const float* kf, const uint8_t* kfm,
                            int hpad, int done, int vall, int known_from, int rows, hipStream_t s) {
    const int64_t n = (int64_t)rows * blen;
    hipLaunchKernelGGL(ts_window, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, ctx, mask, cap_t, t, blen, kf,
                       kfm, hpad, done, vall, known_from, rows);
    return hipGetLastError();
}

hipError_t launch_ts_known_stats(const float* ctx, const uint8_t* mask, int cap_t, int w, int ps, int rows, int vall,
                                 int known_from, float min_scale, float* loc, float* scale, int cap_p,
                                 uint8_t* no_asinh, hipStream_t s) {
    hipLaunchKernelGGL(ts_known_stats, dim3((unsigned)((rows + 63) / 64)), dim3(64), 0, s, ctx, mask, cap_t, w, ps,
                       rows, vall, known_from, min_scale, loc, scale, cap_p, no_asinh);
    return hipGetLastError();
}

namespace {

// StatsJob (src/timestral/model.zig:712-750) continued from step `from` (a patch boundary) to t,
// from the row's saved state (st: cum_w, cum_x, m2, prev_mean; zero when from == 0): loc and
// scale of patches [from / ps, t / ps). In the same pass: key validity of those patches
// (model.zig:343-357: observed, or with attend_missing any patch after the row's first observed
// one), the row's first observed patch (-1 if none yet), and refineBlock's fold of the context's
// per-patch moments (forecaster.zig:613-631) into fold (w, mean, m2).
// One workgroup per row, in tiles of whole patches held in LDS. The chains of rounded operations
// (cum_x, m2, the fold's mean and m2) keep the reference's order, one lane each; the loads, the
// divisions and every term that hangs on no other step are spread over the threads. One thread per
// row did all of it behind each step's load and divisions (24 rows x 1504 steps: 337 us; now
// 36 us, bound by the two chains of 1504 additions).
constexpr int kStatsT = 256, kStatsTile = 1024;

// c += s[i], i < n (n rounded up to 8: the padding is zeros), each partial sum to out[i].
__device__ __forceinline__ double chain_sum(const double* s, double* out, int n, double c) {
    for (int i0 = 0; i0 < n; i0 += 8) {
        double v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = s[i0 + k];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            c += v[k];
            out[i0 + k] = c;
        }
    }
    return c;
}

__global__ __launch_bounds__(kStatsT) void ts_stats(const TsStatsParams p) {
    __shared__ double sx[kStatsTile];                  // w x of each step, then its term of m2, then m2 after it
    __shared__ double cx[kStatsTile], cw[kStatsTile];  // cum_x, cum_w after each step
    // Per patch: observed steps, their mean (then the fold's delta), their m2, 1 / the fold's count.
    __shared__ double pm_cnt[kStatsTile], pm_mean[kStatsTile], pm_m2[kStatsTile], pm_inv[kStatsTile];
    __shared__ double st_s[4], fo_s[3];  // the row's state after the tile
    __shared__ int first_s;              // first observed patch so far
    const int r = blockIdx.x, tid = threadIdx.x;
    const float* x = p.ctx + (int64_t)r * p.cap_t;
    const uint8_t* o = p.mask + (int64_t)r * p.cap_t;
    double* st = p.state + (int64_t)r * 4;
    double* fo = p.fold + (int64_t)r * 3;
    const int ps = p.ps, pt_end = p.t / ps, per = kStatsTile / ps;  // whole patches per tile
    if (tid < 4) st_s[tid] = p.from > 0 ? st[tid] : 0.0;
    else if (tid < 7) fo_s[tid - 4] = p.from > 0 ? fo[tid - 4] : 0.0;
    else if (tid == 7) first_s = p.from > 0 && p.row_first[r] >= 0 ? p.row_first[r] : 0x7fffffff;
    __syncthreads();
    for (int pt0 = p.from / ps; pt0 < pt_end; pt0 += per) {
        const int np = min(per, pt_end - pt0), n = np * ps;
        double xv[kStatsTile / kStatsT];
#pragma unroll
        for (int k = 0; k < kStatsTile / kStatsT; k++) {
            const int i = tid + kStatsT * k;
            const double w = i < n && o[pt0 * ps + i] != 0 ? 1.0 : 0.0;
            xv[k] = i < n ? (double)x[pt0 * ps + i] : 0.0;
            sx[i] = w * xv[k];
            cw[i] = w;
        }
        const double cum_w0 = st_s[0], mean_in = st_s[3], fold_w0 = fo_s[0];
        __syncthreads();
        if (tid == 0) {
            st_s[1] = chain_sum(sx, cx, n, st_s[1]);
        } else if (tid >= 64) {
            // The patch's own moments (forecaster.zig:613-631), each over its observed steps in order.
            for (int q = tid - 64; q < np; q += kStatsT - 64) {
                double cnt = 0, sum = 0, mean = 0, m2 = 0;
                for (int k = 0; k < ps; k++)
                    if (cw[q * ps + k] != 0) {
                        cnt += 1;
                        sum += sx[q * ps + k];
                    }
                if (cnt > 0) {
                    mean = sum / fmax_d(cnt, 1.0);
                    for (int k = 0; k < ps; k++)
                        if (cw[q * ps + k] != 0) {
                            const double dv = sx[q * ps + k] - mean;
                            m2 += dv * dv;
                        }
                    atomicMin(&first_s, pt0 + q);
                }
                pm_cnt[q] = cnt;
                pm_mean[q] = mean;
                pm_m2[q] = m2;
            }
        }
        __syncthreads();
        if (tid < 64) {  // counts: whole numbers, the same in any order
            double c = cum_w0;
            for (int i0 = 0; i0 < n; i0 += 64) {
                double v = i0 + tid < n ? cw[i0 + tid] : 0.0;
#pragma unroll
                for (int d = 1; d < 64; d <<= 1) {
                    const double u = __shfl_up(v, d);
                    if (tid >= d) v += u;
                }
                if (i0 + tid < n) cw[i0 + tid] = c + v;
                c += __shfl(v, 63);
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kStatsTile / kStatsT; k++) {
            const int i = tid + kStatsT * k;
            double term = 0.0;  // zeros past the tile: chain_sum's padding
            if (i < n) {
                const double before = i > 0 ? cw[i - 1] : cum_w0, w = cw[i] - before;
                const double mean = cx[i] / fmax_d(cw[i], 1.0);
                const double prev = i > 0 ? cx[i - 1] / fmax_d(before, 1.0) : mean_in;
                term = (xv[k] - prev) * (xv[k] - mean) * w;
                if ((i + 1) % ps == 0) {
                    p.loc[(int64_t)r * p.cap_p + pt0 + i / ps] = (float)mean;
                    pm_inv[i / ps] = 1.0 / fmax_d(fold_w0 + (cw[i] - cum_w0), 2.2250738585072014e-308);
                }
                if (i == n - 1) st_s[3] = mean;
            }
            sx[i] = term;
        }
        __syncthreads();
        if (tid == 0) {
            st_s[2] = chain_sum(sx, sx, n, st_s[2]);
            st_s[0] = cw[n - 1];
        } else if (tid == 64) {
            // welfordCombine (forecaster.zig:567-577), its mean: a division by the running count w per
            // patch. a / w from y = 1 / w (rounded): q = a y is off by 1.5 ulp at most, a - w q is then
            // exact, and q + (a - w q) y lies within 2^-51 ulp of a / w before it is rounded. It rounds as a / w
            // does because w is a whole number: a / w is at least 1 / (2 w) ulp away from the middle of two
            // doubles. Values past the range of the products divide.
            double fw = fold_w0, fmean = fo_s[1];
#pragma unroll 4
            for (int q = 0; q < np; q++) {
                const double cnt = pm_cnt[q], w = fmax_d(fw + cnt, 2.2250738585072014e-308), y = pm_inv[q];
                const double delta = pm_mean[q] - fmean, a = delta * cnt, q0 = a * y;
                const double quo = __builtin_fma(__builtin_fma(-w, q0, a), y, q0);
                fmean = fmean + (fabs(q0) > 1e-280 && fabs(q0) < 1e300 ? quo : a / w);
                fw = fw + cnt;
                pm_mean[q] = delta;
            }
            fo_s[1] = fmean;
        }
        __syncthreads();
        for (int q = tid; q < np; q += kStatsT) {
            const double cum_w = cw[q * ps + ps - 1], den = fmax_d(cum_w, 1.0), cnt = pm_cnt[q];
            const double variance = sx[q * ps + ps - 1] / fmax_d(den - 1.0, 1.0);
            p.scale[(int64_t)r * p.cap_p + pt0 + q] = (float)fmax_d(sqrt(variance), p.min_scale);
            p.key_valid[(int64_t)r * p.cap_p + pt0 + q] = (uint8_t)(p.attend_missing ? pt0 + q >= first_s : cnt > 0);
            // The fold's term of m2, delta^2 w_before cnt / w.
            const double w = fold_w0 + (cum_w - cum_w0), delta = pm_mean[q];
            pm_inv[q] = delta * delta * (w - cnt) * cnt / fmax_d(w, 2.2250738585072014e-308);
        }
        __syncthreads();
        if (tid == 0) {
            double fm2 = fo_s[2];
#pragma unroll 8
            for (int q = 0; q < np; q++) fm2 = fm2 + pm_m2[q] + pm_inv[q];
            fo_s[2] = fm2;
            fo_s[0] = fold_w0 + (cw[n - 1] - cum_w0);
        }
        __syncthreads();
    }
    if (tid < 4) st[tid] = st_s[tid];
    else if (tid < 7) fo[tid - 4] = fo_s[tid - 4];
    else if (tid == 7) p.row_first[r] = first_s == 0x7fffffff ? -1 : first_s;
}

// predictBlock's patch features (model.zig:281-328) of patches [p0, l): values normalised by their
// patch's statistics (asinh'd unless the row's no_asinh flag is set), then the missing-step mask.
__global__ void ts_features(const float* ctx, const uint8_t* mask, int cap_t, const float* loc, const float* scale,
                            int cap_p, int rows, int p0, int l, int ps, int use_asinh, const uint8_t* no_asinh,
                            float* feats) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int np = l - p0;
    if (idx >= (int64_t)rows * np * ps) return;
    const int i = (int)(idx % ps);
    const int64_t rp = idx / ps;
    const int r = (int)(rp / np), pt = p0 + (int)(rp % np);
    const float lo = loc[(int64_t)r * cap_p + pt];
    const float sc = fmaxf(scale[(int64_t)r * cap_p + pt], 1.1920929e-07f);  // @max(scale, floatEps(f32))
    const int64_t at = (int64_t)r * cap_t + pt * ps + i;
    const bool ob = mask[at] != 0;
    float v = 0.f;
    if (ob) {
        v = (ctx[at] - lo) / sc;
        if (use_asinh && !(no_asinh != nullptr && no_asinh[r])) v = asinhf(v);
    }
    float* f = feats + rp * 2 * ps;
    f[i] = v;
    f[ps + i] = ob ? 0.f : 1.f;
}

// First observed patch of each group (model.zig:343-360: over the group's rows, 0 when none) and
// the RoPE tables of runTransformer (:447-463) for token indices [0, n_tok): encoder token p at time
// p, decoder token ne + j at time l + j = its index minus shift (ne - l: 0 without covariates, so
// one table serves every block; the horizon's patches with covariates).
__global__ void ts_rope_tables(const int* row_first, int vall, int n_tok, int ne, int shift, TsRope rp, float* cos_t,
                               float* sin_t, int* first_obs) {
    const int g = blockIdx.y;
    int first = 0x7fffffff;
    for (int i = 0; i < vall; i++) {
        const int f = row_first[g * vall + i];
        if (f >= 0 && f < first) first = f;
    }
    if (first == 0x7fffffff) first = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) first_obs[g] = first;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)n_tok * 32) return;
    const int tok = (int)(idx / 32), i = (int)(idx % 32);
    const float pos = (float)((tok < ne ? tok : tok - shift) - first);
    const float ang = rp.inv_freq[i] * pos;
    const int64_t at = ((int64_t)g * n_tok + tok) * 32 + i;
    cos_t[at] = cosf(ang);
    sin_t[at] = sinf(ang);
}

// [encoder tokens; decoder tokens] of each row: x[r, i] = emb[r, i] for i < m, the forecast query
// for the h decoder tokens (model.zig:333-341).
__global__ void ts_assemble(const float* emb, const float* query, float* x, int rows, int m, int h, int d) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int sl = m + h, d4 = d / 4;
    if (idx >= (int64_t)rows * sl * d4) return;
    const int c = (int)(idx % d4) * 4;
    const int64_t rt = idx / d4;
    const int r = (int)(rt / sl), tok = (int)(rt % sl);
    const f32x4 v = tok < m ? ld4(emb + ((int64_t)r * m + tok) * d + c) : ld4(query + c);
    st4(x + rt * d + c, v);
}

// nn.mulSigmoid over whole vectors (src/core/nn.zig:423-433): o = o / (1 + exp(-g)).
__global__ void ts_mul_sigmoid(float* o, const float* g, int64_t n4) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n4) return;
    const f32x4 x = ld4(o + 4 * idx), gv = ld4(g + 4 * idx);
    st4(o + 4 * idx, f32x4{x[0] / (1.f + expf(-gv[0])), x[1] / (1.f + expf(-gv[1])), x[2] / (1.f + expf(-gv[2])),
                           x[3] / (1.f + expf(-gv[3]))});
}

// The bf16 time-attention output widened to the f32 buffer the out projection reads, with the
// sigmoid gate of timeAttention (model.zig:517, nn.mulSigmoid) applied as in ts_mul_sigmoid when g is
// given.
__global__ void ts_from_bf16(const uint16_t* oh, const float* g, float* o, int64_t n4) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n4) return;
    const u32x2 w = *reinterpret_cast<const u32x2*>(oh + 4 * idx);
    f32x4 x = {__uint_as_float(w[0] << 16), __uint_as_float(w[0] & 0xffff0000u), __uint_as_float(w[1] << 16),
               __uint_as_float(w[1] & 0xffff0000u)};
    if (g != nullptr) {
        const f32x4 gv = ld4(g + 4 * idx);
        x = f32x4{x[0] / (1.f + expf(-gv[0])), x[1] / (1.f + expf(-gv[1])), x[2] / (1.f + expf(-gv[2])),
                  x[3] / (1.f + expf(-gv[3]))};
    }
    st4(o + 4 * idx, x);
}

// MlpAct.run (model.zig:40-46) with nn.mulSilu (src/core/nn.zig:410-420): a[t, i] = gate * silu(up)
// with gate = h[t, i], up = h[t, hid + i].
__global__ void ts_mul_silu(const float* hbuf, float* a, int64_t tokens, int hid) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int h4 = hid / 4;
    if (idx >= tokens * h4) return;
    const int64_t t = idx / h4;
    const int c = (int)(idx % h4) * 4;
    const f32x4 g = ld4(hbuf + t * 2 * hid + c), u = ld4(hbuf + t * 2 * hid + hid + c);
    st4(a + t * hid + c, f32x4{g[0] * (u[0] / (1.f + expf(-u[0]))), g[1] * (u[1] / (1.f + expf(-u[1]))),
                               g[2] * (u[2] / (1.f + expf(-u[2]))), g[3] * (u[3] / (1.f + expf(-u[3])))});
}

// nn.clampNonfinite (src/core/nn.zig:522-563) of one quantile vector.
__device__ void clamp_nonfinite(float* v, int q) {
    float hi = -INFINITY, lo = INFINITY;
    bool any_inf = false;
    for (int i = 0; i < q; i++) {
        if (isfinite(v[i])) {
            hi = fmaxf(hi, v[i]);
            lo = fminf(lo, v[i]);
        } else if (isinf(v[i])) {
            any_inf = true;
        }
    }
    if (!any_inf) return;
    for (int i = 0; i < q; i++) {
        float d = v[i];
        if (d == INFINITY) d = hi;
        if (d == -INFINITY) d = lo;
        if (isinf(d)) d = 0.f;
        v[i] = d;
    }
}

// The monotone quantile head of predictBlock (model.zig:391-431): per (row, step) the median is
// free and the other levels fan out by cumulative softplus increments scaled by the knot widths,
// then back to data units with the last context patch's (loc, scale). raw: per decoder token
// ps * q outputs ordered (step, level); qs (rows, h * ps, q).
__global__ void ts_head_finish(const float* raw, const float* loc, const float* scale, int cap_p, int l, int rows,
                               int h, TsHead hp, float* qs) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int hl = h * hp.ps, q = hp.q, m = hp.median;
    if (idx >= (int64_t)rows * hl) return;
    const int r = (int)(idx / hl);
    const float* rv = raw + idx * q;  // token j = s / ps, step i = s % ps: (r * h + j) * ps * q + i * q
    float ov[32];
    const float med = rv[m], big = 3.40282347e38f;
    float acc = 0.f;
    for (int i = m + 1; i < q; i++) {
        const float x = rv[i];
        const float sp = x > 20.f ? x : log1pf(expf(x));
        acc += (hp.wf * hp.widths[i]) * sp;
        ov[i] = fmaxf(-big, fminf(med + acc, big));
    }
    acc = 0.f;
    for (int i = m - 1; i >= 0; i--) {
        const float x = rv[i];
        const float sp = x > 20.f ? x : log1pf(expf(x));
        acc += (hp.wf * hp.widths[i]) * sp;
        ov[i] = fmaxf(-big, fminf(med - acc, big));
    }
    ov[m] = med;
    const float lo = loc[(int64_t)r * cap_p + l - 1], sc = scale[(int64_t)r * cap_p + l - 1];
    for (int i = 0; i < q; i++) {
        const float y = hp.use_asinh ? sinhf(ov[i]) : ov[i];
        const float ys = y * sc;
        ov[i] = ys + lo;
    }
    clamp_nonfinite(ov, q);
    float* o = qs + idx * q;
    for (int i = 0; i < q; i++) o[i] = ov[i];
}

// refineBlock's frames (src/timestral/forecaster.zig:602-652): fold the block's medians (in the
// context's last-patch frame) patch by patch into the context's Welford state; frames[r, j] =
// (loc_j, scale_j), patch 0 keeping (loc0, scale0). One wave per row, a lane per step of the patch
// (ps <= 256: four a lane at most): the medians' divisions and their maps into the frame are
// spread over the lanes and the two sums of a patch are walked in the reference's order, by every
// lane alike (one thread per row: 130 us a block of 32 patches; now 27 us).
__global__ __launch_bounds__(64) void ts_refine_frames(const float* qs, const float* loc, const float* scale, int cap_p,
                                                       int l, const double* fold, int h, int ps, int q, int median,
                                                       double min_scale, float* frames) {
    __shared__ double fs[256];
    const int r = blockIdx.x, lane = threadIdx.x;
    const float loc0 = loc[(int64_t)r * cap_p + l - 1], scale0 = scale[(int64_t)r * cap_p + l - 1];
    double w = fold[(int64_t)r * 3 + 0], mean = fold[(int64_t)r * 3 + 1], m2 = fold[(int64_t)r * 3 + 2];
    const double clip = sqrt((double)3.40282347e38f) / 1e3, offset = mean;
    const float* block = qs + (int64_t)r * h * ps * q;
    float* fr = frames + (int64_t)r * h * 2;
    auto frame_units = [&](int j, int k) {
        return ((double)block[(int64_t)(j * ps + k) * q + median] - (double)loc0) / (double)scale0;
    };
    double sm[4];
#pragma unroll
    for (int e = 0; e < 4; e++) sm[e] = lane + 64 * e < ps ? frame_units(0, lane + 64 * e) : 0.0;
    for (int j = 0; j < h; j++) {
        const double variance = fmax_d(m2 / fmax_d(w - 1.0, 1.0), 0.0);
        const double sc = fmax_d(sqrt(variance), min_scale);
        if (lane == 0) {
            fr[2 * j] = j == 0 ? loc0 : (float)mean;
            fr[2 * j + 1] = j == 0 ? scale0 : (float)sc;
        }
        // The block's medians of patch j mapped into this frame.
        double f[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const double v = sm[e] * sc + mean - offset;
            f[e] = fmax_d(-clip, fmin(v, clip)) + offset;
            if (lane + 64 * e < ps) fs[lane + 64 * e] = f[e];
        }
        if (j + 1 < h) {
#pragma unroll
            for (int e = 0; e < 4; e++) sm[e] = lane + 64 * e < ps ? frame_units(j + 1, lane + 64 * e) : 0.0;
        }
        __syncthreads();
        double bsum = 0;
#pragma unroll 8
        for (int k = 0; k < ps; k++) bsum += fs[k];
        const double bmean = bsum / (double)ps;
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (lane + 64 * e < ps) fs[lane + 64 * e] = (f[e] - bmean) * (f[e] - bmean);
        __syncthreads();
        double bm2 = 0;
#pragma unroll 8
        for (int k = 0; k < ps; k++) bm2 += fs[k];
        __syncthreads();
        // welfordCombine(state, (ps, bmean, bm2))
        const double bw = (double)ps, nw = w + bw;
        if (nw == 0) {
            w = 0; mean = 0; m2 = 0;
        } else {
            const double w_safe = fmax_d(nw, 2.2250738585072014e-308);
            const double delta = bmean - mean;
            const double nm = mean + delta * bw / w_safe;
            const double n2 = m2 + bm2 + delta * delta * w * bw / w_safe;
            w = nw; mean = nm; m2 = n2;
        }
    }
}

// refineBlock's rescale (forecaster.zig:653-659): (x - loc0) / scale0 * scale_j + loc_j, then
// nn.clampNonfinite of each step's levels.
__global__ void ts_refine_apply(float* qs, const float* frames, int rows, int h, int ps, int q) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int hl = h * ps;
    if (idx >= (int64_t)rows * hl) return;
    const int r = (int)(idx / hl), s = (int)(idx % hl);
    const float* fr = frames + (int64_t)r * h * 2;
    const float loc0 = fr[0], scale0 = fr[1], lj = fr[2 * (s / ps)], sj = fr[2 * (s / ps) + 1];
    float v[32];
    float* rowq = qs + idx * q;
    for (int i = 0; i < q; i++) {
        const float a = (rowq[i] - loc0) / scale0;
        const float b = a * sj;
        v[i] = b + lj;
    }
    clamp_nonfinite(v, q);
    for (int i = 0; i < q; i++) rowq[i] = v[i];
}

// Store a block's quantiles: steps [done, done + blen) of each row's forecast, those before the
// horizon (blockDecode :502-507). Rows r < R go to out, the mirrored rows to mir.
__global__ void ts_store_block(const float* qs, int rows, int batch, int vall, int V, int blen, int done, int horizon,
                               int q, float* out, float* mir) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)rows * blen * q) return;
    const int i = (int)(idx % q);
    const int64_t rs = idx / q;
    const int r = (int)(rs / blen), s = (int)(rs % blen);
    const int g = r / vall, vi = r % vall;
    if (done + s >= horizon || vi >= V) return;
    const int64_t orow = (int64_t)(g < batch ? g : g - batch) * V + vi;
    float* dst = (g < batch ? out : mir) + (orow * horizon + done + s) * q;
    dst[i] = qs[idx];
}

// blockDecode's feedback (forecaster.zig:512-555) for target rows: the block's medians (0 when not
// finite or at least the extreme threshold) become observed steps [t, t + blen) of the context.
__global__ void ts_feedback(const float* qs, int rows, int vall, int V, int blen, int q, int median, float extreme,
                            float* ctx, uint8_t* mask, int cap_t, int t) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)rows * blen) return;
    const int r = (int)(idx / blen), s = (int)(idx % blen);
    if (r % vall >= V) return;  // covariate rows: the window already holds their next steps
    float mv = qs[idx * q + median];
    if (!isfinite(mv) || fabsf(mv) >= extreme) mv = 0.f;
    ctx[(int64_t)r * cap_t + t + s] = mv;
    mask[(int64_t)r * cap_t + t + s] = 1;
}

// The context window after a drop of the oldest steps (forecaster.zig:514-530): dst[r, j] =
// src[r, start + j] for j < keep.
__global__ void ts_slide(const float* src, const uint8_t* src_mask, float* dst, uint8_t* dst_mask, int rows, int cap_t,
                         int start, int keep) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)rows * keep) return;
    const int r = (int)(idx / keep), j = (int)(idx % keep);
    dst[(int64_t)r * cap_t + j] = src[(int64_t)r * cap_t + start + j];
    dst_mask[(int64_t)r * cap_t + j] = src_mask[(int64_t)r * cap_t + start + j];
}

// forecastRaw's quantile cap (forecaster.zig:396-418) bounds of each row from its original context:
// [min - a, max + a] over the observed values (0 when none), a = scale of the last patch x cap_k.
// One wave per row (a thread per row: 228 us at 24 rows x 1504 steps; now 7 us).
__global__ __launch_bounds__(64) void ts_cap_bounds(const float* ctx, const uint8_t* mask, int cap_t, int t, int ps,
                                                    const float* scale, int cap_p, float cap_k, float* bounds) {
    const int r = blockIdx.x, lane = threadIdx.x;
    float mx = -INFINITY, mn = INFINITY;
    for (int j = lane; j < t; j += 64)
        if (mask[(int64_t)r * cap_t + j]) {
            mx = fmaxf(mx, ctx[(int64_t)r * cap_t + j]);
            mn = fminf(mn, ctx[(int64_t)r * cap_t + j]);
        }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        mx = fmaxf(mx, __shfl_xor(mx, d));
        mn = fminf(mn, __shfl_xor(mn, d));
    }
    if (lane != 0) return;
    if (isinf(mx)) mx = 0.f;
    if (isinf(mn)) mn = 0.f;
    const float a = scale[(int64_t)r * cap_p + t / ps - 1] * cap_k;
    bounds[2 * r] = mn - a;
    bounds[2 * r + 1] = mx + a;
}

// forecast's end (forecaster.zig:107-140, finish :163-178): each pass capped to its own bounds
// (std.math.clamp: @max(lo, @min(x, hi))), the mirrored pass averaged in level-reversed order, and
// series whose observed values are all non-negative clipped at 0.
__global__ void ts_final(float* out, const float* mir, const float* bounds, const uint8_t* nonneg, int R, int V,
                         int vall, int horizon, int q, int cap, int symmetric, int clip) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)R * horizon) return;
    const int r = (int)(idx / horizon);
    // bounds are per context row: target i of series s is row s * vall + i, its mirror R / V groups on
    const int fr = (r / V) * vall + r % V, mr = fr + (R / V) * vall;
    float* o = out + idx * q;
    float v[32];
    for (int j = 0; j < q; j++) {
        float f = o[j];
        if (cap) f = fmaxf(bounds[2 * fr], fminf(f, bounds[2 * fr + 1]));
        v[j] = f;
    }
    if (symmetric) {
        const float* m = mir + idx * q;
        for (int j = 0; j < q; j++) {
            float g = m[q - 1 - j];
            if (cap) g = fmaxf(bounds[2 * mr], fminf(g, bounds[2 * mr + 1]));
            const float s = v[j] + -g;
            v[j] = 0.5f * s;
        }
    }
    const bool cl = clip && nonneg[r];
    for (int j = 0; j < q; j++) o[j] = cl ? fmaxf(v[j], 0.f) : v[j];
}

unsigned blocks_for(int64_t n, int per) { return (unsigned)((n + per - 1) / per); }

}  // namespace

hipError_t launch_ts_stats(const TsStatsParams& p, hipStream_t s) {
    hipLaunchKernelGGL(ts_stats, dim3((unsigned)p.rows), dim3(kStatsT), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_ts_features(const float* ctx, const uint8_t* mask, int cap_t, const float* loc, const float* scale,
                              int cap_p, int rows, int p0, int l, int ps, int use_asinh, const uint8_t* no_asinh,
                              float* feats, hipStream_t s) {
    const int64_t n = (int64_t)rows * (l - p0) * ps;
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(ts_features, dim3(blocks_for(n, 256)), dim3(256), 0, s, ctx, mask, cap_t, loc, scale, cap_p, rows,
                       p0, l, ps, use_asinh, no_asinh, feats);
    return hipGetLastError();
}

hipError_t launch_ts_rope_tables(const int* row_first, int groups, int vall, int n_tok, int ne, int shift,
                                 const TsRope& rp, float* cos_t, float* sin_t, int* first_obs, hipStream_t s) {
    hipLaunchKernelGGL(ts_rope_tables, dim3(blocks_for((int64_t)n_tok * 32, 256), (unsigned)groups), dim3(256), 0, s,
                       row_first, vall, n_tok, ne, shift, rp, cos_t, sin_t, first_obs);
    return hipGetLastError();
}

hipError_t launch_ts_assemble(const float* emb, const float* query, float* x, int rows, int m, int h, int d,
                              hipStream_t s) {
    hipLaunchKernelGGL(ts_assemble, dim3(blocks_for((int64_t)rows * (m + h) * (d / 4), 256)), dim3(256), 0, s, emb,
                       query, x, rows, m, h, d);
    return hipGetLastError();
}

hipError_t launch_ts_mul_sigmoid(float* o, const float* g, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL(ts_mul_sigmoid, dim3(blocks_for(n / 4, 256)), dim3(256), 0, s, o, g, n / 4);
    return hipGetLastError();
}

hipError_t launch_ts_from_bf16(const uint16_t* oh, const float* g, float* o, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL(ts_from_bf16, dim3(blocks_for(n / 4, 256)), dim3(256), 0, s, oh, g, o, n / 4);
    return hipGetLastError();
}

hipError_t launch_ts_mul_silu(const float* hbuf, float* a, int64_t tokens, int hid, hipStream_t s) {
    hipLaunchKernelGGL(ts_mul_silu, dim3(blocks_for(tokens * (hid / 4), 256)), dim3(256), 0, s, hbuf, a, tokens, hid);
    return hipGetLastError();
}

hipError_t launch_ts_head_finish(const float* raw, const float* loc, const float* scale, int cap_p, int l, int rows,
                                 int h, const TsHead& hp, float* qs, hipStream_t s) {
    hipLaunchKernelGGL(ts_head_finish, dim3(blocks_for((int64_t)rows * h * hp.ps, 128)), dim3(128), 0, s, raw, loc,
                       scale, cap_p, l, rows, h, hp, qs);
    return hipGetLastError();
}

hipError_t launch_ts_refine(float* qs, const float* loc, const float* scale, int cap_p, int l, const double* fold,
                            int rows, int h, int ps, int q, int median, double min_scale, float* frames,
                            hipStream_t s) {
    if (ps > 256) return hipErrorInvalidValue;  // four steps a lane
    hipLaunchKernelGGL(ts_refine_frames, dim3((unsigned)rows), dim3(64), 0, s, qs, loc, scale, cap_p, l, fold, h, ps, q,
                       median, min_scale, frames);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(ts_refine_apply, dim3(blocks_for((int64_t)rows * h * ps, 128)), dim3(128), 0, s, qs, frames, rows,
                       h, ps, q);
    return hipGetLastError();
}

hipError_t launch_ts_store_block(const float* qs, int rows, int batch, int vall, int V, int blen, int done, int horizon,
                                 int q, float* out, float* mir, hipStream_t s) {
    hipLaunchKernelGGL(ts_store_block, dim3(blocks_for((int64_t)rows * blen * q, 256)), dim3(256), 0, s, qs, rows,
                       batch, vall, V, blen, done, horizon, q, out, mir);
    return hipGetLastError();
}

hipError_t launch_ts_feedback(const float* qs, int rows, int vall, int V, int blen, int q, int median, float extreme,
                              float* ctx, uint8_t* mask, int cap_t, int t, hipStream_t s) {
    hipLaunchKernelGGL(ts_feedback, dim3(blocks_for((int64_t)rows * blen, 256)), dim3(256), 0, s, qs, rows, vall, V,
                       blen, q, median, extreme, ctx, mask, cap_t, t);
    return hipGetLastError();
}

hipError_t launch_ts_slide(const float* src, const uint8_t* src_mask, float* dst, uint8_t* dst_mask, int rows,
                           int cap_t, int start, int keep, hipStream_t s) {
    hipLaunchKernelGGL(ts_slide, dim3(blocks_for((int64_t)rows * keep, 256)), dim3(256), 0, s, src, src_mask, dst,
                       dst_mask, rows, cap_t, start, keep);
    return hipGetLastError();
}

hipError_t launch_ts_cap_bounds(const float* ctx, const uint8_t* mask, int cap_t, int t, int ps, const float* scale,
                                int cap_p, int rows, float cap_k, float* bounds, hipStream_t s) {
    hipLaunchKernelGGL(ts_cap_bounds, dim3((unsigned)rows), dim3(64), 0, s, ctx, mask, cap_t, t, ps, scale, cap_p, cap_k,
                       bounds);
    return hipGetLastError();
}

hipError_t launch_ts_final(float* out, const float* mir, const float* bounds, const uint8_t* nonneg, int R, int V,
                           int vall, int horizon, int q, int cap, int symmetric, int clip, hipStream_t s) {
    hipLaunchKernelGGL(ts_final, dim3(blocks_for((int64_t)R * horizon, 128)), dim3(128), 0, s, out, mir, bounds, nonneg,
                       R, V, vall, horizon, q, cap, symmetric, clip);
    return hipGetLastError();
}

}  // namespace tsfm
