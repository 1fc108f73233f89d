// cts_bbi.hip -- broadband impedance in the frequency domain, longitudinal,
// dipolar and quadrupolar planes (MPBunch::BBImpBunchInteraction,
// src/MPBunch.cpp:2143-2312).
//
// The reference bins a bunch on the centred grid of BoardBandImp::ReadInImp
// (src/BoardBandImp.cpp:71-90: N = 2 nimp - 1 bins of dz = c beta/(2 f_max)
// from -z_max), smooths the profile over one RF bucket, takes its real FFT,
// multiplies by Z_k, and returns V = -c2r(...)/N.  With Z extended as a
// Hermitian sequence (the c2r transform ignores Im Z_0) that is the circular
// convolution V_j = -sum_i p_i g_{(j - i) mod N} with the real kernel
//   g_m = (1/N) [Re Z_0 + 2 sum_{k=1}^{nimp-1} Re(Z_k e^{2 pi i k m / N})],
// computed once on the host.  The transverse planes multiply the spectrum by
// i Z and keep the + sign; the quadrupolar ones use the charge profile, the
// dipolar ones the x- and y-weighted profiles (sum of charge times x per
// bin).  Per turn: LDS histograms of shares of the bunches (with the
// dipolar planes, the per-bin sums of x and y as two-limb fixed-point
// integers, so they do not depend on the order of the atomics), a block per
// profile for the smoothing, a block per 256 bins and plane for the
// convolutions, and a kick with a particle per thread.  The smoothing is GSL's gsl_filter_gaussian (GSL 2.8, the version the
// reference builds against) with K = 51, alpha = 10 and
// GSL_FILTER_END_PADVALUE: y_i = sum_j w_j x_{clamp(i + j - 25)},
// w_j = exp(-alpha^2 ((j - 25)/25)^2 / 2) normalised to sum 1, followed by
// the reference's rescaling to the input's sum (src/MPBunch.cpp:2373-2410).
//
// The time-domain method (MPBunch::BBImpBunchInteractionTD,
// src/MPBunch.cpp:2029-2142, the reference's default) bins a bunch over one
// RF bucket, (int)((z + L/2)/dz) on (int)(L/dz) bins with dz the wake
// table's step, smooths the charge profile rho (charge per bin) the same
// way, takes the mean x and y of each bin, and sums the wake table over the
// bins behind each one: V_i = -sum_{j >= i} w[j - i] rho_j (the dipolar
// planes rho_j <x>_j).  No transform: the sums run over the bins where rho
// is nonzero (zeros add nothing).
#include <climits>
#include <cmath>
#include <string>
#include <vector>

#include "cts_internal.hpp"

namespace cts {

namespace {

// time domain: the wake table stands in for the kernels
int bbimp_table_td(const cts_bbimp_config &c, const cts_ring &ring, BbiTable &t, std::string &err)
{
    const double *w[5] = {c.wake_z, c.wake_dx, c.wake_dy, c.wake_qx, c.wake_qy};
    bool given = c.wake_pos != nullptr;
    for (int q = 0; q < 5; q++) given = given && (!t.planes[q] || w[q]);
    if (c.nwake < 2 || !given) {
        err = "cts_set_bbimp: time domain: nwake >= 2, wake_pos and the wake of every plane switched on";
        return CTS_ERR_ARG;
    }
    // dzBin and nBinBunchDen of src/MPBunch.cpp:2036-2040
    const double dz = std::fabs(c.wake_pos[1] - c.wake_pos[0]);
    const double rf_len = ring.t0 / ring.harmonic * kClight;
    const double nbins = rf_len / dz;
    if (!(dz > 0) || !(nbins >= 1.0) || !(nbins < kBbiMaxGridTD + 1.0)) {
        err = "cts_set_bbimp: time domain: the wake's step must cut the RF bucket (" + std::to_string(rf_len) +
              " m) into 1 to " + std::to_string(kBbiMaxGridTD) + " bins";
        return CTS_ERR_ARG;
    }
    t.td = 1;
    t.nw = c.nwake;
    t.n = (int)(1 * rf_len / dz);
    t.dz = dz;
    t.zmin = -1 * rf_len / 2;
    t.half = 0.0;
    t.is = 0;
    t.ie = t.n;
    t.g.assign(5 * (size_t)t.nw, 0.0);
    for (int q = 0; q < 5; q++)
        if (t.planes[q]) std::copy(w[q], w[q] + t.nw, t.g.begin() + (size_t)q * t.nw);
    return CTS_OK;
}

}  // namespace

int bbimp_table(const cts_bbimp_config &c, const cts_ring &ring, BbiTable &t, std::string &err)
{
    // planes in the reference's flag order: Z, Dx, Dy, Qx, Qy
    for (int q = 0; q < 5; q++) t.planes[q] = c.flags[q] != 0;
    const bool tx = t.planes[1] || t.planes[3], ty = t.planes[2] || t.planes[4];
    if ((tx && !(c.beta_x > 0)) || (ty && !(c.beta_y > 0))) {
        err = "cts_set_bbimp: beta_x, beta_y > 0 for the transverse planes";
        return CTS_ERR_ARG;
    }
    t.bx = tx ? c.beta_x : 1.0;
    t.by = ty ? c.beta_y : 1.0;
    int rc;
    if (c.time_domain == 1) {
        if ((rc = bbimp_table_td(c, ring, t, err))) return rc;
    } else if (c.time_domain == 0) {
        const double *zr[5] = {c.zz_re, c.zdx_re, c.zdy_re, c.zqx_re, c.zqy_re};
        const double *zi[5] = {c.zz_im, c.zdx_im, c.zdy_im, c.zqx_im, c.zqy_im};
        bool given = true;
        for (int q = 0; q < 5; q++) given = given && (!t.planes[q] || (zr[q] && zi[q]));
        const int n = 2 * c.nimp - 1;
        if (c.nimp < 2 || n > kBbiMaxGridFD || !(c.f_max > 0) || !given) {
            err = "cts_set_bbimp: nimp in [2, " + std::to_string((kBbiMaxGridFD + 1) / 2) +
                  "], f_max > 0, the impedance of every plane switched on";
            return CTS_ERR_ARG;
        }
        const int nimp = c.nimp;
        const double dt = 1.0 / (2 * c.f_max);
        t.n = n;
        t.dz = dt * kClight * ring.rbeta;
        t.half = t.dz / 2;
        const double zmax = t.dz * (nimp - 1);
        t.zmin = -zmax;
        // one RF bucket, indexed as GetSmoothedBunchProfileGassionFilter does
        const double rf_len = ring.t0 / ring.harmonic * kClight;
        t.is = (int)((-rf_len / 2. - t.zmin + t.dz / 2) / t.dz);
        t.ie = (int)((rf_len / 2. - t.zmin + t.dz / 2) / t.dz);
        if (-rf_len / 2. - t.zmin + t.dz / 2 < 0 || t.ie > n || t.ie <= t.is) {
            err = "cts_set_bbimp: the impedance grid (z_max " + std::to_string(zmax) +
                  " m) must cover one RF bucket (" + std::to_string(rf_len) + " m)";
            return CTS_ERR_ARG;
        }
        t.g.assign(5 * (size_t)n, 0.0);
        for (int q = 0; q < 5; q++) {
            if (!t.planes[q]) continue;
            // the transverse planes multiply the spectrum by i Z: (re, im) -> (-im, re)
            auto re = [&](int k) { return q == 0 ? zr[q][k] : -zi[q][k]; };
            auto im = [&](int k) { return q == 0 ? zi[q][k] : zr[q][k]; };
            for (int m = 0; m < n; m++) {
                double s = 0;
                for (int k = 1; k < nimp; k++) {
                    // exact reduction of the phase k m / n
                    const double ph = 2 * M_PI * (double)(((int64_t)k * m) % n) / n;
                    s += re(k) * std::cos(ph) - im(k) * std::sin(ph);
                }
                t.g[(size_t)q * n + m] = (re(0) + 2 * s) / n;
            }
        }
    } else {
        // the reference prints "wrong setting in BoardBandImpedance namelist"
        // every turn and applies nothing (src/MPBeam.cpp:1345)
        err = "cts_set_bbimp: time_domain 0 (frequency domain) or 1 (time domain)";
        return CTS_ERR_ARG;
    }
    const int half = (kBbiTaps - 1) / 2;
    const double alpha = 10.0;
    double sum = 0;
    for (int j = 0; j < kBbiTaps; j++) {
        const double xj = (j - half) / (double)half;
        t.taps[j] = std::exp(-0.5 * alpha * alpha * xj * xj);
        sum += t.taps[j];
    }
    for (int j = 0; j < kBbiTaps; j++) t.taps[j] /= sum;
    return CTS_OK;
}

namespace {

// bin of z as the reference indexes it, (int)((z - zmin + dz/2)/dz) in the
// frequency domain, (int)((z - zmin)/dz) in the time domain, or -1 off the
// grid (the reference does not test the range).  With the reciprocal, and
// the division where the two could truncate apart.
__device__ __forceinline__ double bbi_pos(double z, const BbiParams &P)
{
    const double d = z - P.zmin + P.half;
    double q = d * P.inv_dz;
    if (fabs(q - rint(q)) < 1e-9) q = d / P.dz;
    return q;
}
__device__ __forceinline__ int bbi_bin(double z, const BbiParams &P)
{
    const double q = bbi_pos(z, P);
    return (q > -1.0 && q < (double)P.n) ? (int)q : -1;
}

// survivors before this turn's loss marking
__device__ __forceinline__ bool bbi_alive(uint8_t f) { return (f & 3u) == 0u || (f & kNewLost); }

// a coordinate as two integer limbs, v ~ hi 2^-30 + lo 2^-62, hi =
// floor(v 2^30), 0 <= lo <= 2^32: the limb sums of up to 2^31 values with
// |v| < 1 stay inside 64 bits, and their total does not depend on the order
// of the additions (the conversion is exact up to 2^-85 for |v| < 2^-30
// below zero, a fixed rounding of the value itself)
__device__ __forceinline__ void fx2_split(double v, unsigned long long &hi, unsigned long long &lo)
{
    const double h = floor(ldexp(v, 30));
    hi = (unsigned long long)(long long)h;
    lo = (unsigned long long)(long long)rint(ldexp(v - ldexp(h, -30), 62));
}
__device__ __forceinline__ double fx2_value(unsigned long long hi, unsigned long long lo)
{
    return ldexp((double)(long long)hi, -30) + ldexp((double)(long long)lo, -62);
}

}  // namespace

// LDS of the binning: counts, then (dipolar planes) four limb sums per bin
__host__ __device__ constexpr int bbi_count_words(bool dip) { return dip ? ((kBbiDipWin + 1) & ~1) : kBbiWin; }

// Binning, a share of one bunch per block, bound by the time its few loads
// and LDS atomics take one after another.  The window is the bins of the
// survivors' z range, which the turn's moments hold (no sweep for the range);
// a macroparticle marked lost this turn may lie outside and goes to the
// bunch's sums directly.  A bunch fills few bins, so the window is kept in as
// many copies as fit, up to one per wave: the atomics of different waves do
// not meet.  With one window of the whole grid per workgroup of the pass 37 us
// on 60 bunches of 6e4 with both dipolar planes, 31 now by events around the
// launch, 28 in a kernel trace (by events, blocks of 512 threads 30, of 1024
// 40); without the planes 15 (512: 16, 1024: 22).
__global__ void __launch_bounds__(kBbiBinBlock) k_bbi_bin(BbiParams P)
{
    extern __shared__ __attribute__((aligned(16))) uint32_t hl[];
    constexpr int U = 4, kCopies = kBbiBinBlock / 64;
    const int tid = threadIdx.x, b = P.item_bunch[blockIdx.x];
    if (P.scale[b] == 0.0) return;  // uniform
    const bool dipx = P.planes[1] != 0, dipy = P.planes[2] != 0, dip = dipx || dipy;
    const int64_t first = P.bunch_off[b], n = P.bunch_off[b + 1] - first;
    const int nblk = P.item_first[b + 1] - P.item_first[b];
    const int64_t per = (n + nblk - 1) / nblk;
    const int64_t i0 = first + (int64_t)(blockIdx.x - P.item_first[b]) * per, i1 = min(first + n, i0 + per);
    if (i0 >= i1) return;
    const auto edge = [&](double z) {
        const double q = bbi_pos(z, P);
        return q > 0.0 ? (q < (double)P.n ? (int)q : P.n - 1) : 0;
    };
    const int klo = edge(P.cur[b].zmin), khi = max(klo, edge(P.cur[b].zmax)), R = khi - klo + 1;
    const int cap = dip ? kBbiDipWin : kBbiWin, W = min(R, cap), nc = min(kCopies, cap / W);
    // [copy][bin] counts; [copy][limb][bin] x hi, x lo, y hi, y lo
    const int copy = tid / 64 % nc;
    uint32_t *hc = hl + copy * W;
    unsigned long long *ds = reinterpret_cast<unsigned long long *>(hl + bbi_count_words(dip));
    unsigned long long *dc = ds + (size_t)copy * 4 * W;
    uint32_t *gh = P.hist + (int64_t)b * P.n;
    unsigned long long *gd = P.dsum + (int64_t)b * 4 * P.n;  // not read without the dipolar planes
    for (int w0 = klo; w0 <= khi; w0 += W) {
        const int wn = min(W, khi - w0 + 1);
        for (int j = tid; j < nc * W; j += kBbiBinBlock) hl[j] = 0u;
        if (dip)
            for (int j = tid; j < 4 * nc * W; j += kBbiBinBlock) ds[j] = 0ull;
        __syncthreads();
        for (int64_t i = i0 + tid; i < i1; i += U * kBbiBinBlock) {
            double zz[U], xx[U], yy[U];
            uint8_t ff[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int64_t k = min(i + u * kBbiBinBlock, i1 - 1);
                ff[u] = P.flag[k];
                zz[u] = P.z[k];
                xx[u] = dipx ? P.x[k] : 0.0;
                yy[u] = dipy ? P.y[k] : 0.0;
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (i + u * kBbiBinBlock >= i1 || !bbi_alive(ff[u])) continue;
                const int k = bbi_bin(zz[u], P), kw = k - w0;
                unsigned long long xh, xl, yh, yl;
                if (dipx) fx2_split(xx[u], xh, xl);
                if (dipy) fx2_split(yy[u], yh, yl);
                if (kw >= 0 && kw < wn) {
                    atomicAdd(&hc[kw], 1u);
                    if (dipx) {
                        atomicAdd(&dc[kw], xh);
                        atomicAdd(&dc[W + kw], xl);
                    }
                    if (dipy) {
                        atomicAdd(&dc[2 * W + kw], yh);
                        atomicAdd(&dc[3 * W + kw], yl);
                    }
                } else if (w0 == klo && k >= 0 && (k < klo || k > khi)) {
                    atomicAdd(&gh[k], 1u);
                    if (dipx) {
                        atomicAdd(&gd[4 * k], xh);
                        atomicAdd(&gd[4 * k + 1], xl);
                    }
                    if (dipy) {
                        atomicAdd(&gd[4 * k + 2], yh);
                        atomicAdd(&gd[4 * k + 3], yl);
                    }
                }
            }
        }
        __syncthreads();
        for (int j = tid; j < wn; j += kBbiBinBlock) {
            uint32_t c = 0;
            for (int q = 0; q < nc; q++) c += hl[q * W + j];
            if (c) atomicAdd(&gh[w0 + j], c);
        }
        if (dip)
            for (int j = tid; j < 4 * wn; j += kBbiBinBlock) {
                unsigned long long v = 0;
                for (int q = 0; q < nc; q++) v += ds[(4 * q + (j & 3)) * W + (j >> 2)];
                if (v) atomicAdd(&gd[4 * (int64_t)w0 + j], v);
            }
        __syncthreads();
    }
}

// One profile of one bunch (blockIdx.y: charge, x- and y-weighted): the
// smoothed values over [is, ie) (the reference's
// GetSmoothedBunchProfileGassionFilter), raw ones elsewhere; the time
// domain's other two are the mean x and y per bin.  The raw profile vanishes
// outside the bins that hold particles, [lo, hi], so the smoothed one does
// outside [lo - 25, hi + 25]: only those are formed, from LDS tiles.  One
// block per bunch did this and the convolutions in 60.9 us on 60 bunches of
// 1200 bins; the two launches take 17.5.
__global__ void __launch_bounds__(kBlock) k_bbi_prof(BbiParams P)
{
    constexpr int T = 1024, half = (kBbiTaps - 1) / 2;
    __shared__ double tile[T + 2 * half], red[2][kBlock];
    __shared__ int krange[2];
    const int b = blockIdx.x, r = blockIdx.y, tid = threadIdx.x;
    if (r > 0 && !P.planes[r]) return;
    const double sc = P.scale[b];
    if (sc == 0.0) return;  // the tables stay zero
    const uint32_t *cnt = P.hist + (int64_t)b * P.n;
    const unsigned long long *ds = P.dsum + (int64_t)b * 4 * P.n + 2 * (r - 1);  // read for r > 0
    double *prof = P.prof + ((int64_t)r * P.nb + b) * P.n;
    if (tid == 0) { krange[0] = INT_MAX; krange[1] = -1; }
    __syncthreads();
    {
        int lo = INT_MAX, hi = -1;
#pragma unroll 8
        for (int j = tid; j < P.n; j += kBlock)
            if (cnt[j]) { lo = min(lo, j); hi = max(hi, j); }
        if (hi >= 0) { atomicMin(&krange[0], lo); atomicMax(&krange[1], hi); }
    }
    __syncthreads();
    const bool any = krange[1] >= krange[0];
    const int lo = any ? krange[0] : 0, hi = any ? krange[1] : -1;
    if (r == 0 && tid == 0) { P.range[2 * b] = lo; P.range[2 * b + 1] = hi; }
    if (P.td && r > 0) {
        for (int j = tid; j < P.n; j += kBlock)
            prof[j] = cnt[j] ? fx2_value(ds[4 * j], ds[4 * j + 1]) / cnt[j] : 0.0;
        return;
    }
    const auto raw = [&](int i) { return r == 0 ? (double)cnt[i] * sc : sc * fx2_value(ds[4 * i], ds[4 * i + 1]); };
    const int a = max(P.is, lo - half), e = min(P.ie, hi + half + 1);
    double s0 = 0, s1 = 0;
    for (int t0 = a; t0 < e; t0 += T) {
        const int tn = min(T, e - t0);
        __syncthreads();  // the tile before
        for (int m = tid; m < tn + 2 * half; m += kBlock)
            tile[m] = raw(min(max(t0 - half + m, P.is), P.ie - 1));
        __syncthreads();
        for (int i = tid; i < tn; i += kBlock) {
            double y = 0;
#pragma unroll
            for (int j = 0; j < kBbiTaps; j++) y += P.taps[j] * tile[i + j];
            s0 += tile[i + half];
            s1 += y;
            prof[t0 + i] = y;  // scaled below by the same thread
        }
    }
    red[0][tid] = s0;
    red[1][tid] = s1;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if (tid < w) { red[0][tid] += red[0][tid + w]; red[1][tid] += red[1][tid + w]; }
        __syncthreads();
    }
    const double f = red[1][0] != 0.0 ? red[0][0] / red[1][0] : 0.0;
    for (int i = a + tid; i < e; i += kBlock) prof[i] *= f;
    for (int i = tid; i < P.n; i += kBlock)
        if (i < a || i >= e) prof[i] = (i >= P.is && i < P.ie) ? 0.0 : raw(i);
}

// The induced voltage of one plane (blockIdx.z) on 256 bins of one bunch:
// frequency domain, longitudinal V = -IDFT(I Z) and transverse
// V = +IDFT(I i Z), circular convolutions of the profile (dipolar planes: the
// weighted ones); time domain, V_i = -sum_{j >= i} w[j - i] rho_j (dipolar
// planes rho_j <x>_j) over the rows of the wake (src/MPBunch.cpp:2100-2111).
// Both sum over the nonzero part of the profile in the order of its bins, with
// tiles of profile and weights in LDS.  The voltage over energy, beta^2 (and
// beta function, where the kick has it first) goes to the kick's own table:
// no division per macroparticle.  Clears the bins' sums for the next turn
// (stores, no memset node).
__global__ void __launch_bounds__(kBlock) k_bbi_wake(BbiParams P)
{
    constexpr int T = 256;
    __shared__ double pr[T], gt[T + kBlock];
    const int b = blockIdx.x, q = blockIdx.z, tid = threadIdx.x;
    const int o0 = blockIdx.y * kBlock, o = o0 + tid, n = P.n;
    if (P.scale[b] == 0.0) return;  // the tables stay zero
    const int lo = P.range[2 * b], hi = P.range[2 * b + 1];
    if (q == 0 && o < n) {
        P.hist[(int64_t)b * n + o] = 0u;
        if (P.dsum)
            for (int c = 0; c < 4; c++) P.dsum[((int64_t)b * n + o) * 4 + c] = 0ull;
    }
    if (!P.planes[q]) return;
    const int half = (kBbiTaps - 1) / 2;
    // every nonzero value of a profile lies in [plo, phi]
    const int plo = max(0, lo - half), phi = min(n - 1, hi + half);
    const double *g = P.g + (int64_t)q * (P.td ? P.nw : n);
    const double *rho = P.prof + ((P.td || q > 2 ? 0 : (int64_t)q * P.nb) + b) * n;
    const double *avg = P.td && (q == 1 || q == 2) ? P.prof + ((int64_t)q * P.nb + b) * n : nullptr;
    double v = 0;
    // a tile of sources can matter to the time domain's bins only where
    // 0 <= j - i < nw for some pair
    const int s_first = P.td ? max(plo, o0) : plo;
    const int s_last = P.td ? (int)min((int64_t)phi, (int64_t)o0 + kBlock - 1 + P.nw - 1) : phi;
    for (int s0 = s_first; s0 <= s_last; s0 += T) {
        const int sn = min(T, s_last - s0 + 1);
        __syncthreads();  // the tiles before
        if (tid < sn) pr[tid] = avg ? rho[s0 + tid] * avg[s0 + tid] : rho[s0 + tid];
        // gt[k]: weight of the source sl of the tile in the bin ol of the
        // block at k = ol - sl + T - 1
        for (int k = tid; k < T + kBlock - 1; k += kBlock) {
            const int d = o0 - s0 + k - (T - 1);  // bin - source
            if (P.td) gt[k] = (d <= 0 && -d < P.nw) ? g[-d] : 0.0;
            else gt[k] = g[((d % n) + n) % n];
        }
        __syncthreads();
        const double *w = gt + tid + T - 1;
#pragma unroll 8
        for (int sl = 0; sl < sn; sl++) v = fma(pr[sl], w[-sl], v);
    }
    if (o >= n) return;
    if (P.td || q == 0) v = -v;
    const int64_t at = ((int64_t)q * P.nb + b) * n + o;
    P.wake[at] = v;
    double k = v / P.energy / P.beta2;
    if (q == 1 || (q == 3 && P.td)) k = k / P.bx;
    if (q == 2 || (q == 4 && P.td)) k = k / P.by;
    P.kick[at] = k;
}

// A block of up to 256 macroparticles of one bunch, one per thread with all
// its loads issued at once (the kick moves 25 bytes of each, 73 with all planes,
// and little else; with four per thread in a loop and the divisions by energy, beta^2
// and the beta functions 59.4 us on 60 bunches of 6e4, now 42).
__global__ void __launch_bounds__(kBlock) k_bbi_kick(BbiParams P)
{
    const int b = P.kick_bunch[blockIdx.x];
    const int64_t i = P.bunch_off[b] + (int64_t)(blockIdx.x - P.kick_first[b]) * kBlock + threadIdx.x;
    if (i >= P.bunch_off[b + 1] || P.scale[b] == 0.0) return;
    const bool dx = P.planes[1] != 0, dy = P.planes[2] != 0, qx = P.planes[3] != 0, qy = P.planes[4] != 0;
    const uint8_t f = P.flag[i];
    const double z = P.z[i];
    double d = 0, px = 0, py = 0, x = 0, y = 0;
    if (P.planes[0]) d = P.dp[i];
    if (dx || qx) px = P.px[i];
    if (dy || qy) py = P.py[i];
    if (qx) x = P.x[i];
    if (qy) y = P.y[i];
    if (!bbi_alive(f)) return;
    const int k = bbi_bin(z, P);
    if (k < 0) return;
    const int64_t nbn = (int64_t)P.nb * P.n;
    const double *w = P.kick + (int64_t)b * P.n + k;
    if (P.planes[0]) P.dp[i] = d + w[0];
    if (P.td) {
        // the time domain's order: Z, Dx, Dy, Qx, Qy (src/MPBunch.cpp:2113-2121)
        if (dx) px += w[nbn];
        if (qx) px += w[3 * nbn] * x;
        if (dy) py += w[2 * nbn];
        if (qy) py += w[4 * nbn] * y;
    } else {
        // the frequency domain's: Z, Qx, Qy, then Dx, Dy
        if (qx) px += w[3 * nbn] * x / P.bx;
        if (dx) px += w[nbn];
        if (qy) py += w[4 * nbn] * y / P.by;
        if (dy) py += w[2 * nbn];
    }
    if (dx || qx) P.px[i] = px;
    if (dy || qy) P.py[i] = py;
}

size_t bbi_bin_lds(bool dip)
{
    return (size_t)bbi_count_words(dip) * sizeof(uint32_t) +
           (dip ? (size_t)4 * kBbiDipWin * sizeof(unsigned long long) : 0);
}

hipError_t launch_bbi_bin(const BbiParams &p, int nitem, hipStream_t st)
{
    if (nitem == 0) return hipSuccess;
    const bool dip = p.planes[1] || p.planes[2];
    hipLaunchKernelGGL(k_bbi_bin, dim3(nitem), dim3(kBbiBinBlock), bbi_bin_lds(dip), st, p);
    return hipGetLastError();
}
hipError_t launch_bbi_wake(const BbiParams &p, hipStream_t st)
{
    const bool dip = p.planes[1] || p.planes[2];
    hipLaunchKernelGGL(k_bbi_prof, dim3(p.nb, dip ? 3 : 1), dim3(kBlock), 0, st, p);
    hipLaunchKernelGGL(k_bbi_wake, dim3(p.nb, (p.n + kBlock - 1) / kBlock, 5), dim3(kBlock), 0, st, p);
    return hipGetLastError();
}
hipError_t launch_bbi_kick(const BbiParams &p, int nitem, hipStream_t st)
{
    if (nitem == 0) return hipSuccess;
    hipLaunchKernelGGL(k_bbi_kick, dim3(nitem), dim3(kBlock), 0, st, p);
    return hipGetLastError();
}

}  // namespace cts
