// Kernels of the STFT + Bark stage for any power-of-two FFT length and any hop:
// n_fft = 32 .. 1024, hop >= 1, up to kGenMaxBands bands of a binary,
// contiguous filterbank.  Shared by the stand-alone operator
// (stft_generic.hip) and the pipeline at geometries other than its own
// (pipeline.hip).
//
// Forward, one wavefront per frame: the real frame u (window applied) is
// folded into the half length complex sequence z_n = u_{2n} + i u_{2n+1},
// transformed in float64, unfolded into X_f, f < half, and |X_f|^2 (DC dropped)
// summed per band.  n_fft = 512 runs the radix-4 transform of spectral.hpp,
// n_fft = 1024 three radix-8 passes, eight points per lane (fft512); both hold
// the points in registers and exchange them through LDS between passes, with
// the twiddles staged in LDS once per workgroup of several frames per
// wavefront.  The other lengths run a radix-2 Stockham FFT in LDS (log2(half)
// passes, the pass's butterflies spread over the lanes).
//
// Backward: the same spectrum per frame, V_f = g_P(f) X_f, the adjoint of the
// fold and an inverse FFT give the frame's sample gradient, which is written
// (times the window) to a [rows, frames, n_fft] scratch; a gather kernel then
// adds, for each sample, the contributions of the frames that cover it in
// increasing frame order (deterministic, no atomics, any hop including hops
// longer than n_fft, whose uncovered samples get exactly zero).
//
// Bound by issue (float64) and LDS.  32 rows of 64123 samples at 1024 / 256:
// forward 44 -> 27.5 us, backward frames 78 -> 44, gather 11 -> 8.4 against
// radix-2 passes in LDS for every length; 32 rows of 64000 at 512 / 160, window
// 400: forward 39 -> 25.6, backward frames (16 rows) 63 -> 41.  The radix-2
// variant holds two points per lane and a buffer of 128 (63 and 76 registers,
// eight and six wavefronts per SIMD; with room for 512 points, 168 and 239: three
// and two).  64000 samples, forward and backward with the gather, against one
// frame per wavefront of that size: 32 / 16 over 64 rows 200 + 367 -> 114 + 244,
// 64 / 32 over 64 rows 116 + 217 -> 70 + 151, 128 / 64 over 32 rows 33 + 68 -> 25
// + 54, 256 / 64 over 32 rows 41 + 89 -> 31 + 73.
#pragma once

#include "common.hpp"
#include "pair_scale.hpp"
#include "spectral.hpp"

namespace pesq {

constexpr int kGenMaxHalf = 512;   // n_fft <= 1024
constexpr int kGenMinHalf = 16;    // n_fft >= 32
constexpr int kGenMaxBands = 128;
constexpr int kGenSmallHalf = 128;                     // the radix-2 transform's longest
constexpr int kGenBfly = kGenSmallHalf / 2 / kWave;    // its butterflies per lane
constexpr int kGenWaves = 4;                           // frames per workgroup

struct StftTable {
    int32_t n_fft, half, hop, nbarks;
    double2 tw[kGenMaxHalf];          // e^{-2 pi i m / half}, m < half
    double2 fold[kGenMaxHalf];        // e^{-2 pi i f / n_fft}, f < half
    float window[2 * kGenMaxHalf];    // n_fft taps, centred
    int32_t band_start[kGenMaxBands];
    int32_t band_end[kGenMaxBands];
    int32_t bin_band[kGenMaxHalf];    // band of bin f, -1 for none and for f = 0
    double corr[kGenMaxBands];
};

struct GenArgs {
    const StftTable *tab;
    const float *x;       // [rows, len]
    float *bark;          // [rows, frames, nbarks]
    const float *gbark;   // [rows, frames, nbarks]
    float *gx;            // [rows, len]
    float *scratch;       // [rows, frames, n_fft]
    int64_t rows, len, frames, ftiles;
    int n_fft, half, hop, nbarks;
    int per;              // frames per wavefront
    // the pipeline's (null for the operator): the rows are to be scaled to
    // scale^2 |X|^2, scale from the row's energy partials (forward, which
    // leaves the row constants) or from the row constants (backward, rows of
    // x, bark and gbark in step); the backward's mean band power gradient
    // gmean [items][2][nbarks], added to gbark in the frames that count
    // (keep) where the Bark value exceeds 100 thresholds
    const double *energy;
    const float *peaks;   // [batch, kPairParts]: of the factor that x and energy have (null: 1)
    double *rowconst;     // [rows, 4]: that factor, E, scale, -
    const double *gmean, *threshs;
    const float *keep;    // [items, frames]
    double *spart;        // [rows, nhop]: sums of gx . x per 256 samples
    int64_t nblk, nhop, batch;
    int row0;             // stacked row of row 0
};

using c64g = cplx<double>;

// In place radix-2 Stockham FFT of buf[0 .. half) (natural order in and out),
// e^{-2 pi i / half} forward, conjugate twiddles for the inverse; unnormalised.
// Pass s (sub-transform size ns = 2^s): butterfly j takes buf[j] and
// buf[j + half / 2], k = j mod ns, w = e^{-2 pi i k / (2 ns)}, and writes
// positions (j / ns) 2 ns + k and that plus ns.  Every lane reads all of its
// butterflies' inputs before the wave's writes start.
template <bool kInv>
__device__ __forceinline__ void gen_fft(c64g *buf, const double2 *tw, int half, int lane) {
    const int nb = half / 2;
    for (int ns = 1; ns < half; ns *= 2) {
        c64g a[kGenBfly], b[kGenBfly];
#pragma unroll
        for (int q = 0; q < kGenBfly; ++q) {
            const int j = lane + kWave * q;
            if (j < nb) {
                a[q] = buf[j];
                b[q] = buf[j + nb];
            }
        }
        wave_lds_fence();
#pragma unroll
        for (int q = 0; q < kGenBfly; ++q) {
            const int j = lane + kWave * q;
            if (j < nb) {
                const int k = j & (ns - 1);
                const double2 w = tw[k * (nb / ns)];
                const c64g v = cmul(b[q], c64g{w.x, kInv ? -w.y : w.y});
                const int o = (j / ns) * 2 * ns + k;
                buf[o] = {a[q].re + v.re, a[q].im + v.im};
                buf[o + ns] = {a[q].re - v.re, a[q].im - v.im};
            }
        }
        wave_lds_fence();
    }
}

// --------------------------------------------------------------------------
// half = 512: radix-8 passes, lane l holding points l + 64 r
// --------------------------------------------------------------------------

// LDS slot of element i: one element of padding per 8, so that the writes of a
// pass (8 elements apart) and the unit stride reads fall on distinct banks
__device__ __forceinline__ int slot8(int i) { return i + (i >> 3); }
constexpr int kSlots512 = kGenMaxHalf + kGenMaxHalf / 8;

// radix-8 DFT, e^{-2 pi i / 8} forward
template <bool kInv>
__device__ __forceinline__ void dft8(c64g (&v)[8]) {
#pragma clang fp contract(off)
    constexpr double h = 0.70710678118654752440;
    c64g a[4] = {v[0], v[2], v[4], v[6]}, b[4] = {v[1], v[3], v[5], v[7]};
    dft4<double, kInv>(a);
    dft4<double, kInv>(b);
    // b[k] times e^{-+2 pi i k / 8}
    const c64g b1 = kInv ? c64g{h * (b[1].re - b[1].im), h * (b[1].re + b[1].im)}
                         : c64g{h * (b[1].re + b[1].im), h * (b[1].im - b[1].re)};
    const c64g b2 = kInv ? c64g{-b[2].im, b[2].re} : c64g{b[2].im, -b[2].re};
    const c64g b3 = kInv ? c64g{-h * (b[3].re + b[3].im), h * (b[3].re - b[3].im)}
                         : c64g{h * (b[3].im - b[3].re), -h * (b[3].re + b[3].im)};
    const c64g w[4] = {b[0], b1, b2, b3};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        v[k] = {a[k].re + w[k].re, a[k].im + w[k].im};
        v[k + 4] = {a[k].re - w[k].re, a[k].im - w[k].im};
    }
}

// v[r] = z_{lane + 64 r} to Z_{lane + 64 r}; tw = e^{-2 pi i m / 512} in LDS
template <bool kInv>
__device__ __forceinline__ void fft512(c64g (&v)[8], c64g *buf, const double2 *tw, int lane) {
#pragma unroll
    for (int pass = 0; pass < 3; ++pass) {
        const int ns = 1 << (3 * pass);
        const int k = lane & (ns - 1);
        if (pass > 0) {
#pragma unroll
            for (int r = 0; r < 8; ++r) v[r] = buf[slot8(lane + 64 * r)];
            wave_lds_fence();
#pragma unroll
            for (int r = 1; r < 8; ++r) {
                const double2 w = tw[k * r * (64 / ns)];
                v[r] = cmul(v[r], c64g{w.x, kInv ? -w.y : w.y});
            }
        }
        dft8<kInv>(v);
        if (pass == 2) break;
        const int base = (lane / ns) * ns * 8 + k;
#pragma unroll
        for (int r = 0; r < 8; ++r) buf[slot8(base + r * ns)] = v[r];
        wave_lds_fence();
    }
}

// --------------------------------------------------------------------------
// the transforms by half length: kHalf 256, 512, or 0 for any up to 128
// --------------------------------------------------------------------------
template <int kH>
struct GenFft {
    static constexpr int kPoints = (kH == 0 ? kGenSmallHalf : kH) / kWave;  // per lane
    static constexpr int kBuffer = kH == 0 ? kGenSmallHalf : (kH == 512 ? kSlots512 : kH);
    // twiddles staged in LDS: the pass twiddles (256: per pass layout), the fold's
    static constexpr int kTw = kH == 512 ? 512 : (kH == 256 ? kPassTwiddles : 1);
    static constexpr int kFold = kH == 0 ? 1 : kH;

    static __device__ __forceinline__ void stage(const StftTable &t, double2 *tw, double2 *fold) {
        if constexpr (kH != 0) {
            for (int i = threadIdx.x; i < kH; i += kWave * kGenWaves) {
                if constexpr (kH == 512) {
                    tw[i] = t.tw[i];
                } else {
                    if (i < kPassTwiddles) tw[i] = pass_twiddle_entry(t.tw, i);
                }
                fold[i] = t.fold[i];
            }
            __syncthreads();
        }
    }

    // X_f of the windowed samples in pairs u[r] = (u_{2n}, u_{2n+1}), n = lane + 64 r
    static __device__ __forceinline__ void spectrum(const StftTable &t, c64g (&u)[kPoints],
                                                    c64g *buf, const double2 *tw,
                                                    const double2 *fold, int half, int lane,
                                                    c64g (&x)[kPoints]) {
        if constexpr (kH == 256) {
            const LdsTwiddles<double> lt{tw, fold, lane};
            auto load = [&](int k) -> double {
                return (k & 1) ? u[k >> 7].im : u[k >> 7].re;
            };
            frame_spectrum<double>(load, x, buf, lt, lane);
        } else if constexpr (kH == 512) {
            fft512<false>(u, buf, tw, lane);
            wave_lds_fence();
#pragma unroll
            for (int r = 0; r < kPoints; ++r) buf[slot8(lane + 64 * r)] = u[r];
            wave_lds_fence();
#pragma unroll
            for (int r = 0; r < kPoints; ++r) {
                const int f = lane + 64 * r;
                x[r] = unfold(u[r], buf[slot8((kH - f) & (kH - 1))], fold[f]);
            }
            wave_lds_fence();
        } else {
#pragma unroll
            for (int r = 0; r < kPoints; ++r) {
                if (lane + kWave * r < half) buf[lane + kWave * r] = u[r];
            }
            wave_lds_fence();
            gen_fft<false>(buf, t.tw, half, lane);
#pragma unroll
            for (int r = 0; r < kPoints; ++r) {
                const int f = lane + kWave * r;
                if (f < half) x[r] = unfold(buf[f], buf[(half - f) & (half - 1)], t.fold[f]);
            }
            wave_lds_fence();
        }
    }
    static __device__ __forceinline__ c64g unfold(c64g zf, c64g zm, double2 c) {
        const c64g e = {(zf.re + zm.re) * 0.5, (zf.im - zm.im) * 0.5};
        const c64g o = {(zf.im + zm.im) * 0.5, -(zf.re - zm.re) * 0.5};
        const c64g v = cmul(c64g{c.x, c.y}, o);
        return {e.re + v.re, e.im + v.im};
    }

    // Z'_f = (V_f + conj V_{half-f}) + i e^{+2 pi i f / n} (V_f - conj V_{half-f}), V_half = 0
    static __device__ __forceinline__ c64g refold(c64g va, c64g vb, double2 c) {
        const c64g s = {va.re + vb.re, va.im - vb.im};
        const c64g d = {va.re - vb.re, va.im + vb.im};
        const c64g v = cmul(c64g{c.x, -c.y}, d);
        return {s.re - v.im, s.im + v.re};
    }
    // the adjoint: V_f, f = lane + 64 r (zero at f = 0), to the sample pairs z_n
    static __device__ __forceinline__ void adjoint(const StftTable &t, c64g (&v)[kPoints],
                                                   c64g *buf, const double2 *tw,
                                                   const double2 *fold, int half, int lane,
                                                   c64g (&z)[kPoints]) {
        if constexpr (kH == 256) {
            const LdsTwiddles<double> lt{tw, fold, lane};
            double ev[kPoints], od[kPoints];
            frame_adjoint<double>(v, ev, od, buf, lt, lane);
#pragma unroll
            for (int r = 0; r < kPoints; ++r) z[r] = {ev[r], od[r]};
        } else if constexpr (kH == 512) {
#pragma unroll
            for (int r = 0; r < kPoints; ++r) buf[slot8(lane + 64 * r)] = v[r];
            wave_lds_fence();
#pragma unroll
            for (int r = 0; r < kPoints; ++r) {
                const int f = lane + 64 * r;
                const c64g vb = f == 0 ? c64g{0.0, 0.0} : buf[slot8(f == 0 ? 0 : kH - f)];
                z[r] = refold(v[r], vb, fold[f]);
            }
            wave_lds_fence();
            fft512<true>(z, buf, tw, lane);
            wave_lds_fence();
        } else {
#pragma unroll
            for (int r = 0; r < kPoints; ++r) {
                if (lane + kWave * r < half) buf[lane + kWave * r] = v[r];
            }
            wave_lds_fence();
#pragma unroll
            for (int r = 0; r < kPoints; ++r) {
                const int f = lane + kWave * r;
                if (f < half) {
                    const c64g vb = f == 0 ? c64g{0.0, 0.0} : buf[half - f];
                    z[r] = refold(v[r], vb, t.fold[f]);
                }
            }
            wave_lds_fence();
#pragma unroll
            for (int r = 0; r < kPoints; ++r) {
                if (lane + kWave * r < half) buf[lane + kWave * r] = z[r];
            }
            wave_lds_fence();
            gen_fft<true>(buf, t.tw, half, lane);
#pragma unroll
            for (int r = 0; r < kPoints; ++r) {
                if (lane + kWave * r < half) z[r] = buf[lane + kWave * r];
            }
            wave_lds_fence();
        }
    }
};

// The frame's raw sample pairs x[start + 2 n], x[start + 2 n + 1], n = lane +
// 64 r < half (zero past len): 8-byte loads where the frame lies in the row.
template <int kPoints>
__device__ __forceinline__ void gen_load(const float *x, int64_t start, int64_t len, int half,
                                         int lane, float (&s)[2 * kPoints]) {
    if (start + 2 * half <= len) {
#pragma unroll
        for (int r = 0; r < kPoints; ++r) {
            const int n = lane + kWave * r;
            __builtin_memcpy(&s[2 * r], x + start + 2 * (n < half ? n : half - 1), 8);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 2 * kPoints; ++i) {
            const int n = lane + kWave * (i / 2);
            s[i] = load_or_zero(x, start + 2 * (n < half ? n : half - 1) + i % 2, len);
        }
    }
}

// sum of power[lo .. hi) in ascending order, eight reads in flight
__device__ __forceinline__ double gen_band_sum(const double *power, int lo, int hi) {
    double acc = 0.0;
    for (int f = lo; f < hi; f += 8) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = power[f + u < hi ? f + u : hi - 1];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (f + u < hi) acc += v[u];
        }
    }
    return acc;
}

// this wavefront's frames first .. first + count - 1 of a row
__device__ __forceinline__ int gen_frames(const GenArgs &a, int64_t &row, int64_t &first) {
    row = blockIdx.x / a.ftiles;
    const int64_t tile = blockIdx.x - row * a.ftiles;
    first = (tile * kGenWaves + wave_index()) * a.per;
    const int64_t left = a.frames - first;
    return left <= 0 ? 0 : static_cast<int>(left < a.per ? left : a.per);
}

// the energy of a row from its blocks' partials (a whole wavefront's call)
__device__ __forceinline__ double gen_energy(const GenArgs &a, int64_t row, int lane) {
    const int mine = lane < a.nblk ? static_cast<int>((a.nblk - 1 - lane) / kWave + 1) : 0;
    return wave_sum(mine > 0 ? strided_sum(a.energy + row * a.nblk + lane, mine, kWave) : 0.0);
}

template <int kH>
__global__ void __launch_bounds__(kWave *kGenWaves) stft_gen_fwd_kernel(GenArgs a) {
    using F = GenFft<kH>;
    constexpr int P = F::kPoints;
    __shared__ c64g bufs[kGenWaves][F::kBuffer];
    __shared__ double2 tw[F::kTw], fold[F::kFold];
    const StftTable &t = *a.tab;
    const int lane = static_cast<int>(threadIdx.x) % kWave;
    int64_t row, first;
    const int count = gen_frames(a, row, first);
    const float *x = a.x + row * a.len;
    const int half = kH == 0 ? a.half : kH;
    float raw[2 * P];
    if (count > 0) gen_load<P>(x, first * a.hop, a.len, half, lane, raw);
    F::stage(t, tw, fold);
    if (count == 0) return;  // whole wavefronts; no barrier follows
    double scale2 = 1.0;
    if (a.energy != nullptr) {
        const double e = gen_energy(a, row, lane);
        const double power = e / static_cast<double>(a.len + 5120) / 1.04684;
        const double scale = sqrt(1e7 / power);
        scale2 = scale * scale;
        if (first == 0) {  // uniform
            const int64_t pair = row < a.batch ? row : row - a.batch;
            const double factor = a.peaks != nullptr ? pair_factor(a.peaks, pair, lane) : 1.0;
            if (lane == 0) {
                double *rc = a.rowconst + row * 4;
                rc[0] = factor;
                rc[1] = e;
                rc[2] = scale;
                rc[3] = 0.0;
            }
        }
    }
    c64g *buf = bufs[wave_index()];
    double *power = reinterpret_cast<double *>(buf);
    for (int q = 0; q < count; ++q) {
        const int64_t frame = first + q;
        c64g u[P], spec[P];
#pragma unroll
        for (int r = 0; r < P; ++r) {
            const int n = lane + kWave * r;
            float2 w = make_float2(0.0f, 0.0f);
            if (n < half) w = *reinterpret_cast<const float2 *>(t.window + 2 * n);
            u[r] = {static_cast<double>(raw[2 * r]) * static_cast<double>(w.x),
                    static_cast<double>(raw[2 * r + 1]) * static_cast<double>(w.y)};
        }
        // the next frame's samples load while this one is transformed
        if (q + 1 < count) gen_load<P>(x, (frame + 1) * a.hop, a.len, half, lane, raw);
        F::spectrum(t, u, buf, tw, fold, half, lane, spec);
#pragma unroll
        for (int r = 0; r < P; ++r) {
            const int f = lane + kWave * r;
            if (f < half) {
                const double v = f == 0 ? 0.0 : spec[r].re * spec[r].re + spec[r].im * spec[r].im;
                power[f] = v * scale2;
            }
        }
        wave_lds_fence();
        float *out = a.bark + (row * a.frames + frame) * a.nbarks;
        for (int b = lane; b < a.nbarks; b += kWave) {
            out[b] = static_cast<float>(gen_band_sum(power, t.band_start[b], t.band_end[b]) * t.corr[b]);
        }
        wave_lds_fence();
    }
}

// per frame: the frame's windowed sample gradient into the scratch
template <int kH>
__global__ void __launch_bounds__(kWave *kGenWaves) stft_gen_bwd_frames_kernel(GenArgs a) {
    using F = GenFft<kH>;
    constexpr int P = F::kPoints;
    __shared__ c64g bufs[kGenWaves][F::kBuffer];
    __shared__ double2 tw[F::kTw], fold[F::kFold];
    __shared__ float gbands[kGenWaves][kGenMaxBands];
    const StftTable &t = *a.tab;
    const int lane = static_cast<int>(threadIdx.x) % kWave;
    int64_t row, first;
    const int count = gen_frames(a, row, first);
    const float *x = a.x + row * a.len;
    const int half = kH == 0 ? a.half : kH;
    float raw[2 * P];
    if (count > 0) gen_load<P>(x, first * a.hop, a.len, half, lane, raw);
    F::stage(t, tw, fold);
    if (count == 0) return;
    const int stacked = a.row0 + static_cast<int>(row);
    const int item = a.batch > 0 ? stacked % static_cast<int>(a.batch) : 0;
    const double scale = a.rowconst != nullptr ? a.rowconst[row * 4 + 2] : 1.0;
    c64g *buf = bufs[wave_index()];
    float *gband = gbands[wave_index()];
    for (int q = 0; q < count; ++q) {
        const int64_t frame = first + q;
        for (int b = lane; b < a.nbarks; b += kWave) {
            const int64_t at = (row * a.frames + frame) * a.nbarks + b;
            double g = static_cast<double>(a.gbark[at]);
            if (a.gmean != nullptr && a.keep[item * a.frames + frame] != 0.0f &&
                static_cast<double>(a.bark[at]) > 100.0 * a.threshs[b]) {
                // (rounded to float32 between the two sums, as gbark is)
                const double mean = a.gmean[(int64_t(item) * 2 + (stacked < a.batch ? 0 : 1)) * a.nbarks + b];
                g = static_cast<double>(static_cast<float>(g + mean));
            }
            gband[b] = static_cast<float>(g * t.corr[b]);
        }
        c64g u[P], v[P];
#pragma unroll
        for (int r = 0; r < P; ++r) {
            const int n = lane + kWave * r;
            float2 w = make_float2(0.0f, 0.0f);
            if (n < half) w = *reinterpret_cast<const float2 *>(t.window + 2 * n);
            u[r] = {static_cast<double>(raw[2 * r]) * static_cast<double>(w.x),
                    static_cast<double>(raw[2 * r + 1]) * static_cast<double>(w.y)};
        }
        if (q + 1 < count) gen_load<P>(x, (frame + 1) * a.hop, a.len, half, lane, raw);
        F::spectrum(t, u, buf, tw, fold, half, lane, v);
        // V_f = g_P(f) X_f (zero at DC and outside the bands)
#pragma unroll
        for (int r = 0; r < P; ++r) {
            const int f = lane + kWave * r;
            if (f < half) {
                const int band = t.bin_band[f];
                const double gp = band >= 0 ? static_cast<double>(gband[band]) * scale : 0.0;
                v[r] = {gp * v[r].re, gp * v[r].im};
            }
        }
        wave_lds_fence();
        c64g z[P];
        F::adjoint(t, v, buf, tw, fold, half, lane, z);
        float *dst = a.scratch + (row * a.frames + frame) * a.n_fft;
#pragma unroll
        for (int r = 0; r < P; ++r) {
            const int n = lane + kWave * r;
            if (n < half) {
                const float2 w = *reinterpret_cast<const float2 *>(t.window + 2 * n);
                *reinterpret_cast<float2 *>(dst + 2 * n) =
                    make_float2(static_cast<float>(z[r].re * static_cast<double>(w.x)),
                                static_cast<float>(z[r].im * static_cast<double>(w.y)));
            }
        }
    }
}

constexpr int kGatherThreads = 256;
constexpr int kGatherPer = 4;  // consecutive samples per thread
constexpr int kGatherSpan = kGatherThreads * kGatherPer;

// per sample: sum of the contributions of the frames covering it, in
// increasing frame order; in the pipeline also the sum of gx . x over every
// 256 samples (a wavefront's).  Int: int where sample indices fit, else int64_t.
template <typename Int>
__global__ void __launch_bounds__(kGatherThreads) stft_gen_bwd_gather_kernel(GenArgs a) {
    const int64_t nblk = cdiv(a.len, kGatherSpan);
    const int64_t row = blockIdx.x / nblk;
    const Int n0 = static_cast<Int>((blockIdx.x - row * nblk) * kGatherSpan) +
                   kGatherPer * static_cast<Int>(threadIdx.x);
    const Int len = static_cast<Int>(a.len), frames = static_cast<Int>(a.frames);
    double g[kGatherPer] = {};
    if (n0 < len) {
        // frames t with t hop <= n < t hop + n_fft, t < frames, for n = n0 .. n0 + 3
        Int t = n0 < a.n_fft ? 0 : (n0 - a.n_fft) / a.hop + 1;
        const Int last = (n0 + kGatherPer - 1) / a.hop;
        const Int t_hi = last < frames - 1 ? last : frames - 1;
        const float *src = a.scratch + row * a.frames * a.n_fft;
        for (; t <= t_hi; ++t) {
            const Int k = n0 - t * a.hop;  // -3 .. n_fft - 1
            const float *frame = src + int64_t(t) * a.n_fft;
            float v[kGatherPer];
            if (k >= 0 && k + kGatherPer <= a.n_fft) {
                __builtin_memcpy(v, frame + k, sizeof(v));
            } else {
#pragma unroll
                for (int e = 0; e < kGatherPer; ++e) {
                    const Int i = k + e;
                    const float w = frame[i < 0 ? 0 : (i < a.n_fft ? i : a.n_fft - 1)];
                    v[e] = i >= 0 && i < a.n_fft ? w : 0.0f;
                }
            }
#pragma unroll
            for (int e = 0; e < kGatherPer; ++e) g[e] += static_cast<double>(v[e]);
        }
    }
    float *out = a.gx + row * a.len;
    const float *x = a.spart != nullptr ? a.x + row * a.len : nullptr;
    double acc = 0.0;
#pragma unroll
    for (int e = 0; e < kGatherPer; ++e) {
        if (n0 + e < len) {
            out[n0 + e] = static_cast<float>(g[e]);
            if (x != nullptr) acc = fma(g[e], static_cast<double>(x[n0 + e]), acc);
        }
    }
    if (a.spart != nullptr) {
        acc = wave_sum(acc);
        const int64_t hop = (blockIdx.x - row * nblk) * (kGatherThreads / kWave) + wave_index();
        if (threadIdx.x % kWave == 0 && hop < a.nhop) a.spart[row * a.nhop + hop] = acc;
    }
}

// frames per wavefront: more where the grid has wavefronts to spare (the
// staged tables and the next frame's loads are shared)
inline int gen_per(int64_t rows, int64_t frames) {
    const int64_t waves = rows * frames / (3 * 4 * 256);
    return static_cast<int>(waves < 1 ? 1 : (waves > 4 ? 4 : waves));
}

inline void launch_gen_fwd(GenArgs a, hipStream_t stream) {
    a.per = gen_per(a.rows, a.frames);
    a.ftiles = cdiv(a.frames, int64_t(kGenWaves) * a.per);
    const dim3 grid(static_cast<unsigned>(a.rows * a.ftiles)), block(kWave * kGenWaves);
    if (a.half == 256) {
        hipLaunchKernelGGL(stft_gen_fwd_kernel<256>, grid, block, 0, stream, a);
    } else if (a.half == 512) {
        hipLaunchKernelGGL(stft_gen_fwd_kernel<512>, grid, block, 0, stream, a);
    } else {
        hipLaunchKernelGGL(stft_gen_fwd_kernel<0>, grid, block, 0, stream, a);
    }
}

inline void launch_gen_bwd(GenArgs a, hipStream_t stream) {
    a.per = gen_per(a.rows, a.frames);
    a.ftiles = cdiv(a.frames, int64_t(kGenWaves) * a.per);
    const dim3 grid(static_cast<unsigned>(a.rows * a.ftiles)), block(kWave * kGenWaves);
    if (a.half == 256) {
        hipLaunchKernelGGL(stft_gen_bwd_frames_kernel<256>, grid, block, 0, stream, a);
    } else if (a.half == 512) {
        hipLaunchKernelGGL(stft_gen_bwd_frames_kernel<512>, grid, block, 0, stream, a);
    } else {
        hipLaunchKernelGGL(stft_gen_bwd_frames_kernel<0>, grid, block, 0, stream, a);
    }
    const dim3 spans(static_cast<unsigned>(a.rows * cdiv(a.len, kGatherSpan)));
    if (a.len + 2 * a.n_fft + a.hop < (int64_t(1) << 31)) {
        hipLaunchKernelGGL(stft_gen_bwd_gather_kernel<int>, spans, dim3(kGatherThreads), 0, stream, a);
    } else {
        hipLaunchKernelGGL(stft_gen_bwd_gather_kernel<int64_t>, spans, dim3(kGatherThreads), 0,
                           stream, a);
    }
}

}  // namespace pesq
