// Stand-alone STFT + Bark operator for any power-of-two FFT length and any
// hop (the general TritonStftBark, torch_pesq/triton_ops/spectral.py:584-774):
// table packing, argument checks and launches of the kernels of
// stft_generic.hpp.  The PESQ geometry (512 / 256 / 49 bands) has its own fused
// and stand-alone kernels; this file serves every other configuration.
#include <cmath>
#include <cstring>

#include "stft_generic.hpp"

namespace pesq {

static int check_geometry(int64_t rows, int64_t len, int64_t n_padded, int n_fft, int hop,
                          int nbarks, int64_t &frames) {
    PESQ_CHECK_ARG(rows >= 0 && len >= 0, "invalid sizes");
    PESQ_CHECK_ARG(n_fft >= 2 * kGenMinHalf && n_fft <= 2 * kGenMaxHalf && (n_fft & (n_fft - 1)) == 0,
                   "n_fft has to be a power of two in [%d, %d], got %d", 2 * kGenMinHalf,
                   2 * kGenMaxHalf, n_fft);
    PESQ_CHECK_ARG(hop >= 1, "hop_length has to be positive, got %d", hop);
    PESQ_CHECK_ARG(nbarks >= 1 && nbarks <= kGenMaxBands, "1..%d bands, got %d", kGenMaxBands,
                   nbarks);
    PESQ_CHECK_ARG(n_padded >= len && n_padded >= n_fft,
                   "n_padded (%lld) has to cover the signal (%lld) and one frame (%d)",
                   (long long)n_padded, (long long)len, n_fft);
    frames = 1 + (n_padded - n_fft) / hop;
    PESQ_CHECK_ARG(rows * cdiv(frames, kGenWaves) < (int64_t(1) << 31) &&
                       rows * cdiv(len, kGatherThreads) < (int64_t(1) << 31),
                   "problem too large for one launch");
    return PESQ_OK;
}

}  // namespace pesq

using namespace pesq;

extern "C" size_t pesq_stft_table_bytes(void) { return sizeof(StftTable); }

extern "C" int pesq_stft_table_pack(int n_fft, int hop, const float *window, int nbarks,
                                    const int32_t *band_start, const int32_t *band_end,
                                    const double *corr, void *out) {
    PESQ_CHECK_ARG(window && band_start && band_end && corr && out, "null argument");
    int64_t frames = 0;
    if (int st = check_geometry(0, 0, n_fft, n_fft, hop, nbarks, frames)) return st;
    StftTable *t = new StftTable;
    std::memset(t, 0, sizeof(*t));
    const int half = n_fft / 2;
    t->n_fft = n_fft;
    t->half = half;
    t->hop = hop;
    t->nbarks = nbarks;
    const double two_pi = 6.283185307179586476925286766559;
    for (int m = 0; m < half; ++m) {
        t->tw[m] = make_double2(std::cos(two_pi * m / half), -std::sin(two_pi * m / half));
    }
    for (int f = 0; f < half; ++f) {
        t->fold[f] = make_double2(std::cos(two_pi * f / n_fft), -std::sin(two_pi * f / n_fft));
        t->bin_band[f] = -1;
    }
    std::memcpy(t->window, window, sizeof(float) * n_fft);
    int prev = 0;
    for (int b = 0; b < nbarks; ++b) {
        const int lo = band_start[b], hi = band_end[b];
        if (lo < prev || hi < lo || hi > half) {
            delete t;
            set_error("Bark band %d covers [%d, %d): bands must be sorted, disjoint and inside "
                      "[0, %d)", b, lo, hi, half);
            return PESQ_ERR_ARGUMENT;
        }
        t->band_start[b] = lo;
        t->band_end[b] = hi;
        t->corr[b] = corr[b];
        for (int f = lo; f < hi; ++f) t->bin_band[f] = b;
        prev = hi;
    }
    t->bin_band[0] = -1;  // the DC bin is dropped
    std::memcpy(out, t, sizeof(*t));
    delete t;
    return PESQ_OK;
}

extern "C" int pesq_stft_workspace(int64_t rows, int64_t len, int64_t n_padded, int n_fft,
                                   int hop, size_t *bytes) {
    PESQ_CHECK_ARG(bytes != nullptr, "null argument");
    int64_t frames = 0;
    if (int st = check_geometry(rows, len, n_padded, n_fft, hop, 1, frames)) return st;
    *bytes = size_t(rows) * size_t(frames) * size_t(n_fft) * sizeof(float);
    return PESQ_OK;
}

extern "C" int pesq_stft_forward(const float *x, int64_t rows, int64_t len, int64_t n_padded,
                                 const void *table, int n_fft, int hop, int nbarks, float *bark,
                                 hipStream_t stream) {
    PESQ_CHECK_ARG(x && table && bark, "null pointer argument");
    GenArgs a{};
    int64_t frames = 0;
    if (int st = check_geometry(rows, len, n_padded, n_fft, hop, nbarks, frames)) return st;
    if (rows == 0) return PESQ_OK;
    PESQ_CHECK_ARG(len > 0, "empty signal with frames to fill");
    a.tab = static_cast<const StftTable *>(table);
    a.x = x;
    a.bark = bark;
    a.rows = rows;
    a.len = len;
    a.frames = frames;
    a.n_fft = n_fft;
    a.half = n_fft / 2;
    a.hop = hop;
    a.nbarks = nbarks;
    launch_gen_fwd(a, stream);
    PESQ_CHECK_LAUNCH("stft forward");
    return PESQ_OK;
}

extern "C" int pesq_stft_backward(const float *gbark, const float *x, int64_t rows, int64_t len,
                                  int64_t n_padded, const void *table, int n_fft, int hop,
                                  int nbarks, float *gx, void *workspace, hipStream_t stream) {
    PESQ_CHECK_ARG(gbark && x && table && gx && workspace, "null pointer argument");
    GenArgs a{};
    int64_t frames = 0;
    if (int st = check_geometry(rows, len, n_padded, n_fft, hop, nbarks, frames)) return st;
    if (rows == 0 || len == 0) return PESQ_OK;
    a.tab = static_cast<const StftTable *>(table);
    a.x = x;
    a.gbark = gbark;
    a.gx = gx;
    a.scratch = static_cast<float *>(workspace);
    a.rows = rows;
    a.len = len;
    a.frames = frames;
    a.n_fft = n_fft;
    a.half = n_fft / 2;
    a.hop = hop;
    a.nbarks = nbarks;
    launch_gen_bwd(a, stream);
    PESQ_CHECK_LAUNCH("stft backward");
    return PESQ_OK;
}
