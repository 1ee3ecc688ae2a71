// preprocess.h - shared pieces of the host (preprocess.cpp) and device (preprocess.hip) preprocessing.
#pragma once
#include "../../include/jepa.h"

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <vector>

// a shortest-edge resize whose intermediate would exceed this many pixels is refused (the aspect
// ratio, not the file size, makes it large; reference src/preprocess.cpp:195-200)
#define JEPA_PRE_MAX_PIXELS (64ll * 1024 * 1024)

// One axis of a separable uint8 resize, as a compressed-row table: output o reads the inputs
// lo[o], lo[o] + 1, ... with the integer taps taps[beg[o]] .. taps[beg[o + 1] - 1], accumulates
// 2^(shift-1) + sum(tap * pixel) in int32 and keeps clamp(acc >> shift, 0, 255). The rows have
// their own lengths (no padding), and the same arrays are uploaded for the device passes.
struct resample_axis {
    int n_in = 0, n_out = 0, shift = 0;
    std::vector<int32_t> lo;      // [n_out]
    std::vector<int32_t> beg;     // [n_out + 1]
    std::vector<int16_t> taps;    // [beg[n_out]]
    bool identity() const { return n_in == n_out; }
};
resample_axis resample_axis_for(int n_in, int n_out, int resample);

// The filter of one axis and the window and weights of one output, for the host tables and for the
// kernel that makes the taps of its own tile (the same doubles on both: plain IEEE operations, built
// without contraction).
struct axis_filter {
    double scale, reach, step;    // input pixels per output; half width of the window; 1 / stretch
    int n_in, n_out, cubic;
    // at most this many inputs reach one output
    int max_taps() const { return (int) std::ceil(2.0 * reach) + 1; }
};
inline axis_filter axis_filter_for(int n_in, int n_out, int resample) {
    axis_filter f;
    f.n_in = n_in; f.n_out = n_out;
    f.cubic = resample == JEPA_RESAMPLE_BICUBIC ? 1 : 0;
    f.scale = (double) n_in / (double) n_out;
    const double stretch = f.scale > 1.0 ? f.scale : 1.0;   // the filter widens only when shrinking
    f.reach = (f.cubic ? 2.0 : 1.0) * stretch;
    f.step = 1.0 / stretch;
    return f;
}
// inputs [first, end) of output o: those whose window rounds into [centre - reach, centre + reach), clipped
// to the image (in double before the conversion, so that a very wide input cannot push it past INT_MAX)
__host__ __device__ inline double axis_window(const axis_filter & f, int o, int & first, int & end) {
    const double centre = f.scale * (o + 0.5), a = centre - f.reach + 0.5, b = centre + f.reach + 0.5;
    first = (int) (0.0 < a ? a : 0.0);
    end = (int) (b < (double) f.n_in ? b : (double) f.n_in);
    return centre;
}
// The two antialias filters at distance x: triangle; Keys (1981) cubic convolution, a = -0.5, in the
// nested form torch evaluates (the weights must be the same doubles for the int16 rounding to agree):
// inner piece ((a+2)|x| - (a+3))|x|^2 + 1, outer piece ((a|x| - 5a)|x| + 8a)|x| - 4a
__host__ __device__ inline double axis_weight(const axis_filter & f, int x, double centre) {
    const double d = fabs((x - centre + 0.5) * f.step);
    if (!f.cubic) return d < 1.0 ? 1.0 - d : 0.0;
    constexpr double a = -0.5;
    if (d >= 2.0) return 0.0;
    if (d >= 1.0) return ((a * d - 5.0 * a) * d + 8.0 * a) * d - 4.0 * a;
    return ((a + 2.0) * d - (a + 3.0)) * d * d + 1.0;
}
// round half away from zero the way the method writes it, (int)(0.5 + |v|) with the sign put back
__host__ __device__ inline int16_t round_tap(double v) {
    const int mag = (int) (0.5 + fabs(v));
    return (int16_t) (v < 0.0 ? -mag : mag);
}
// the tables' shift: the first s in 0..21 whose next step would round the peak weight to 2^15 or more, else 22
int axis_shift_of_peak(double peak);
// the same without the tables (one division per output: a quotient by one total grows with its numerator)
int axis_shift(const axis_filter & f);

// geometry and normalisation of one preprocessing call
struct pre_plan {
    int rh = 0, rw = 0;        // resized size
    int crop = 0;              // output is crop x crop
    int oy = 0, ox = 0;        // crop pixel (y, x) = resized pixel (y + oy, x + ox), zero outside
    float inv = 255.0f;        // 1 / rescale
    bool fused = true;
    float mean[3] = {0, 0, 0}, stdv[3] = {1, 1, 1};   // fused: mean / rescale and std / rescale
};
bool pre_plan_for(const jepa_preprocess_params * p, int h, int w, pre_plan & g);

// normalised value of channel c of a uint8 pixel (the reference's two formulas, src/preprocess.cpp:283-287)
__host__ __device__ inline float pre_normalize_v(bool fused, float inv, float mean, float stdv, uint8_t v) {
    return fused ? ((float) v - mean) / stdv : ((float) v / inv - mean) / stdv;
}
inline float pre_normalize(const pre_plan & g, int c, uint8_t v) { return pre_normalize_v(g.fused, g.inv, g.mean[c], g.stdv[c], v); }

// device: n_frames HWC uint8 frames [n][h][w][3] (device memory) -> NCTHW floats [3][n][crop][crop]
// (device memory), equal bit for bit to jepa_preprocess_frames_rgb_ex. Where preprocess_tiled() says so
// one kernel does both passes and needs no scratch (nullptr); elsewhere tables are built on the host
// and uploaded into `scratch` (preprocess_scratch_bytes). Returns false on a bad geometry.
bool preprocess_tiled(const jepa_preprocess_params * p, const pre_plan & g, int n_frames, int h, int w);
// at least preprocess_scratch_bytes, without building the tables
size_t preprocess_scratch_bound(const jepa_preprocess_params * p, const pre_plan & g, int n_frames, int h, int w);
size_t preprocess_scratch_bytes(const jepa_preprocess_params * p, const pre_plan & g, int n_frames, int h, int w);
bool launch_preprocess(const jepa_preprocess_params * p, const pre_plan & g, const uint8_t * frames, int n_frames, int h, int w,
                       float * out, void * scratch, hipStream_t s);

// The allocation-free variant's scratch: a static device array of this size on every GPU the library
// runs on (tap tables + the horizontal-pass image of all frames), and its device address on
// `device` (looked up once per device with that device current; nullptr on failure).
#define PRE_NOALLOC_SCRATCH_BYTES ((size_t) 32 << 20)
void * preprocess_static_scratch(int device);
