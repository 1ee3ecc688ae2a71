// preprocess.hip - uint8 antialiased resize + centre crop + normalisation on the device, equal bit for
// bit to the host jepa_preprocess_frames_rgb_ex (preprocess.cpp; reference src/preprocess.cpp).
//
// k_resize_tile does both passes of one output tile and keeps the uint8 image between them in LDS; every
// workgroup makes the taps of its own columns and rows from the host's own double arithmetic. Only
// the tables' shift, which depends on every output, comes from the host.
//
// Tiles that need more LDS than that (reductions of more than about twelve times) take the two kernels
// of the separable order: the horizontal pass writes only the resized columns the crop keeps, as uint8
// (the host rounds to uint8 between the passes too); the vertical pass computes the crop's pixels,
// applies the zero padding of an undersized image and writes the normalised floats in NCTHW order.
// Their tables are built on the host and uploaded once per call.
#include "preprocess.h"
#include "common.h"
#include "lds_dma.h"

#include <algorithm>
#include <cstring>
#include <mutex>

namespace {

// one resample_axis on the device: output o reads inputs lo[o] + t - beg[o] with taps[t],
// beg[o] <= t < beg[o + 1]
struct dev_axis {
    const int32_t * lo;
    const int32_t * beg;
    const int16_t * taps;
    int shift;
    int identity;   // size unchanged: the host skips this pass (a copy)
};

__device__ __forceinline__ uint8_t settle(int32_t acc, int shift) {
    const int32_t v = acc >> shift;
    return (uint8_t) (v < 0 ? 0 : v > 255 ? 255 : v);
}

// mid[t][y][x][c] = horizontal pass of source row y at resized column x + ox, for the crop columns
// that fall inside the resized image
__global__ void k_resize_rows(const uint8_t * __restrict__ src, uint8_t * __restrict__ mid, int n, int h, int w, int crop, int ox,
                              int rw, dev_axis ha) {
    const int64_t id = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t total = (int64_t) n * h * crop;
    if (id >= total) return;
    const int x = (int) (id % crop);
    const int64_t ty = id / crop;                      // t * h + y
    const int sx = x + ox;
    uint8_t * o = mid + id * 3;
    if (sx < 0 || sx >= rw) return;                    // padding column, never read
    const uint8_t * row = src + ty * w * 3;
    if (ha.identity) {
        o[0] = row[sx * 3]; o[1] = row[sx * 3 + 1]; o[2] = row[sx * 3 + 2];
        return;
    }
    const int32_t half = ha.shift > 0 ? 1 << (ha.shift - 1) : 0;
    int32_t a0 = half, a1 = half, a2 = half;
    const uint8_t * p = row + (int64_t) ha.lo[sx] * 3;
    for (int32_t t = ha.beg[sx], e = ha.beg[sx + 1]; t < e; t++, p += 3) {
        const int32_t k = ha.taps[t];
        a0 += (int32_t) p[0] * k;
        a1 += (int32_t) p[1] * k;
        a2 += (int32_t) p[2] * k;
    }
    o[0] = settle(a0, ha.shift);
    o[1] = settle(a1, ha.shift);
    o[2] = settle(a2, ha.shift);
}

struct norm_params {
    float mean[3], stdv[3], inv;
    int fused;
};

// out[c][t][y][x] for crop pixel (y, x) of frame t: vertical pass over mid, zero outside the resized
// image, then the normalisation
__global__ void k_resize_cols_norm(const uint8_t * __restrict__ mid, float * __restrict__ out, int n, int h, int crop, int oy, int ox,
                                   int rh, int rw, dev_axis va, norm_params np) {
    const int64_t id = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t plane = (int64_t) crop * crop;
    if (id >= (int64_t) n * plane) return;
    const int t = (int) (id / plane);
    const int64_t r = id - (int64_t) t * plane;
    const int y = (int) (r / crop), x = (int) (r - (int64_t) y * crop);
    const int sy = y + oy, sx = x + ox;
    uint8_t v[3] = {0, 0, 0};
    if (sy >= 0 && sy < rh && sx >= 0 && sx < rw) {
        const uint8_t * col = mid + ((int64_t) t * h * crop + x) * 3;   // row y of mid: + y * crop * 3
        if (va.identity) {
            const uint8_t * p = col + (int64_t) sy * crop * 3;
            v[0] = p[0]; v[1] = p[1]; v[2] = p[2];
        } else {
            const int32_t half = va.shift > 0 ? 1 << (va.shift - 1) : 0;
            int32_t a0 = half, a1 = half, a2 = half;
            const uint8_t * p = col + (int64_t) va.lo[sy] * crop * 3;
            for (int32_t k = va.beg[sy], e = va.beg[sy + 1]; k < e; k++, p += (int64_t) crop * 3) {
                const int32_t tap = va.taps[k];
                a0 += (int32_t) p[0] * tap;
                a1 += (int32_t) p[1] * tap;
                a2 += (int32_t) p[2] * tap;
            }
            v[0] = settle(a0, va.shift);
            v[1] = settle(a1, va.shift);
            v[2] = settle(a2, va.shift);
        }
    }
#pragma unroll
    for (int c = 0; c < 3; c++)
        out[((int64_t) c * n + t) * plane + r] = pre_normalize_v(np.fused != 0, np.inv, np.mean[c], np.stdv[c], v[c]);
}

typedef short s2v __attribute__((ext_vector_type(2)));
typedef unsigned int u3v __attribute__((ext_vector_type(3)));

__device__ __forceinline__ int32_t dot2(uint32_t px, uint32_t taps, int32_t acc) {
    return __builtin_amdgcn_sdot2(__builtin_bit_cast(s2v, px), __builtin_bit_cast(s2v, taps), acc, false);
}

constexpr int TILE_W = 64;   // output columns of a tile: one per lane in the horizontal pass

// LDS of a tile of th rows: [TILE_W] first inputs, [th] first inputs, taps of the columns and of the
// rows (npx and npy each, zeros behind an output's own), then the horizontal result as [row][channel][column]
struct tile_shape {
    int th, npx, npy, rows;   // rows: source rows a tile may need, and one more for the odd tap
    __host__ __device__ size_t lds() const {
        return (size_t) (TILE_W + th) * 4 + ((size_t) TILE_W * npx + (size_t) th * npy) * 2 + (size_t) rows * 3 * TILE_W;
    }
};

// taps [0, np) of output o of an axis, item k of them; 0 where the output lies outside the resized image
__device__ __forceinline__ int16_t tile_tap(const axis_filter & f, double unit, int o, int k, int & first) {
    first = 0;
    if (o < 0 || o >= f.n_out) return 0;
    int end;
    const double centre = axis_window(f, o, first, end);
    if (k >= end - first) return 0;
    double total = 0.0;
    for (int x = first; x < end; x++) total += axis_weight(f, x, centre);
    double v = axis_weight(f, first + k, centre);
    if (total != 0.0) v /= total;
    return round_tap(v * unit);
}

// One tile of one frame: out[c][t][y][x] for TILE_W columns and ts.th rows of the crop.
// Horizontal pass: lane = column, its taps in registers (NC groups of four; NC = 0: read from LDS as
// they are used), waves take the source rows in turn. Four pixels are twelve bytes, loaded as dwords
// and realigned; v_perm makes pairs of one channel, v_dot2_i32_i16 sums them with pairs of taps.
// Vertical pass: a thread takes four columns of one channel and pairs of rows.
// Sixteen 720 x 1280 frames to 256 x 256 of short edge 292: 19 us, where the two kernels and the five
// table uploads took 61 us of kernels, most of it in three byte loads per tap and 11.8 MB of
// intermediate written and read back (22 MB in and 12.6 MB out would take 4.5 us at the card's copy rate:
// the taps' VALU work and the latency of each row's loads bound it now).
// tile_tap sums an output's weights again for each of its taps: ~1 us of those 19, more where an output has more
// taps, and still ahead of the two kernels at the largest reduction a tile holds (whole calls: four frames of 2160
// x 3840 to 192, bicubic with 46 taps, 220 us against 625).
template <int NC>
__global__ __launch_bounds__(256) void k_resize_tile(const uint8_t * __restrict__ src, float * __restrict__ out, int n, int h, int w,
                                                     int crop, int oy, int ox, int tx, int ty, axis_filter fx, axis_filter fy, int xshift,
                                                     int yshift, tile_shape ts, norm_params np) {
    extern __shared__ __attribute__((aligned(16))) unsigned char sm[];
    int * xlo = (int *) sm, * ylo = xlo + TILE_W;
    int16_t * xt = (int16_t *) (ylo + ts.th), * yt = xt + TILE_W * ts.npx;
    uint8_t * mid = (uint8_t *) (yt + ts.th * ts.npy);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int per = tx * ty, t = (int) (blockIdx.x / (unsigned) per), tile = (int) blockIdx.x - t * per;
    const int y0 = tile / tx * ts.th, x0 = tile % tx * TILE_W;

    const double xunit = (double) (1 << xshift), yunit = (double) (1 << yshift);
    for (int i = tid; i < TILE_W * ts.npx; i += 256) {
        const int o = i / ts.npx, k = i - o * ts.npx;
        int first;
        xt[i] = tile_tap(fx, xunit, x0 + o < crop ? x0 + o + ox : -1, k, first);
        if (k == 0) xlo[o] = first;
    }
    // source rows of the tile: those of its first and last row inside the resized image
    const int sy0 = max(y0 + oy, 0), sy1 = min(min(y0 + ts.th, crop) + oy, fy.n_out) - 1;
    int r0 = 0, r1 = 0, unused;
    if (sy0 <= sy1) {
        axis_window(fy, sy0, r0, unused);
        axis_window(fy, sy1, unused, r1);
    }
    const int nrows = min(r1 - r0, ts.rows - 1);
    for (int i = tid; i < ts.th * ts.npy; i += 256) {
        const int o = i / ts.npy, k = i - o * ts.npy;
        int first;
        yt[i] = tile_tap(fy, yunit, y0 + o < crop ? y0 + o + oy : -1, k, first);
        if (k == 0) ylo[o] = min(max(first - r0, 0), max(nrows - 1, 0));
    }
    __syncthreads();

    {
        // dwords from the source row r0 on, up to the dword that holds the last byte of the frames
        const uint8_t * base = src + ((int64_t) t * h + r0) * w * 3;
        const uint32_t mis = (uint32_t) ((uintptr_t) base & 3);
        const int64_t left = (int64_t) ((int64_t) n - t) * h * w * 3 - (int64_t) r0 * w * 3;
        const brsrc rs = make_brsrc(base - mis, (left + mis + 3) & ~(int64_t) 3);
        const uint32_t pitch = (uint32_t) w * 3, col = mis + (uint32_t) xlo[lane] * 3;
        const int32_t half = xshift > 0 ? 1 << (xshift - 1) : 0;
        const uint2 * taps = (const uint2 *) (xt + lane * ts.npx);
        auto row_of = [&](int r, int nc, auto tap) {
            const uint32_t at = col + (uint32_t) r * pitch, off = at & ~3u;
            int32_t a0 = half, a1 = half, a2 = half;
            uint32_t d = (uint32_t) __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0);
#pragma unroll
            for (int k = 0; k < nc; k++) {
                const u3v v = __builtin_amdgcn_raw_buffer_load_b96(rs, off + 4 + 12 * k, 0, 0);
                const uint32_t e0 = __builtin_amdgcn_alignbyte(v.x, d, at), e1 = __builtin_amdgcn_alignbyte(v.y, v.x, at);
                const uint32_t e2 = __builtin_amdgcn_alignbyte(v.z, v.y, at);
                d = v.z;
                const uint2 q = tap(k);
                a0 = dot2(__builtin_amdgcn_perm(e0, e0, 0x0c030c00), q.x, a0);
                a1 = dot2(__builtin_amdgcn_perm(e1, e0, 0x0c040c01), q.x, a1);
                a2 = dot2(__builtin_amdgcn_perm(e1, e0, 0x0c050c02), q.x, a2);
                a0 = dot2(__builtin_amdgcn_perm(e2, e1, 0x0c050c02), q.y, a0);
                a1 = dot2(__builtin_amdgcn_perm(e2, e1, 0x0c060c03), q.y, a1);
                a2 = dot2(__builtin_amdgcn_perm(e2, e2, 0x0c030c00), q.y, a2);
            }
            uint8_t * o = mid + r * 3 * TILE_W + lane;
            o[0] = settle(a0, xshift);
            o[TILE_W] = settle(a1, xshift);
            o[2 * TILE_W] = settle(a2, xshift);
        };
        if constexpr (NC > 0) {
            uint2 q[NC];
#pragma unroll
            for (int k = 0; k < NC; k++) q[k] = taps[k];
#pragma unroll 4
            for (int r = wave; r < nrows; r += 4) row_of(r, NC, [&](int k) { return q[k]; });
        } else {
            for (int r = wave; r < nrows; r += 4) row_of(r, ts.npx / 4, [&](int k) { return taps[k]; });
        }
    }
    __syncthreads();

    const int32_t half = yshift > 0 ? 1 << (yshift - 1) : 0;
    const int64_t plane = (int64_t) crop * crop;
    for (int i = tid; i < ts.th * 3 * (TILE_W / 4); i += 256) {
        const int q = i & 15, c = (i >> 4) % 3, yl = (i >> 4) / 3;
        const int y = y0 + yl, x = x0 + 4 * q;
        if (y >= crop || x >= crop) continue;
        int32_t acc[4] = {half, half, half, half};
        const uint8_t * p = mid + (ylo[yl] * 3 + c) * TILE_W + 4 * q;
        const uint32_t * tp = (const uint32_t *) (yt + yl * ts.npy);
        if (nrows > 0) {
            // rows past the tile's last (taps of zero) repeat it
            const uint8_t * last = mid + ((nrows - 1) * 3 + c) * TILE_W + 4 * q;
            for (int k = 0; k < ts.npy / 2; k++, p += 6 * TILE_W) {
                const uint32_t d0 = *(const uint32_t *) (p < last ? p : last);
                const uint32_t d1 = *(const uint32_t *) (p + 3 * TILE_W < last ? p + 3 * TILE_W : last);
                const uint32_t tk = tp[k];
                acc[0] = dot2(__builtin_amdgcn_perm(d1, d0, 0x0c040c00), tk, acc[0]);
                acc[1] = dot2(__builtin_amdgcn_perm(d1, d0, 0x0c050c01), tk, acc[1]);
                acc[2] = dot2(__builtin_amdgcn_perm(d1, d0, 0x0c060c02), tk, acc[2]);
                acc[3] = dot2(__builtin_amdgcn_perm(d1, d0, 0x0c070c03), tk, acc[3]);
            }
        }
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = pre_normalize_v(np.fused != 0, np.inv, np.mean[c], np.stdv[c], settle(acc[e], yshift));
        float * o = out + ((int64_t) c * n + t) * plane + (int64_t) y * crop + x;
        if ((crop & 3) == 0 && ((uintptr_t) out & 15) == 0) *(float4 *) o = make_float4(v[0], v[1], v[2], v[3]);
        else
            for (int e = 0; e < 4 && x + e < crop; e++) o[e] = v[e];
    }
}

size_t align256(size_t b) { return (b + 255) & ~(size_t) 255; }

size_t axis_bytes(const resample_axis & ax) {
    return align256(ax.lo.size() * 4) + align256(ax.beg.size() * 4) + align256(ax.taps.size() * 2);
}

}  // namespace

// The tile of a call, or false where the two kernels serve. A tile is 64 columns by 16 rows (at a
// reduction of 2.5 a taller tile saves little: 45 source rows for 16, 84 for 32), fewer rows while the
// chip's 256 CUs would get fewer than two workgroups each. LDS is held to 48 KB (three workgroups per CU).
namespace {
bool tile_for(const jepa_preprocess_params * p, const pre_plan & g, int n_frames, int h, int w, tile_shape & ts) {
    const axis_filter fx = axis_filter_for(w, g.rw, p->resample), fy = axis_filter_for(h, g.rh, p->resample);
    if (!(fx.reach < 1000.0) || !(fy.reach < 1000.0)) return false;
    ts.npx = (fx.max_taps() + 3) / 4 * 4;
    ts.npy = (fy.max_taps() + 1) / 2 * 2;
    const int64_t tx = (g.crop + TILE_W - 1) / TILE_W;
    for (ts.th = 16; ts.th > 4 && tx * ((g.crop + ts.th - 1) / ts.th) * n_frames < 512; ts.th /= 2) {}
    ts.rows = (int) std::ceil((ts.th - 1) * fy.scale + 2.0 * fy.reach) + 3;
    return ts.lds() <= 48 * 1024 && (int64_t) ts.rows * w * 3 < (1ll << 30) && tx * ((g.crop + ts.th - 1) / ts.th) * n_frames < (1ll << 31);
}
}  // namespace

bool preprocess_tiled(const jepa_preprocess_params * p, const pre_plan & g, int n_frames, int h, int w) {
    tile_shape ts;
    return tile_for(p, g, n_frames, h, w, ts);
}

size_t preprocess_scratch_bound(const jepa_preprocess_params * p, const pre_plan & g, int n_frames, int h, int w) {
    auto axis = [&](int n_in, int n_out) {
        const size_t taps = (size_t) n_out * axis_filter_for(n_in, n_out, p->resample).max_taps();
        return 2 * align256(((size_t) n_out + 1) * 4) + align256(taps * 2);
    };
    return axis(w, g.rw) + axis(h, g.rh) + align256((size_t) n_frames * h * g.crop * 3);
}

size_t preprocess_scratch_bytes(const jepa_preprocess_params * p, const pre_plan & g, int n_frames, int h, int w) {
    return axis_bytes(resample_axis_for(w, g.rw, p->resample)) + axis_bytes(resample_axis_for(h, g.rh, p->resample)) +
           align256((size_t) n_frames * h * g.crop * 3);
}

namespace {

// Table bytes travel to the device as kernel arguments, PUT_CHUNK bytes per launch: a launch copies
// its arguments when it is enqueued (and a captured launch keeps them in its graph node), so no host
// buffer has to outlive the call, no pinned staging is needed and nothing waits on the stream.
constexpr int PUT_CHUNK = 3072;
struct put_args {
    unsigned char * dst;
    uint32_t n;
    unsigned char b[PUT_CHUNK];
};

__global__ void k_put_bytes(put_args a) {
    for (uint32_t i = threadIdx.x; i < a.n; i += blockDim.x) a.dst[i] = a.b[i];
}

}  // namespace

bool launch_preprocess(const jepa_preprocess_params * p, const pre_plan & g, const uint8_t * frames, int n_frames, int h, int w,
                       float * out, void * scratch, hipStream_t s) {
    norm_params np;
    for (int c = 0; c < 3; c++) { np.mean[c] = g.mean[c]; np.stdv[c] = g.stdv[c]; }
    np.inv = g.inv;
    np.fused = g.fused ? 1 : 0;
    tile_shape ts;
    if (tile_for(p, g, n_frames, h, w, ts)) {
        const axis_filter fx = axis_filter_for(w, g.rw, p->resample), fy = axis_filter_for(h, g.rh, p->resample);
        const int tx = (g.crop + TILE_W - 1) / TILE_W, ty = (g.crop + ts.th - 1) / ts.th;
        const unsigned grid = (unsigned) ((int64_t) tx * ty * n_frames);
        auto k = ts.npx == 4 ? k_resize_tile<1> : ts.npx == 8 ? k_resize_tile<2> : ts.npx == 12 ? k_resize_tile<3> : k_resize_tile<0>;
        k<<<grid, 256, ts.lds(), s>>>(frames, out, n_frames, h, w, g.crop, g.oy, g.ox, tx, ty, fx, fy, axis_shift(fx), axis_shift(fy), ts, np);
        return hipGetLastError() == hipSuccess;
    }
    const resample_axis hx = resample_axis_for(w, g.rw, p->resample), vx = resample_axis_for(h, g.rh, p->resample);
    // table blob: lo / beg / taps of both passes, 256-byte aligned pieces
    std::vector<unsigned char> blob(axis_bytes(hx) + axis_bytes(vx), 0);
    unsigned char * dev = (unsigned char *) scratch;
    size_t off = 0;
    auto put = [&](const void * src, size_t bytes) -> const void * {
        if (bytes) memcpy(blob.data() + off, src, bytes);
        const void * d = dev + off;
        off += align256(bytes);
        return d;
    };
    auto upload = [&](const resample_axis & ax, bool identity) {
        dev_axis d;
        d.lo = (const int32_t *) put(ax.lo.data(), ax.lo.size() * 4);
        d.beg = (const int32_t *) put(ax.beg.data(), ax.beg.size() * 4);
        d.taps = (const int16_t *) put(ax.taps.data(), ax.taps.size() * 2);
        d.shift = ax.shift;
        d.identity = identity ? 1 : 0;
        return d;
    };
    const dev_axis dh = upload(hx, g.rw == w), dv = upload(vx, g.rh == h);
    uint8_t * mid = (uint8_t *) dev + off;
    for (size_t o = 0; o < off; o += PUT_CHUNK) {
        put_args pa;
        pa.dst = dev + o;
        pa.n = (uint32_t) std::min<size_t>(PUT_CHUNK, off - o);
        memcpy(pa.b, blob.data() + o, pa.n);
        k_put_bytes<<<1, 256, 0, s>>>(pa);
    }
    const int64_t n1 = (int64_t) n_frames * h * g.crop, n2 = (int64_t) n_frames * g.crop * g.crop;
    k_resize_rows<<<(unsigned) ((n1 + 255) / 256), 256, 0, s>>>(frames, mid, n_frames, h, w, g.crop, g.ox, g.rw, dh);
    k_resize_cols_norm<<<(unsigned) ((n2 + 255) / 256), 256, 0, s>>>(mid, out, n_frames, h, g.crop, g.oy, g.ox, g.rh, g.rw, dv, np);
    return hipGetLastError() == hipSuccess;
}

// ---------------------------------------------------------------------------------------------------
// The same preprocessing without any allocation: the tables and the horizontal-pass image live in a
// file-scope device array. A host reference to `scratch` names a host-side stand-in, not device
// memory; the device address of each GPU's copy comes from hipGetSymbolAddress with that GPU
// current, and only that address is handed to copies and kernels.
// ---------------------------------------------------------------------------------------------------
namespace {
__device__ __align__(256) unsigned char scratch[PRE_NOALLOC_SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void * g_scratch_ptr[MAX_DEVICES] = {};
}  // namespace

void * preprocess_static_scratch(int device) {
    if (device < 0 || device >= MAX_DEVICES) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void * ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            jepa_log("jepa: hipGetSymbolAddress(scratch) failed on device %d: %s\n", device, hipGetErrorString(e));
            (void) hipGetLastError();
            return nullptr;
        }
        g_scratch_ptr[device] = ptr;
    }
    return g_scratch_ptr[device];
}
