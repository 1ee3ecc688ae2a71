// rope3d.cpp - host RoPE tables (see rope3d.h; reference src/rope3d.cpp:9-134).
#include "rope3d.h"

#include <cmath>
#include <numeric>

int rope3d_axis_dim(int head_dim) { return 2 * ((head_dim / 3) / 2); }

namespace {

// (rescaled) coordinate of grid index `i` along one axis; t is never rescaled (reference
// src/rope3d.cpp:13-28, Meta's interpolate_rope)
float axis_pos(const rope3d_params & p, int axis, int i) {
    float v = (float) i;
    if (!p.interpolate) return v;
    if (axis == 1 && p.grid_h > 1) v = (v * (float) (p.train_grid_h - 1)) / (float) (p.grid_h - 1);
    if (axis == 2 && p.grid_w > 1) v = (v * (float) (p.train_grid_w - 1)) / (float) (p.grid_w - 1);
    return v;
}

}  // namespace

void rope3d_axis_tables(const rope3d_params & p, const std::vector<int32_t> & times, std::vector<float> & c, std::vector<float> & s) {
    const int d = rope3d_axis_dim(p.head_dim), half = d / 2;
    const size_t dims[3] = {times.size(), (size_t) p.grid_h, (size_t) p.grid_w};
    c.resize((dims[0] + dims[1] + dims[2]) * d);
    s.resize(c.size());
    std::vector<float> omega((size_t) half);
    for (int k = 0; k < half; k++) omega[(size_t) k] = 1.0f / powf(p.theta, (float) k / (float) half);
    size_t at = 0;
    for (int a = 0; a < 3; a++)
        for (size_t i = 0; i < dims[a]; i++) {
            const float pos = axis_pos(p, a, a == 0 ? times[i] : (int) i);
            for (int j = 0; j < d; j++, at++) {
                const int k = p.variant == 0 ? (j % half) : (j / 2);
                const float ang = pos * omega[(size_t) k];
                c[at] = cosf(ang);
                s[at] = sinf(ang);
            }
        }
}

void rope3d_compact(const rope3d_params & p, const int32_t * ids, int64_t n, std::vector<int32_t> & times, std::vector<int32_t> & compact_ids) {
    const int32_t per_frame = p.grid_h * p.grid_w;
    std::vector<int32_t> slot((size_t) p.grid_t, -1);
    times.clear();
    compact_ids.resize((size_t) n);
    for (int64_t i = 0; i < n; i++) {
        const int32_t t = ids[i] / per_frame;
        if (slot[(size_t) t] < 0) { slot[(size_t) t] = (int32_t) times.size(); times.push_back(t); }
        compact_ids[(size_t) i] = slot[(size_t) t] * per_frame + ids[i] % per_frame;
    }
}

void rope3d_tables(const rope3d_params & p, const int32_t * ids, int64_t n_rows, std::vector<float> & c,
                   std::vector<float> & s, bool signed_sin) {
    const int D = p.head_dim, d = rope3d_axis_dim(D);
    c.assign((size_t) n_rows * D, 1.0f);
    s.assign((size_t) n_rows * D, 0.0f);
    if (d == 0) return;
    std::vector<float> ac, as;
    std::vector<int32_t> times((size_t) p.grid_t);
    std::iota(times.begin(), times.end(), 0);
    rope3d_axis_tables(p, times, ac, as);
    const int first[3] = {0, p.grid_t, p.grid_t + p.grid_h};   // axis a's first row
    const int64_t per_frame = (int64_t) p.grid_h * p.grid_w;
    for (int64_t r = 0; r < n_rows; r++) {
        const int64_t id = ids ? ids[r] : r;
        const int64_t idx[3] = {id / per_frame, (id % per_frame) / p.grid_w, id % p.grid_w};
        float * cr = &c[(size_t) r * D];
        float * sr = &s[(size_t) r * D];
        for (int a = 0; a < 3; a++)
            for (int j = 0; j < d; j++) {
                cr[a * d + j] = ac[(size_t) (first[a] + idx[a]) * d + j];
                sr[a * d + j] = as[(size_t) (first[a] + idx[a]) * d + j];
            }
        if (signed_sin)
            for (int j = 0; j < D; j += 2) sr[j] = -sr[j];
    }
}
