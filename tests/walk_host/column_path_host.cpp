// Host build of the importance map's path replay (column_path, path_ray_*):
// every entry of one sample's map, and the map by whole column walks
// (column_entries) beside it.  Test infrastructure only.
#include <vector>

#include "../../haseongpu_amd/csrc/edge_records.h"
#include "../../haseongpu_amd/csrc/importance_walk.h"

using namespace hase;

extern "C" int column_path_host(uint32_t T, uint32_t layers, float h, const uint32_t* rec, const float* pts,
                                uint32_t np, const float* beta,
                                const float* bv, const float* refl, const float* nidx, float clad_alpha,
                                const float* c1, const float* c2, uint32_t n_lambda, float px, float py, int plane,
                                uint32_t R, int transfer, uint32_t cap, float* replay, float* columns,
                                unsigned long long* replay_steps, unsigned long long* column_steps, uint32_t* full)
{
    MeshDev m{};
    m.rec = reinterpret_cast<const uint4*>(rec);
    m.beta = beta;
    m.bv = bv;
    m.refl = refl;
    m.T = T;
    m.layers = layers;
    m.h = h;
    m.clad_alpha = clad_alpha;
    if (nidx) {
        m.has_nidx = 1;
        m.nin_b = nidx[0]; m.nout_b = nidx[1]; m.nin_t = nidx[2]; m.nout_t = nidx[3];
    }
    std::vector<float> col((size_t)T * layers);
    for (uint32_t l = 0; l < layers; ++l)
        for (uint32_t t = 0; t < T; ++t) col[(size_t)t * layers + l] = beta[t + (size_t)l * T];
    m.beta_col = col.data();
    const EdgeRecords er = edge_records(m.rec, T, reinterpret_cast<const float2*>(pts), np);
    m.edges = er.global.data();
    const uint32_t P = T * layers;
    const GlobalTriangles fetch;
    const ColumnItems ci(T, layers, R);
    *column_steps = *replay_steps = 0;
    *full = 0;
    for (uint32_t it = 0; it < ci.per_sample(); ++it) {
        uint32_t t0, k;
        int lv0, nlev;
        ci.decode(it, t0, k, lv0, nlev);
        float v[kLevelGroup];
        *column_steps += column_entries(m, fetch, c1, c2, n_lambda, 1.0f / (float)n_lambda, t0, lv0, nlev, k, px, py,
                                        plane, transfer != 0, v);
        float u[kLevelGroup];
        column_entries(m, GlobalEdges{}, c1, c2, n_lambda, 1.0f / (float)n_lambda, t0, lv0, nlev, k, px, py, plane,
                       transfer != 0, u);
        for (int g = 0; g < nlev; ++g)
            if (u[g] != v[g]) return 1;   // the same walk over the edge records
        for (int g = 0; g < nlev; ++g) columns[(size_t)k * P + t0 + (size_t)(lv0 + g) * T] = v[g];
    }
    std::vector<uint2> entries(cap + 2u);
    for (uint32_t t0 = 0; t0 < T; ++t0) {
        const ColumnPath path = column_path(m, GlobalEdges{}, t0, px, py, [&](uint32_t i, uint32_t t, float s) {
            if (i >= cap) return false;
            entries[i] = make_uint2(4u * t, __builtin_bit_cast(uint32_t, s));
            return true;
        });
        if (path.full) {
            ++*full;
            continue;
        }
        entries[path.steps] = make_uint2(0u, kPathEnd);
        const float d2 = path.d2;
        for (uint32_t k = 0; k < R; ++k) {
            const uint32_t nr = (k + 1u) >> 1, first = k & 1u;
            for (uint32_t l = 0; l < layers; ++l) {
                const int end = image_plane(plane, (int)layers, nr, first);
                PathRay w = path_ray_begin(m, (int)l, end);
                const uint32_t last = path_ray_replay(m, w, d2, nr, entries.data(), 1u);
                *replay_steps += path.steps + path_ray_planes(w, (int)l, end);
                const float b = m.bv[t0 + l * T];
                float v = 0.0f;
                if (path.ok && (b > 0.0f || transfer))
                    v = path_ray_value(m, w, last, path.clad, path.s, d2, nr, first, c1, c2, n_lambda,
                                       1.0f / (float)n_lambda, b, transfer != 0);
                replay[(size_t)k * P + t0 + (size_t)l * T] = v;
            }
        }
    }
    return 0;
}
