// Host build of the walk over edge records (walk_edges) in each of their
// formats (kind 0: global), packed by the library's own packing, beside the
// walk over the 48-byte records (walk_ray).  Test infrastructure only.
#include "../../haseongpu_amd/csrc/edge_records.h"

using namespace hase;

static void put(const WalkOut& w, float* out, uint32_t* steps, int32_t* status)
{
    out[0] = w.beta_len;
    out[1] = w.gain_len;
    out[2] = w.clad_len;
    out[3] = w.refl;
    out[4] = w.length;
    *steps = w.steps;
    *status = w.status;
}

template <uint32_t kKind>
static WalkOut walk(const MeshDev& m, const EdgeRecords& er, const float* a, uint32_t t, uint32_t l, const float* e,
                    uint32_t nr, uint32_t first)
{
    const auto edges = edge_fetch<kKind>(er.staged.data(), m.T, m.np);
    return walk_edges(m, a[0], a[1], a[2], t, l, edges.vertex(m, t, 0u), edges.vertex(m, t, 1u), edges.vertex(m, t, 2u),
                      e[0], e[1], e[2], nr, first, edges);
}

extern "C" uint32_t edge_kind_host(uint32_t T, uint32_t np)
{
    size_t bytes;
    return edge_kind(T, np, bytes);
}

extern "C" int edge_walk_host(uint32_t T, uint32_t layers, float h, const uint32_t* rec, const float* pts, uint32_t np,
                              uint32_t kind, const float* beta, const float* refl, const float* nidx, uint32_t n,
                              const float* start, const uint32_t* prism, const float* end, const uint32_t* nrefl,
                              const uint32_t* first, float* out, uint32_t* steps, int32_t* status, float* out_ref,
                              uint32_t* steps_ref, int32_t* status_ref)
{
    MeshDev m{};
    m.rec = reinterpret_cast<const uint4*>(rec);
    m.beta = beta;
    m.refl = refl;
    m.T = T;
    m.np = np;
    m.layers = layers;
    m.h = h;
    if (nidx) {
        m.has_nidx = 1;
        m.nin_b = nidx[0]; m.nout_b = nidx[1]; m.nin_t = nidx[2]; m.nout_t = nidx[3];
    }
    const EdgeRecords er = edge_records(m.rec, T, reinterpret_cast<const float2*>(pts), np, kind);
    m.edges = er.global.data();
    for (uint32_t i = 0; i < n; ++i) {
        const uint32_t t = prism[i] % T, l = prism[i] / T;
        const float *a = start + 3 * i, *e = end + 3 * i;
        const WalkOut w = kind == kLdsEdges          ? walk<kLdsEdges>(m, er, a, t, l, e, nrefl[i], first[i])
                          : kind == kLdsIndexedEdges ? walk<kLdsIndexedEdges>(m, er, a, t, l, e, nrefl[i], first[i])
                          : kind == kLdsTwins        ? walk<kLdsTwins>(m, er, a, t, l, e, nrefl[i], first[i])
                                                     : walk<0u>(m, er, a, t, l, e, nrefl[i], first[i]);
        put(w, out + 5 * i, steps + i, status + i);
        put(walk_ray(m, a[0], a[1], a[2], t, l, e[0], e[1], e[2], nrefl[i], first[i]), out_ref + 5 * i, steps_ref + i,
            status_ref + i);
    }
    return 0;
}

extern "C" uint32_t fast_div_host(uint32_t d, uint32_t n) { return fast_div(d)(n); }
