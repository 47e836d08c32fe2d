// edge_records.h - the host's packing of the edge records (prism_walk.h): the
// global ones and, where the mesh fits, the ones that a kernel stages in LDS.
#pragma once

#include <cstring>
#include <vector>

#include "prism_walk.h"

namespace hase {

struct EdgeRecords {
    std::vector<uint4> global, staged;
    uint32_t kind = 0;        // format of staged: 0 (none), kLdsEdges, kLdsIndexedEdges or kLdsTwins
};

// The widest format that LDS holds, none for larger meshes (their walks read
// the global records): each step down the list costs a walk step one or two
// more dependent LDS reads, still under the ~500 cycles of a global record
// that misses L1.  16-bit links hold meshes below 10,922 triangles.
inline uint32_t edge_kind(uint32_t T, uint32_t np, size_t& bytes)
{
    const size_t room = (size_t)kLdsStageWords * 16u, table = 8u * (size_t)np;
    bytes = 0;
    if (3u * (size_t)T >= ShortLinks::kNone || np > 0x10000u) return 0u;
    if ((bytes = 36u * (size_t)T) <= room) return kLdsEdges;
    if ((bytes = table + 18u * (size_t)T) <= room) return kLdsIndexedEdges;
    if ((bytes = table + 12u * (size_t)T) <= room) return kLdsTwins;
    bytes = 0;
    return 0u;
}

// From the 48-byte records (3 per triangle) and the FP32 points; kind: a
// staged format to pack in place of the one edge_kind chooses.
inline EdgeRecords edge_records(const uint4* rec, uint32_t T, const float2* pts, uint32_t np, uint32_t kind = 0u)
{
    EdgeRecords e;
    size_t bytes = 0;
    const uint32_t chosen = edge_kind(T, np, bytes);
    if (!kind) kind = chosen;
    if (kind == kLdsEdges) bytes = 36u * (size_t)T;
    if (kind == kLdsIndexedEdges) bytes = 8u * (size_t)np + 18u * (size_t)T;
    if (kind == kLdsTwins) bytes = 8u * (size_t)np + 12u * (size_t)T;
    e.kind = kind;
    e.global.resize(4u * (size_t)T, make_uint4(0u, 0u, 0u, 0u));
    e.staged.resize((bytes + 15u) / 16u, make_uint4(0u, 0u, 0u, 0u));
    // the two smaller formats: points, links, point indices
    float2* xy = reinterpret_cast<float2*>(e.staged.data());
    uint32_t* words32 = reinterpret_cast<uint32_t*>(xy + np);
    uint16_t* words16 = reinterpret_cast<uint16_t*>(words32);
    if (kind == kLdsIndexedEdges || kind == kLdsTwins)
        for (uint32_t i = 0; i < np; ++i) xy[i] = pts[i];
    for (uint32_t t = 0; t < T; ++t) {
        const uint4 b = rec[3u * (size_t)t + 1u], c = rec[3u * (size_t)t + 2u];
        const uint32_t words[3] = {b.z, b.w, c.x}, point[3] = {c.y & 0x7FFFFFFFu, c.z, c.w};
        const uint32_t clad = record_cladding(c);
        uint32_t link[3], brief[3];
        for (uint32_t k = 0; k < 3u; ++k) {
            const uint32_t n = nw_next(words[k]), f = nw_edge(words[k]);
            const bool rim = nw_boundary(words[k]);
            link[k] = (rim ? GlobalEdges::kNone : (4u * n + f) * 16u) | clad;
            brief[k] = rim ? ShortLinks::kNone : 3u * n + f;
        }
        for (uint32_t f = 0; f < 3u; ++f) {
            const uint32_t e1 = (f + 1u) % 3u, e2 = (f + 2u) % 3u;   // vertex e2 is opposite edge f
            const size_t i = 3u * (size_t)t + f;
            const float2 n = pts[point[e2]];
            const uint32_t both = brief[e1] | brief[e2] << 15 | clad << 31;
            e.global[4u * (size_t)t + f] =
                make_uint4(__builtin_bit_cast(uint32_t, n.x), __builtin_bit_cast(uint32_t, n.y), link[e1], link[e2]);
            if (kind == kLdsEdges) {
                reinterpret_cast<LdsEdge*>(e.staged.data())[i] = LdsEdge{n.x, n.y, both};
            } else if (kind == kLdsIndexedEdges) {
                words32[i] = both;
                reinterpret_cast<uint16_t*>(words32 + 3u * (size_t)T)[i] = (uint16_t)point[e2];
            } else if (kind == kLdsTwins) {
                words16[i] = (uint16_t)(brief[f] | clad << 15);
                words16[3u * (size_t)T + i] = (uint16_t)point[f];
            }
        }
    }
    return e;
}

}  // namespace hase
