// Tet chunks of the local step: the host builder of their lists and the
// device body shared by the kernels that run computeLocal over them.
//
// A chunk is up to kChunkTets consecutive tets of some order (one workgroup).  It
// lists the vertices it touches (sorted; an entry is a (chunk, vertex) pair),
// its tets' corners as indices into that list, and per entry the (tet, corner)
// pairs that touch it in tet order.  The forces of an entry's tets are summed
// inside the chunk and written once, in vertex-major order over all chunks, so
// every consumer reads a vertex's partial forces as one run.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

#include "common.hpp"
#include "svd3.hpp"

#ifndef SBS_CHUNK_TETS
#define SBS_CHUNK_TETS 256
#endif
// Unroll of the local step's per-vertex incidence sums: the LDS reads of
// several incidences are in flight together (the sum keeps its order).
#ifndef SBS_GATHER_UNROLL
#define SBS_GATHER_UNROLL 2
#endif
#define SBS_PRAGMA(x) _Pragma(#x)
#define SBS_UNROLL(n) SBS_PRAGMA(unroll n)

namespace sbs {

constexpr int kChunkTets = SBS_CHUNK_TETS;  // tets per chunk (one workgroup)

// flags of the local step
constexpr int kLocalResidual = 1;  // P = R - F (Jacobi mode) instead of R
constexpr int kLocalPolar = 2;     // FP32: rotation by Newton's polar iteration (SVD fallback)

struct ChunkLists {
    int chunks = 0, max_verts = 0;      // most vertices of one chunk
    std::vector<int> vptr;              // chunks + 1: first entry of each chunk
    std::vector<uint32_t> verts;        // vertex of each entry
    std::vector<uint32_t> pos;          // entry -> its slot in vertex-major order
    std::vector<uint32_t> entry;        // slot -> entry
    std::vector<int> vert_ptr;          // nv + 1: slots of each vertex
    std::vector<uint2> lidx;            // per tet 4 x u16 corners as indices into the chunk's list
    std::vector<uint16_t> inc_codes;    // per chunk 4 kChunkTets: (tet << 2 | corner) grouped by entry
    std::vector<uint16_t> inc_end;      // per entry: end of its codes in the chunk's list
};

// tets: 4 vertices (below nv) per tet, in the chunks' order; chunk c holds the
// tets starts[c] .. starts[c + 1] (kChunkTets at most).
inline ChunkLists build_chunk_lists(int nv, const std::vector<uint32_t>& tets, const std::vector<int>& starts) {
    ChunkLists o;
    const int nt = (int)(tets.size() / 4);
    o.chunks = (int)starts.size() - 1;
    o.vptr.assign(o.chunks + 1, 0);
    o.verts.reserve((size_t)nt * 2);
    o.lidx.resize(nt);
    o.inc_end.reserve((size_t)nt * 2);
    o.inc_codes.assign((size_t)o.chunks * 4 * kChunkTets, 0);
    std::vector<uint32_t> tmp;
    std::vector<int> cnt(4 * kChunkTets), at;
    for (int c = 0; c < o.chunks; ++c) {
        const int t0 = starts[c], t1 = starts[c + 1];
        tmp.assign(tets.begin() + 4 * (size_t)t0, tets.begin() + 4 * (size_t)t1);
        std::sort(tmp.begin(), tmp.end());
        tmp.erase(std::unique(tmp.begin(), tmp.end()), tmp.end());
        const size_t nloc = tmp.size();
        o.max_verts = std::max(o.max_verts, (int)nloc);
        std::fill(cnt.begin(), cnt.end(), 0);
        for (int i = t0; i < t1; ++i) {
            uint32_t l[4];
            for (int j = 0; j < 4; ++j) {
                l[j] = (uint32_t)(std::lower_bound(tmp.begin(), tmp.end(), tets[4 * (size_t)i + j]) - tmp.begin());
                cnt[l[j]]++;
            }
            o.lidx[i] = make_uint2(l[0] | (l[1] << 16), l[2] | (l[3] << 16));
        }
        at.assign(nloc + 1, 0);
        for (size_t k = 0; k < nloc; ++k) at[k + 1] = at[k] + cnt[k];
        for (size_t k = 0; k < nloc; ++k) o.inc_end.push_back((uint16_t)at[k + 1]);
        uint16_t* codes = &o.inc_codes[(size_t)c * 4 * kChunkTets];
        for (int i = t0; i < t1; ++i)
            for (int j = 0; j < 4; ++j) {
                const uint32_t word = j < 2 ? o.lidx[i].x : o.lidx[i].y;
                const uint32_t lv = (j & 1) ? word >> 16 : word & 0xffffu;
                codes[at[lv]++] = (uint16_t)(((i - t0) << 2) | j);
            }
        o.verts.insert(o.verts.end(), tmp.begin(), tmp.end());
        o.vptr[c + 1] = (int)o.verts.size();
    }
    const size_t ne = o.verts.size();
    o.vert_ptr.assign(nv + 1, 0);
    for (uint32_t g : o.verts) o.vert_ptr[g + 1]++;
    for (int v = 0; v < nv; ++v) o.vert_ptr[v + 1] += o.vert_ptr[v];
    o.entry.resize(ne);
    o.pos.resize(ne);
    std::vector<int> fill(o.vert_ptr.begin(), o.vert_ptr.end() - 1);
    for (size_t e = 0; e < ne; ++e) o.entry[fill[o.verts[e]]++] = (uint32_t)e;
    for (size_t j = 0; j < ne; ++j) o.pos[o.entry[j]] = (uint32_t)j;
    return o;
}

// Chunks of kChunkTets tets, the last one of what is left.
inline ChunkLists build_chunk_lists(int nv, const std::vector<uint32_t>& tets) {
    const int nt = (int)(tets.size() / 4);
    std::vector<int> starts;
    for (int t = 0; t < nt; t += kChunkTets) starts.push_back(t);
    starts.push_back(nt);
    return build_chunk_lists(nv, tets, starts);
}

// LDS of one workgroup: corner forces, staged q, incidence list.
template <class T> size_t chunk_lds_bytes(int max_verts) {
    const size_t b = (12 * (size_t)kChunkTets + 3 * (size_t)max_verts) * sizeof(T) +
                     (4 * (size_t)kChunkTets + (size_t)max_verts) * sizeof(uint16_t);
    return (b + 15) & ~(size_t)15;
}

template <class T> __device__ __forceinline__ void load_dminv(const T* __restrict__ dminv, int nt, unsigned t, T (&m)[9]) {
#pragma unroll
    for (int k = 0; k < 9; ++k) m[k] = dminv[(size_t)k * nt + t];
}

// Chunk c of the lists, the tets t0 .. t1 (thread i the tet t0 + i), by a
// workgroup of kChunkTets threads:
//   1. the chunk's vertices are staged into LDS (stage(entry, vertex, x, y, z)
//      gives the position), with the chunk's incidence list;
//   2. one thread per tet: F = Ds Dm^-1, the rotation in registers, R (or
//      R - F), the 4 corner forces of w R Dm^-T G^T written to LDS;
//   3. one thread per entry sums its incidences in list order (the three
//      components together, each code decoded once) and writes the partial
//      force at its slot.
// No atomics anywhere, so the result is deterministic.
template <class T, class Stage>
__device__ __forceinline__ void local_chunk(unsigned c, unsigned t0, unsigned t1, int nt,
                                            const uint2* __restrict__ lidx,
                                            const int* __restrict__ chunk_vptr,
                                            const uint32_t* __restrict__ chunk_verts,
                                            const uint32_t* __restrict__ entry_pos,
                                            const uint16_t* __restrict__ inc_codes,
                                            const uint16_t* __restrict__ inc_end, const T* __restrict__ dminv,
                                            const T* __restrict__ w, T* __restrict__ partial, int flags,
                                            unsigned char* smem_raw, Stage&& stage) {
    const int e0 = chunk_vptr[c], nu = chunk_vptr[c + 1] - e0;
    T* fs = reinterpret_cast<T*>(smem_raw);                    // [12][kChunkTets] corner forces
    T* qs = fs + 12 * kChunkTets;                              // [nu][3] staged q
    uint16_t* codes = reinterpret_cast<uint16_t*>(qs + 3 * (size_t)nu);  // [4 kChunkTets] tet<<2 | corner
    uint16_t* ends = codes + 4 * kChunkTets;                   // [nu] end of each vertex's incidences
    for (int i = threadIdx.x; i < nu; i += kChunkTets) {
        const uint32_t g = chunk_verts[e0 + i];
        T x, y, z;
        stage(e0 + i, g, x, y, z);
        qs[3 * i] = x; qs[3 * i + 1] = y; qs[3 * i + 2] = z;
        ends[i] = inc_end[e0 + i];
    }
    {
        const uint32_t* src = reinterpret_cast<const uint32_t*>(inc_codes) + (size_t)c * (2 * kChunkTets);
        uint32_t* dst = reinterpret_cast<uint32_t*>(codes);
        for (int k = threadIdx.x; k < 2 * kChunkTets; k += kChunkTets) dst[k] = src[k];
    }
    __syncthreads();
    const unsigned t = t0 + threadIdx.x;
    if (t < t1) {
        const uint2 li = lidx[t];
        const unsigned l0 = li.x & 0xffffu, l1 = li.x >> 16, l2 = li.y & 0xffffu, l3 = li.y >> 16;
        T m[9];
        load_dminv(dminv, nt, t, m);
        const T ww = w[t];
        T F[3][3];
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const T x0 = qs[3 * l0 + r];
            const T d0 = qs[3 * l1 + r] - x0, d1 = qs[3 * l2 + r] - x0, d2 = qs[3 * l3 + r] - x0;
#pragma unroll
            for (int k = 0; k < 3; ++k) F[r][k] = d0 * m[k] + d1 * m[3 + k] + d2 * m[6 + k];
        }
        T P[3][3];
        pd_projection(F, (flags & kLocalResidual) != 0, P, (flags & kLocalPolar) != 0);
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            // column j of w P Dm^-T is w P (row j of Dm^-1); corner 0 gets minus their sum
            const T f1 = ww * (P[r][0] * m[0] + P[r][1] * m[1] + P[r][2] * m[2]);
            const T f2 = ww * (P[r][0] * m[3] + P[r][1] * m[4] + P[r][2] * m[5]);
            const T f3 = ww * (P[r][0] * m[6] + P[r][1] * m[7] + P[r][2] * m[8]);
            fs[(0 * 3 + r) * kChunkTets + threadIdx.x] = -(f1 + f2 + f3);
            fs[(1 * 3 + r) * kChunkTets + threadIdx.x] = f1;
            fs[(2 * 3 + r) * kChunkTets + threadIdx.x] = f2;
            fs[(3 * 3 + r) * kChunkTets + threadIdx.x] = f3;
        }
    }
    __syncthreads();
    // one thread per chunk vertex sums all three components, so each
    // incidence code is read and decoded once
    for (int i = threadIdx.x; i < nu; i += kChunkTets) {
        const int k1 = ends[i];
        T a0 = 0, a1 = 0, a2 = 0;
        SBS_UNROLL(SBS_GATHER_UNROLL)
        for (int k = i ? ends[i - 1] : 0; k < k1; ++k) {
            const unsigned code = codes[k];
            const T* f = fs + (code & 3u) * 3 * kChunkTets + (code >> 2);
            a0 += f[0];
            a1 += f[kChunkTets];
            a2 += f[2 * kChunkTets];
        }
        T* out = partial + 3 * (size_t)entry_pos[e0 + i];  // vertex-major: the consumers read contiguously
        out[0] = a0;
        out[1] = a1;
        out[2] = a2;
    }
}

}  // namespace sbs
