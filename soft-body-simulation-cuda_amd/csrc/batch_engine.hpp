// Batched PD step for many independent bodies on gfx950: every body advances
// with its own Jacobi-PCG global solve (its own alpha, beta and stop test,
// pcgJacobi.cu:134-135 applied per body).  The step (pdSolver.cu:141-208) is a
// sequence of launches over all bodies: the prologue, then per local/global
// iteration computeLocal over the tet chunks of all bodies (so the tets of the
// largest body spread over the CUs) and one launch with a workgroup per body
// that gathers the right-hand side, runs the whole PCG solve and applies the
// Chebyshev recurrence, then updateVelPos.  One stream, so a captured step is
// a chain.  (One workgroup running a body's whole step, local step included,
// was bound by the largest body's chain: 256 bodies of 3..20 hexes per axis,
// 10 iterations, 10.5-12.9 ms a step; this form 3.17 ms;
// 1,024 such bodies 19.3 -> 6.3 ms.)
//
// Bodies are the connected components of the tet mesh (the reference's
// DataLoader concatenates bodies, dataLoader.cu:292-378; they stay
// independent because no tet spans two).  Internally the vertices are
// renumbered body by body; caller arrays are read and written through that
// permutation at the step's ends.
//
// Precision: each body's vectors are held relative to a local origin (the rest
// position of its first vertex), so FP32 rounds offsets of the body's size
// rather than of its distance from the world origin; dot products accumulate
// in FP64.
//
// Tile choice: the workgroup size (64..1024 threads, shared by all bodies)
// comes from an autotuner that times one step with every candidate on a copy
// of the state at prepare.
#pragma once

#include <memory>
#include <string>
#include <vector>

#include "common.hpp"

namespace sbs {

struct BatchBody {
    int verts = 0, tets = 0, iterations = 0, solves = 0, max_per_solve = 0, unconverged = 0;
};

// Bodies by size, for reports: the classes share the launches.
struct BatchClass {
    int min_tets = 0, max_tets = 0, bodies = 0, threads = 0;  // threads per workgroup chosen by the tuner
    std::vector<std::pair<int, double>> tried;               // (threads, ms of one step) the tuner measured
};

// Host inputs of the batched system, all in the caller's vertex and tet order.
template <class T> struct BatchSystem {
    int nv = 0, nt = 0;
    std::vector<uint32_t> tets;       // 4 per tet
    std::vector<T> dminv, w;          // 9 (row-major) and 1 per tet
    std::vector<T> c0, diagA, mass, dbc;  // per vertex
    std::vector<T> x0;                // 3 per vertex: rest positions (the bodies' local origins)
    std::vector<int> rowptr, col;     // CSR of the scalar matrix, diagonal included
    std::vector<T> val;
};

struct BatchParams {
    int iterations = 10;
    double dt = 1.0 / 60.0, gravity = 9.8, rho = 0.9992;
    double pcg_tol = 1e-6, pcg_floor = 1e-8;
    int pcg_max_iter = 200;
    bool write_x = true;  // false when the collision response decides X
    bool polar = false;   // FP32 local step: rotation by Newton's polar iteration (SVD fallback)
};

template <class T> class BatchEngine {
public:
    explicit BatchEngine(const BatchSystem<T>& sys);
    // One step of every body on `stream`; X, V, XTilde and DBCX are the caller's
    // arrays.
    void step(T* X, T* V, T* XTilde, const T* DBCX, const BatchParams& p, hipStream_t stream);
    // Chooses the workgroup size by timing one step per candidate on
    // copies of X, V, XTilde (the caller's state is not changed).
    void autotune(const T* X, const T* V, const T* DBCX, const BatchParams& p, hipStream_t stream);
    int num_bodies() const { return nb_; }
    const std::vector<BatchClass>& classes() const { return cls_; }
    // Per-body PCG statistics accumulated since the last reset (waits for the GPU).
    std::vector<BatchBody> body_stats();
    void reset_stats();

private:
    void launch_step(T* X, T* V, T* XTilde, const T* DBCX, const BatchParams& p, hipStream_t s, int threads);
    void set_threads(int threads);

    int nv_ = 0, nt_ = 0, nb_ = 0, max_verts_ = 0, threads_ = 256;
    std::vector<int> verts_h_, tets_h_;  // per body, the caller's order
    // the tets in chunks
    int chunks_ = 0;
    size_t local_lds_ = 0;               // of a chunk's workgroup
    DevBuf<uint2> lidx_;
    DevBuf<int> chunk_tptr_, chunk_vptr_, vent_ptr_;
    DevBuf<uint32_t> chunk_verts_, entry_pos_;
    DevBuf<uint16_t> inc_codes_, inc_end_;
    DevBuf<T> dminv_, w_, partial_;
    size_t lds_p_limit_ = 0;  // largest search direction (bytes) a workgroup keeps in LDS
    size_t solve_lds_ = 0;    // of the largest body that fits
    DevBuf<int> vptr_, eptr_, ew_, orig_, vbody_;
    DevBuf<uint32_t> perm_, ecol_wide_;
    DevBuf<uint16_t> ecol_;
    DevBuf<T> eval_, diagA_, dinv_, c0_, mass_, dbc_, origin_;
    DevBuf<T> sn_, sn_old_, prev_, x_, r_, p_, q_;
    DevBuf<int> stats_;
    std::vector<BatchClass> cls_;
};

}  // namespace sbs
