// Explicit inverse of the prefactored PD matrix for the direct global solve.
//
// The direct modes solve one small system many times (every local/global
// iteration of every step) with the same matrix.  Triangular solves with its
// band factor are a chain of dependent 64-row blocks that three workgroups
// walk while the rest of the GPU idles; the product with the explicit inverse
// has no chain, so it runs on every CU at the memory's rate.  The inverse is
// computed once from the FP64 factor, column by column (L y = e_j, L^T x = y)
// in FP64 on the GPU, and rounded once to the solve precision.
#pragma once

#include <vector>

#include "band_factor.hpp"
#include "common.hpp"

namespace sbs {

// The outer loop's end of iteration (computeError, pdSolver.cu:243-253, and
// the early exit, :164) done by the product itself: sum (prev - x)^2, sn and
// prev take x, and the last workgroup decides.
template <class T> struct OuterStep {
    T* sn;
    T* prev;
    double* err;   // mean squared difference of the last iteration
    int* done;     // set when its square root falls below tol
    double tol;
};

template <class T> class InverseOperator {
public:
    // Whether the inverse of the systems (row ranges sys[s] .. sys[s+1]) takes no
    // more than most_bytes nor a quarter of the free memory: the rule by which
    // the product replaces the triangular solves, see its comment.
    static bool fits(const std::vector<int>& sys, size_t most_bytes);
    void setup(const BandFactor& f, const std::vector<int>& sys, hipStream_t stream);
    bool ready() const { return n_ > 0; }
    size_t bytes() const { return inv_.bytes(); }
    // The right-hand side's place: component c of vertex v at
    // rhs()[c * stride() + pos()[v]] (padding between systems stays 0).
    T* rhs() const { return rhs_.get(); }
    const int* pos() const { return pos_.get(); }
    int stride() const { return npad_; }
    // x = A^-1 rhs() for the 3 components (x interleaved, vertex order);
    // returns early when *skip != 0 (device flag, may be null).
    void apply(T* x, hipStream_t stream, const int* skip) const;
    // The same into sn and prev with the outer loop's error and decision.
    void apply_outer(const OuterStep<T>& o, hipStream_t stream, const int* skip) const;
    // The interleaved b (vertex order) into rhs().
    void load_rhs(const T* b, hipStream_t stream, const int* skip) const;

private:
    int n_ = 0, npad_ = 0;
    unsigned groups_ = 0;
    DevBuf<T> inv_;            // per system n_s rows of ld_s values, factor order
    DevBuf<T> rhs_;            // 3 x npad
    DevBuf<int> pos_, vert_;   // vertex -> padded position; padded position -> vertex
    DevBuf<int> job_;          // per workgroup: first padded position, rows, ld, first row
    DevBuf<long long> job_off_;  // per workgroup: first value of its first row
    DevBuf<double> parts_;     // per workgroup, then per stripe: its sum of squared differences
    DevBuf<unsigned> ticket_;  // stripes, then per stripe workgroups, that have stored theirs
};

}  // namespace sbs
