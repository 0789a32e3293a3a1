// Batched PD step: per body and outer iteration i (pdSolver.cu:164-205 with
// the Jacobi-PCG global solve, as the PCG global step of pd_engine):
//   computeLocal (pdUtil.cu:97-145) over the tet chunks of all bodies (one
//   workgroup per chunk, see local_chunk);
//   b = c sn_old + the vertex's partial forces, pinned rows overwritten with
//   DBCX 1e6/h^2 (pdUtil.cu:147-178);
//   Jacobi-PCG warm-started from sn, per component stopping when
//   ||D^-1 r_k|| <= max(tol ||D^-1 r_0||, floor ||D^-1 b||);
//   the Chebyshev recurrence (pdSolver.cu:196-198, pdUtil.cu:216-226);
// the last three by one workgroup per body in one launch.  A body's forces are
// summed in an order of its own and reductions are block reductions in a fixed
// order, so its result does not depend on scheduling.  On the other bodies it
// depends through two orders of summation only: the workgroup size (the
// tuner's, or half a thread per vertex of the largest body) sets that of the
// block sums, and the scene's box, whose Morton curve the assembly follows,
// that of the matrix entries.  See batch_engine.hpp.
#include "batch_engine.hpp"

#include <algorithm>
#include <numeric>
#include <type_traits>

#include "halo_tiles.hpp"
#include "local_chunk.hpp"

namespace sbs {
namespace {

constexpr int kMaxWaves = kRowWaves;  // 1024-thread workgroups at most
constexpr int kTpbB = 256;     // threads of the per-vertex kernels
constexpr int kMaxNarrow = 65535 / 3 - 1;  // vertices of a body whose columns fit 16 bits
constexpr int kFixedPlaces = 6;  // from this many rows per thread on, workgroups have 1,024 threads
constexpr int kBufferFlags = 0x00020000;  // raw buffer descriptor: 32-bit data format, no swizzle
constexpr int kRegWidth = 16;  // widest matrix row kept in registers

template <class T> struct BatchArgs {
    const int* vptr;      // first vertex of each body
    const int* eptr;      // first pair of matrix entries
    const int* ew;        // entries per row
    const int* orig;      // the caller's number of the body
    const int* vbody;     // body of each vertex
    const uint32_t* perm; // vertex -> caller's vertex
    const uint16_t* ecol; // 3 x the column's place in the body
    const uint32_t* ecol_wide;  // the same for bodies past the 16 bits
    const T* eval;
    const T* diagA;
    const T* dinv;
    const T* c0;
    const T* mass;
    const T* dbc;
    const T* origin;      // 3 per body: the body's local origin
    int nv;
    const int* vent_ptr;  // partial forces of vertex i: [vent_ptr[i], vent_ptr[i + 1])
    const T* partial;
    T* X;
    T* V;
    T* XT;
    const T* DBCX;
    T* sn;
    T* sn_old;
    T* prev;
    T* x;                 // vectors of the bodies whose rows do not fit the registers
    T* r;
    T* p;
    T* q;
    int* stats;
    int max_iter;
    int write_x;
    T dt;
    T gravity;
    T wdbc;
    T tol2;
    T floor2;
};

// The Chebyshev step's damping in double (the reference's 0.9 is a double
// literal), then (damped - prev) omega + prev.
template <class T> __device__ __forceinline__ T cheb(T x, T s, T prev, T omega) {
    const T damped = (T)fma(0.9, (double)(x - s), (double)s);
    return fma(damped - prev, omega, prev);
}

// A value of lanes 0, 16 and 32 (components 0, 1, 2) as three uniform values.
__device__ __forceinline__ void from_rows(float v, float (&o)[3]) {
    o[0] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
    o[1] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
    o[2] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
}
__device__ __forceinline__ void from_rows(double v, double (&o)[3]) {
    o[0] = readlane_f64<0>(v);
    o[1] = readlane_f64<16>(v);
    o[2] = readlane_f64<32>(v);
}

// Prologue (pdSolver.cu:154-162): s_n = x + h v +
// f_ext / c, sn_old, prev.  Every vector of a body is held relative to its
// origin o (the step is translation invariant: L o = 0, so A (y + o) = b
// becomes A y = b - c o), so FP32 rounds offsets of the body's size, not of
// its distance from the world origin.
template <class T> __global__ void __launch_bounds__(kTpbB) batch_begin_kernel(BatchArgs<T> a) {
    const int i = (int)(blockIdx.x * kTpbB + threadIdx.x);
    if (i >= a.nv) return;
    const uint32_t g = a.perm[i];
    const T* o = a.origin + 3 * (size_t)a.vbody[i];
    const T fy = -a.gravity * a.mass[i], inv = (T)1 / a.c0[i], dt = a.dt;
    const T s0 = (a.X[3 * (size_t)g] - o[0]) + dt * a.V[3 * (size_t)g];
    const T s1 = (a.X[3 * (size_t)g + 1] - o[1]) + dt * a.V[3 * (size_t)g + 1] + inv * fy;
    const T s2 = (a.X[3 * (size_t)g + 2] - o[2]) + dt * a.V[3 * (size_t)g + 2];
    for (T* out : {a.sn, a.sn_old, a.prev}) {
        out[3 * (size_t)i] = s0;
        out[3 * (size_t)i + 1] = s1;
        out[3 * (size_t)i + 2] = s2;
    }
}

// updateVelPos (pdUtil.cu:180-193) and X <- XTilde (pdSolver.cu:227).
template <class T> __global__ void __launch_bounds__(kTpbB) batch_end_kernel(BatchArgs<T> a) {
    const int i = (int)(blockIdx.x * kTpbB + threadIdx.x);
    if (i >= a.nv) return;
    const T dt_inv = (T)1 / a.dt;
    const uint32_t g = a.perm[i];
    const T* o = a.origin + 3 * (size_t)a.vbody[i];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const T n = a.sn[3 * (size_t)i + k];
        const size_t j = 3 * (size_t)g + k;
        a.V[j] = (n - (a.XT[j] - o[k])) * dt_inv;
        const T xa = n + o[k];
        a.XT[j] = xa;
        if (a.write_x) a.X[j] = xa;
    }
}

template <class T>
__global__ void __launch_bounds__(kChunkTets) batch_local_kernel(
    int nt, const int* __restrict__ chunk_tptr, const uint2* __restrict__ lidx, const int* __restrict__ chunk_vptr,
    const uint32_t* __restrict__ chunk_verts, const uint32_t* __restrict__ entry_pos,
    const uint16_t* __restrict__ inc_codes, const uint16_t* __restrict__ inc_end, const T* __restrict__ dminv,
    const T* __restrict__ w, const T* __restrict__ q, T* __restrict__ partial, int flags) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const unsigned c = xcd_block(blockIdx.x, gridDim.x);
    local_chunk<T>(c, chunk_tptr[c], chunk_tptr[c + 1], nt, lidx, chunk_vptr, chunk_verts, entry_pos, inc_codes,
                   inc_end, dminv, w, partial, flags, smem_raw, [&](int, uint32_t g, T& x, T& y, T& z) {
        x = q[3 * (size_t)g];
        y = q[3 * (size_t)g + 1];
        z = q[3 * (size_t)g + 2];
    });
}

template <class T> constexpr int kPairBatch = sizeof(T) == 4 ? 4 : 2;  // pairs of matrix entries in flight per row

// Right-hand side, PCG solve and Chebyshev step of one body (a workgroup).
// The body's rows are dealt to the threads, row
// k blockDim + tid to the thread's place k < K, and r and q of a row stay in
// registers for the whole solve (the diagonal and x too where they are few:
// !kXg); with kRegs the row's matrix entries as well, read once per solve.
// K = 0 keeps the vectors in memory and takes any number of rows.  With kLds
// the search direction lives in LDS (first the iterate, for A x), so the
// product's neighbour reads are LDS reads.  Matrix entries are stored in
// pairs (two values, two 16-bit columns: a load of 8 and one of 4 bytes for
// FP32), since a load costs its lanes' addresses whatever its width.  What
// bounds it: instructions for small bodies (an iteration of a 280-row body
// took 2.6 us, 700 instructions a wavefront of which the reductions were 280),
// LDS reads and the matrix from L2 for the largest.
template <class T, int K, bool kRegs, bool kLds, bool kXg, bool kWide = false>
__device__ __forceinline__ void batch_solve_body(const BatchArgs<T>& a, int b, int v0, int n, int width, T omega, T* lp,
                                                 double (*red)[12 * kMaxWaves]) {
    static_assert(K > 0 || (!kRegs && kXg), "vectors in memory: no matrix in registers");
    static_assert(!kWide || (K == 0 && !kLds), "wide bodies keep their vectors in memory");
    constexpr int KR = K > 0 ? K : 1;
    constexpr bool kDiag = K > 0 && K * sizeof(T) <= 16;  // the diagonal and its inverse in registers
    typedef T V2 __attribute__((ext_vector_type(2)));
    const size_t ebase = 2 * (size_t)__builtin_amdgcn_readfirstlane(a.eptr[b]);
    // rows k B + tid: with the k B part in a uniform base and the thread's part a
    // 32-bit byte offset, a load needs one address register for all places
    const int B = K >= kFixedPlaces ? 1024 : blockDim.x;
    const unsigned tid = threadIdx.x;
    const int lane = tid & 63, row = lane >> 4;
    const bool live = (int)(tid & ~63u) < n;  // the wavefront has rows
    const int places = K > 0 ? K : (n + B - 1) / B;
    const T o[3] = {a.origin[3 * (size_t)b], a.origin[3 * (size_t)b + 1], a.origin[3 * (size_t)b + 2]};
    T rr[KR][3], qr[KR][3], xr[kXg ? 1 : KR][3], da[kDiag ? KR : 1], dr[kDiag ? KR : 1];
    // (with many rows per thread: one row's loads at a time, all rows' would spill)
    auto fence = [] {
        if constexpr (K >= kFixedPlaces) __builtin_amdgcn_sched_barrier(0);
    };
    const unsigned o1 = tid * (unsigned)sizeof(T), o3 = 3 * o1;
    auto elem = [](auto* base, unsigned byte, int c) -> auto& {
        using E = std::remove_pointer_t<decltype(base)>;
        using Bytes = std::conditional_t<std::is_const_v<E>, const char, char>;
        return reinterpret_cast<E*>(reinterpret_cast<Bytes*>(base) + byte)[c];
    };
    // (readfirstlane where a base is used: hoisted out of the iterations, the
    // places' addresses would take more registers than their vectors)
    auto at = [&](int k) -> size_t { return (size_t)__builtin_amdgcn_readfirstlane(v0 + k * B); };
    auto vec = [&](T (&reg)[KR][3], T* mem, int k, int c) -> T& {
        if constexpr (K > 0) return reg[k][c];
        else return elem(mem + 3 * at(k), o3, c);
    };
    auto X = [&](int k, int c) -> T& {
        if constexpr (kXg) return elem(a.x + 3 * at(k), o3, c);
        else return xr[k][c];
    };
    auto diag = [&](int k) -> T {
        if constexpr (kDiag) return da[k];
        else return elem(a.diagA + at(k), o1, 0);
    };
    auto dinv = [&](int k) -> T {
        if constexpr (kDiag) return dr[k];
        else return elem(a.dinv + at(k), o1, 0);
    };
    // entry j (3 per row) of the vector whose neighbours are read
    T* const pm = kLds ? lp : a.p + 3 * (size_t)v0;
    auto P = [&](int k, int c) -> T& { return (pm + 3 * (size_t)k * B)[3 * tid + c]; };
    // pair j2 of the row in place k: values and 3 x columns.  Buffer loads: the
    // body's base in a descriptor, the pair's and place's part a scalar offset,
    // the thread's one register for all of them (address arithmetic per load
    // was most of the product's instructions, and spilled).
    const unsigned entries = (unsigned)width * (unsigned)n;
    const auto rval = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(a.eval) + ebase, 0, (int)(entries * sizeof(T)),
                                                        kBufferFlags);
    const auto rcol = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.ecol) + ebase, 0, (int)(entries * 2),
                                                        kBufferFlags);
    auto pair = [&](int j2, int k, V2& m, unsigned& c0, unsigned& c1) {
        const unsigned at2 = 2u * ((unsigned)j2 * (unsigned)n + (unsigned)(k * B));
        if constexpr (kWide) {
            const size_t e = ebase + at2 + 2 * (size_t)tid;
            m = *reinterpret_cast<const V2*>(a.eval + e);
            const uint2 c = *reinterpret_cast<const uint2*>(a.ecol_wide + e);
            c0 = c.x;
            c1 = c.y;
        } else {
            if constexpr (sizeof(T) == 4)
                m = __builtin_bit_cast(V2, __builtin_amdgcn_raw_buffer_load_b64(rval, 2 * o1, at2 * sizeof(T), 0));
            else
                m = __builtin_bit_cast(V2, __builtin_amdgcn_raw_buffer_load_b128(rval, 2 * o1, at2 * sizeof(T), 0));
            const unsigned c = __builtin_amdgcn_raw_buffer_load_b32(rcol, 4 * tid, at2 * 2, 0);
            c0 = c & 0xffffu;
            c1 = c >> 16;
        }
    };
    const int pairs = width / 2;  // rows are padded to whole pairs
    V2 mv[kRegs ? KR : 1][kRegWidth / 2];
    unsigned mc[kRegs ? KR : 1][kRegWidth / 2];
    if constexpr (kRegs) {
#pragma unroll
        for (int k = 0; k < KR; ++k) {
            const bool own = k * B + (int)tid < n;
#pragma unroll
            for (int j = 0; j < kRegWidth / 2; ++j) {
                mv[k][j] = V2{(T)0, (T)0};
                mc[k][j] = 0;
                if (j < pairs && own) {
                    unsigned c0, c1;
                    pair(j, k, mv[k][j], c0, c1);
                    mc[k][j] = c0 | (c1 << 16);
                }
            }
        }
    }
    // y += the off-diagonal entries of row (place k) times pm
    auto product = [&](int k, T (&y)[3]) {
        auto add = [&](const V2& m, unsigned c0, unsigned c1) {
#pragma unroll
            for (int c = 0; c < 3; ++c) y[c] += m.x * pm[c0 + c];
#pragma unroll
            for (int c = 0; c < 3; ++c) y[c] += m.y * pm[c1 + c];
        };
        if constexpr (kRegs) {
#pragma unroll
            for (int j = 0; j < kRegWidth / 2; ++j)
                if (j < pairs) add(mv[k][j], mc[k][j] & 0xffffu, mc[k][j] >> 16);
        } else {
            // whole batches, then the rest one pair at a time (no clamped loads)
            auto batch = [&](int j0, auto count) {
                constexpr int NB = decltype(count)::value;
                V2 m[NB];
                unsigned c0[NB], c1[NB];
#pragma unroll
                for (int j = 0; j < NB; ++j) pair(j0 + j, k, m[j], c0[j], c1[j]);
#pragma unroll
                for (int j = 0; j < NB; ++j) add(m[j], c0[j], c1[j]);
            };
            constexpr int NB = kPairBatch<T>;
            int j0 = 0;
#pragma unroll 1
            for (; j0 + NB <= pairs; j0 += NB) batch(j0, std::integral_constant<int, NB>());
#pragma unroll 1
            for (; j0 < pairs; ++j0) batch(j0, std::integral_constant<int, 1>());
        }
    };
#define SBS_ROWS(k) _Pragma("unroll") for (int k = 0; k < places; ++k) if (fence(), k * B + (int)tid < n)
    SBS_ROWS(k) {
        if constexpr (kDiag) {
            da[k] = elem(a.diagA + at(k), o1, 0);
            dr[k] = elem(a.dinv + at(k), o1, 0);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const T s = elem(a.sn + 3 * at(k), o3, c);
            P(k, c) = s;
            X(k, c) = s;
        }
    }
    __syncthreads();
    // right-hand side and the PCG start: x = sn, r = b - A x
    double acc[3][3] = {};  // r.z, z.z, (D^-1 b)^2 per component
    SBS_ROWS(k) {
        const size_t i = at(k) + tid;
        const T cv = a.c0[i];
        T bv[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) bv[c] = cv * a.sn_old[3 * i + c];
        const int e0 = a.vent_ptr[i], e1 = a.vent_ptr[i + 1];
        for (int e = e0; e < e1; e += 4) {
            T f[4][3];
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int c = 0; c < 3; ++c) f[j][c] = a.partial[3 * (size_t)min(e + j, e1 - 1) + c];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (e + j < e1)
#pragma unroll
                    for (int c = 0; c < 3; ++c) bv[c] += f[j][c];
        }
        if (a.dbc[i] > (T)0) {
            // DBCX wdbc - c o (translation of b = DBCX wdbc by A o = c o):
            // (DBCX - o) wdbc - (c - wdbc) o, where both differences are
            // exact (nearby values), so nothing cancels
            const uint32_t g = a.perm[i];
            const T cw = cv - a.wdbc;
#pragma unroll
            for (int c = 0; c < 3; ++c) bv[c] = (a.DBCX[3 * (size_t)g + c] - o[c]) * a.wdbc - cw * o[c];
        }
        const T dA = diag(k), di = dinv(k);
        T Ax[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) Ax[c] = dA * P(k, c);
        product(k, Ax);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const T rk = bv[c] - Ax[c];
            const T zk = di * rk;
            const T dbk = di * bv[c];
            vec(rr, a.r, k, c) = rk;
            acc[0][c] += (double)(rk * zk);
            acc[1][c] += (double)(zk * zk);
            acc[2][c] += (double)(dbk * dbk);
        }
    }
    __syncthreads();  // the iterate has been read
    SBS_ROWS(k) {
#pragma unroll
        for (int c = 0; c < 3; ++c) P(k, c) = dinv(k) * vec(rr, a.r, k, c);
    }
    // the scalars of component c in every lane of row c
    double tot[3];
    block_rows<3>(acc, tot, red[0], live);
    int rb = 1;
    T rz = (T)tot[0];
    const T thr = max(a.tol2 * (T)tot[1], a.floor2 * (T)tot[2]);
    bool act = (T)tot[1] > thr && row < 3;
    int it = 0;
    for (; it < a.max_iter && __ballot(act) != 0ull; ++it) {
        // q = A p and p.q (p of every row was completed before the last barrier)
        double pq[1][3] = {};
        SBS_ROWS(k) {
            const T dA = diag(k);
            T y[3], pv[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                pv[c] = P(k, c);
                y[c] = dA * pv[c];
            }
            product(k, y);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                vec(qr, a.q, k, c) = y[c];
                pq[0][c] += (double)(pv[c] * y[c]);
            }
        }
        double tp[1];
        block_rows<1>(pq, tp, red[rb], live);
        rb ^= 1;
        T alpha[3];
        from_rows(act && tp[0] != 0.0 ? rz / (T)tp[0] : (T)0, alpha);
        // x += alpha p, r -= alpha q, z = D^-1 r
        double nz[2][3] = {};
        SBS_ROWS(k) {
            const T di = dinv(k);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                X(k, c) += alpha[c] * P(k, c);
                T& rv = vec(rr, a.r, k, c);
                const T rk = rv - alpha[c] * vec(qr, a.q, k, c);
                const T zk = di * rk;
                rv = rk;
                nz[0][c] += (double)(rk * zk);
                nz[1][c] += (double)(zk * zk);
            }
        }
        double tn[2];
        block_rows<2>(nz, tn, red[rb], live);
        rb ^= 1;
        T beta[3];
        from_rows(act && rz != (T)0 ? (T)tn[0] / rz : (T)0, beta);
        rz = (T)tn[0];
        SBS_ROWS(k) {
            const T di = dinv(k);
#pragma unroll
            for (int c = 0; c < 3; ++c) P(k, c) = di * vec(rr, a.r, k, c) + beta[c] * P(k, c);
        }
        act = act && (T)tn[1] > thr;
        __syncthreads();
    }
    // Chebyshev (omega = 1 for i <= 10, then the semi-iteration's schedule)
    SBS_ROWS(k) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            T* const sn = a.sn + 3 * at(k);
            T* const prev = a.prev + 3 * at(k);
            T& sv = elem(sn, o3, c);
            T& pv = elem(prev, o3, c);
            const T s = sv, nx = cheb(X(k, c), s, pv, omega);
            pv = s;
            sv = nx;
        }
    }
#undef SBS_ROWS
    const bool cut = __ballot(act) != 0ull;
    if (tid == 0) {
        int* st = a.stats + 4 * (size_t)a.orig[b];
        st[0] += it;
        st[1] += 1;
        st[2] = max(st[2], it);
        st[3] += cut ? 1 : 0;
    }
}

// One workgroup per body, the largest bodies first; the instance by the rows
// per thread (uniform).  All bodies go in one launch: with a launch per size
// class on a stream of its own the classes' launches ran one after the other
// more often than side by side (256 bodies of 3..20 hexes per axis: 4.4 ms a
// step, this form 3.17; 1,024 bodies 7.2 and 6.3).
template <class T>
__global__ void __launch_bounds__(1024) batch_solve_kernel(BatchArgs<T> a, unsigned lds_values, T omega) {
    __shared__ double red[2][12 * kMaxWaves];
    extern __shared__ __align__(16) unsigned char dyn_lds[];
    T* const lp = reinterpret_cast<T*>(dyn_lds);
    const int b = blockIdx.x;
    // (uniform values said to be so: addresses then have scalar bases)
    const int v0 = __builtin_amdgcn_readfirstlane(a.vptr[b]);
    const int n = __builtin_amdgcn_readfirstlane(a.vptr[b + 1]) - v0;
    const int width = __builtin_amdgcn_readfirstlane(a.ew[b]);
    const int places = (n + (int)blockDim.x - 1) / (int)blockDim.x;
    const bool regs = width <= kRegWidth;
    if (n > kMaxNarrow) {
        batch_solve_body<T, 0, false, false, true, true>(a, b, v0, n, width, omega, lp, red);
    } else if (3u * (unsigned)n > lds_values) {
        batch_solve_body<T, 0, false, false, true>(a, b, v0, n, width, omega, lp, red);
    } else if (places <= 1 && regs) {
        batch_solve_body<T, 1, true, true, false>(a, b, v0, n, width, omega, lp, red);
    } else if (places <= 2 && regs && sizeof(T) == 4) {
        if constexpr (sizeof(T) == 4)
            batch_solve_body<T, 2, true, true, false>(a, b, v0, n, width, omega, lp, red);
    } else if (places <= 2) {
        batch_solve_body<T, 2, false, true, false>(a, b, v0, n, width, omega, lp, red);
    } else if (places <= 4) {
        batch_solve_body<T, 4, false, true, (sizeof(T) > 4)>(a, b, v0, n, width, omega, lp, red);
    } else if (places <= 6 && blockDim.x == 1024 && sizeof(T) == 4) {
        if constexpr (sizeof(T) == 4)
            batch_solve_body<T, 6, false, true, true>(a, b, v0, n, width, omega, lp, red);
    } else if (places <= 10 && blockDim.x == 1024 && sizeof(T) == 4) {
        if constexpr (sizeof(T) == 4)
            batch_solve_body<T, 10, false, true, true>(a, b, v0, n, width, omega, lp, red);
    } else {
        batch_solve_body<T, 0, false, true, true>(a, b, v0, n, width, omega, lp, red);
    }
}

__global__ void zero_int_kernel(int n, int* p) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0;
}

template <class T> void upload(DevBuf<T>& d, const std::vector<T>& h) {
    d.alloc(std::max<size_t>(h.size(), 1));
    if (!h.empty()) SBS_HIP(hipMemcpy(d.get(), h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
}

int round64(int n) { return std::max(64, std::min(1024, (n + 63) / 64 * 64)); }

}  // namespace

template <class T> BatchEngine<T>::BatchEngine(const BatchSystem<T>& s) {
    nv_ = s.nv;
    nt_ = s.nt;
    SBS_REQUIRE(nv_ > 0, "batched PD: empty scene");
    // bodies: connected components of the tet mesh (union-find over vertices)
    std::vector<int> parent(nv_);
    std::iota(parent.begin(), parent.end(), 0);
    auto find = [&](int v) {
        while (parent[v] != v) v = parent[v] = parent[parent[v]];
        return v;
    };
    for (int t = 0; t < nt_; ++t)
        for (int k = 1; k < 4; ++k) {
            const int a = find((int)s.tets[4 * (size_t)t]), b = find((int)s.tets[4 * (size_t)t + k]);
            if (a != b) parent[std::max(a, b)] = std::min(a, b);
        }
    std::vector<int> body_of_root(nv_, -1), number(nv_);
    nb_ = 0;
    for (int v = 0; v < nv_; ++v) {  // bodies numbered by their first vertex
        const int r = find(v);
        if (body_of_root[r] < 0) body_of_root[r] = nb_++;
        number[v] = body_of_root[r];
    }
    verts_h_.assign(nb_, 0);
    tets_h_.assign(nb_, 0);
    for (int v = 0; v < nv_; ++v) verts_h_[number[v]]++;
    for (int t = 0; t < nt_; ++t) tets_h_[number[s.tets[4 * (size_t)t]]]++;
    // bodies are held largest first (a launch's workgroups start in that
    // order); the reported classes end at the rows that one, two and four
    // places of 1,024 threads take, and where columns need 32 bits
    std::vector<int> order(nb_);  // place -> the caller's number
    std::iota(order.begin(), order.end(), 0);
    std::sort(order.begin(), order.end(),
              [&](int x, int y) { return verts_h_[x] != verts_h_[y] ? verts_h_[x] > verts_h_[y] : x < y; });
    max_verts_ = verts_h_[order[0]];
    const int bounds[] = {0, 1024, 2048, 4096, kMaxNarrow, 0x7fffffff};
    for (int c = 0; c < 5; ++c) {
        BatchClass bc;
        for (int b = 0; b < nb_; ++b) {
            if (verts_h_[b] <= bounds[c] || verts_h_[b] > bounds[c + 1]) continue;
            bc.min_tets = bc.bodies ? std::min(bc.min_tets, tets_h_[b]) : tets_h_[b];
            bc.max_tets = std::max(bc.max_tets, tets_h_[b]);
            ++bc.bodies;
        }
        if (bc.bodies) cls_.push_back(bc);
    }
    set_threads(round64((max_verts_ + 1) / 2));  // until the tuner chooses
    std::vector<int> place(nb_);
    for (int k = 0; k < nb_; ++k) place[order[k]] = k;
    // internal vertex order: body by body, caller order inside a body
    std::vector<int> vptr(nb_ + 1, 0);
    for (int k = 0; k < nb_; ++k) vptr[k + 1] = vptr[k] + verts_h_[order[k]];
    std::vector<uint32_t> perm(nv_);
    std::vector<int> inv(nv_), vbody(nv_), fill(vptr.begin(), vptr.end() - 1);
    for (int v = 0; v < nv_; ++v) {
        const int k = place[number[v]], i = fill[k]++;
        perm[i] = (uint32_t)v;
        inv[v] = i;
        vbody[i] = k;
    }
    // per-body ELL of the off-diagonal entries, in pairs (entries 2 j and
    // 2 j + 1 of a row side by side, pair-major inside the body, padded with
    // the row's own place and value 0); per-vertex constants
    std::vector<int> eptr(nb_ + 1, 0), ew(nb_, 0);
    std::vector<T> diagA(nv_), dinv(nv_), c0(nv_), mass(nv_), dbc(nv_);
    for (int i = 0; i < nv_; ++i) {
        const int v = (int)perm[i];
        diagA[i] = s.diagA[v];
        c0[i] = s.c0[v];
        mass[i] = s.mass[v];
        dbc[i] = s.dbc[v];
        dinv[i] = (T)1 / s.diagA[v];
        ew[vbody[i]] = std::max(ew[vbody[i]], s.rowptr[v + 1] - s.rowptr[v] - 1);
    }
    // whole pairs; whole batches of pairs where the rows are read in every
    // iteration (a body past the rows that fit the registers)
    for (int b = 0; b < nb_; ++b) {
        const int unit = vptr[b + 1] - vptr[b] > (int)(8192 / sizeof(T)) ? 2 * kPairBatch<T> : 2;
        ew[b] = (ew[b] + unit - 1) / unit * unit;
    }
    size_t entries = 0;
    bool wide = false;
    for (int b = 0; b < nb_; ++b) {
        const size_t n = (size_t)(vptr[b + 1] - vptr[b]);
        wide = wide || n > (size_t)kMaxNarrow;
        entries += n * (size_t)ew[b];
        SBS_REQUIRE(entries < ((size_t)1 << 32), "batched PD: scene too large");
        eptr[b + 1] = (int)(entries / 2);
    }
    std::vector<uint16_t> ecol(std::max<size_t>(entries, 1));
    std::vector<uint32_t> ecol_wide(wide ? entries : 0);
    std::vector<T> eval(std::max<size_t>(entries, 1), (T)0);
    for (int b = 0; b < nb_; ++b) {
        const int n = vptr[b + 1] - vptr[b];
        auto place_of = [&](int j, int il) { return 2 * ((size_t)eptr[b] + (size_t)(j / 2) * n + il) + (j & 1); };
        auto set_col = [&](size_t pos, int col) {
            if (n > kMaxNarrow) ecol_wide[pos] = (uint32_t)(3 * col);
            else ecol[pos] = (uint16_t)(3 * col);
        };
        for (int il = 0; il < n; ++il) {
            const int v = (int)perm[vptr[b] + il];
            int j = 0;
            for (int e = s.rowptr[v]; e < s.rowptr[v + 1]; ++e) {
                if (s.col[e] == v) continue;
                const size_t pos = place_of(j, il);
                set_col(pos, inv[s.col[e]] - vptr[b]);
                eval[pos] = s.val[e];
                ++j;
            }
            for (; j < ew[b]; ++j) set_col(place_of(j, il), il);
        }
    }
    // each body's origin: the rest position of its first vertex
    std::vector<T> origin(3 * (size_t)nb_);
    for (int b = 0; b < nb_; ++b)
        for (int k = 0; k < 3; ++k) origin[3 * (size_t)b + k] = s.x0[3 * (size_t)perm[vptr[b]] + k];
    upload(origin_, origin);
    upload(vptr_, vptr);
    upload(eptr_, eptr);
    upload(ew_, ew);
    upload(orig_, order);
    upload(vbody_, vbody);
    upload(perm_, perm);
    upload(ecol_, ecol);
    if (wide) upload(ecol_wide_, ecol_wide);
    upload(eval_, eval);
    upload(diagA_, diagA);
    upload(dinv_, dinv);
    upload(c0_, c0);
    upload(mass_, mass);
    upload(dbc_, dbc);
    const size_t n3 = 3 * (size_t)nv_;
    sn_.alloc(n3); sn_old_.alloc(n3); prev_.alloc(n3); x_.alloc(n3); r_.alloc(n3); p_.alloc(n3); q_.alloc(n3);
    stats_.alloc(4 * (size_t)nb_);
    reset_stats();
    // the tets in chunks: a body's tets along a Morton curve of the rest
    // centroids, cut every kChunkTets; what is left of each body goes whole
    // into shared chunks at the end.  So the tets whose forces a chunk sums for
    // a vertex, and the order of a vertex's partial forces, are the body's own,
    // whatever other bodies there are.
    std::vector<std::vector<int>> tets_of(nb_);
    for (int t = 0; t < nt_; ++t) tets_of[place[number[s.tets[4 * (size_t)t]]]].push_back(t);
    std::vector<int> seq, starts;
    std::vector<std::vector<int>> rest(nb_);
    std::vector<std::pair<uint32_t, int>> key;
    for (int b = 0; b < nb_; ++b) {
        double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
        for (int i = vptr[b]; i < vptr[b + 1]; ++i)
            for (int k = 0; k < 3; ++k) {
                lo[k] = std::min(lo[k], (double)s.x0[3 * (size_t)perm[i] + k]);
                hi[k] = std::max(hi[k], (double)s.x0[3 * (size_t)perm[i] + k]);
            }
        key.clear();
        for (int t : tets_of[b]) {
            double cen[3] = {0, 0, 0};
            for (int j = 0; j < 4; ++j)
                for (int k = 0; k < 3; ++k) cen[k] += 0.25 * (double)s.x0[3 * (size_t)s.tets[4 * (size_t)t + j] + k];
            key.emplace_back(morton_code(cen, lo, hi), t);
        }
        std::sort(key.begin(), key.end());
        const size_t whole = key.size() / kChunkTets * kChunkTets;
        for (size_t i = 0; i < whole; ++i) {
            if (i % kChunkTets == 0) starts.push_back((int)seq.size());
            seq.push_back(key[i].second);
        }
        for (size_t i = whole; i < key.size(); ++i) rest[b].push_back(key[i].second);
    }
    // largest rests first, each into the shared chunk with the least room that
    // takes it (taken in body order they would leave a quarter of them idle)
    std::vector<int> by_rest(nb_);
    std::iota(by_rest.begin(), by_rest.end(), 0);
    std::stable_sort(by_rest.begin(), by_rest.end(), [&](int x, int y) { return rest[x].size() > rest[y].size(); });
    std::vector<std::vector<int>> shared, with_room(kChunkTets + 1);  // with_room[r]: shared chunks with room for r more
    for (int b : by_rest) {
        size_t r = rest[b].size();
        if (r == 0) break;
        while (r < with_room.size() && with_room[r].empty()) ++r;
        int c = (int)shared.size();
        if (r < with_room.size()) {
            c = with_room[r].back();
            with_room[r].pop_back();
        } else {
            shared.emplace_back();
        }
        shared[c].insert(shared[c].end(), rest[b].begin(), rest[b].end());
        with_room[kChunkTets - shared[c].size()].push_back(c);
    }
    for (const auto& c : shared) {
        starts.push_back((int)seq.size());
        seq.insert(seq.end(), c.begin(), c.end());
    }
    starts.push_back((int)seq.size());
    const int nt = (int)seq.size();
    std::vector<uint32_t> tv(4 * (size_t)nt);
    std::vector<T> dm(9 * (size_t)nt), w(nt);
    for (int i = 0; i < nt; ++i) {
        const size_t t = (size_t)seq[i];
        for (int j = 0; j < 4; ++j) tv[4 * (size_t)i + j] = (uint32_t)(inv[s.tets[4 * t + j]]);
        for (int k = 0; k < 9; ++k) dm[(size_t)k * nt + i] = s.dminv[9 * t + k];
        w[i] = s.w[t];
    }
    const ChunkLists ch = build_chunk_lists(nv_, tv, starts);
    chunks_ = ch.chunks;
    local_lds_ = chunk_lds_bytes<T>(ch.max_verts);
    SBS_REQUIRE(local_lds_ <= 64 * 1024, "batched PD: chunk vertex list exceeds LDS");
    upload(lidx_, ch.lidx);
    upload(chunk_tptr_, starts);
    upload(chunk_vptr_, ch.vptr);
    upload(chunk_verts_, ch.verts);
    upload(entry_pos_, ch.pos);
    upload(inc_codes_, ch.inc_codes);
    upload(inc_end_, ch.inc_end);
    upload(vent_ptr_, ch.vert_ptr);
    upload(dminv_, dm);
    upload(w_, w);
    partial_.alloc(std::max<size_t>(3 * ch.verts.size(), 1));
    // LDS a workgroup may take for the search direction: the device's per-block
    // limit less the kernel's static 2.3 KB (64 KB unless it reports more)
    int dev = 0, lim = 0;
    SBS_HIP(hipGetDevice(&dev));
    if (hipDeviceGetAttribute(&lim, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || lim <= 0)
        lim = 64 * 1024;
    lds_p_limit_ = (size_t)lim - 4096;
    SBS_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&batch_solve_kernel<T>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_p_limit_));
    // the largest body whose direction fits
    for (int k = 0; k < nb_; ++k) {
        const size_t need = 3 * (size_t)verts_h_[order[k]] * sizeof(T);
        if (need <= lds_p_limit_) {
            solve_lds_ = need;
            break;
        }
    }
}

template <class T> void BatchEngine<T>::reset_stats() {
    hipLaunchKernelGGL(zero_int_kernel, dim3(ceil_div(4 * (size_t)nb_, 256)), dim3(256), 0, nullptr, 4 * nb_,
                       stats_.get());
    SBS_HIP(hipGetLastError());
    SBS_HIP(hipDeviceSynchronize());
}

template <class T> std::vector<BatchBody> BatchEngine<T>::body_stats() {
    SBS_HIP(hipDeviceSynchronize());
    std::vector<int> h(4 * (size_t)nb_);
    SBS_HIP(hipMemcpy(h.data(), stats_.get(), h.size() * sizeof(int), hipMemcpyDeviceToHost));
    std::vector<BatchBody> out(nb_);
    for (int b = 0; b < nb_; ++b) {
        out[b].verts = verts_h_[b];
        out[b].tets = tets_h_[b];
        out[b].iterations = h[4 * b];
        out[b].solves = h[4 * b + 1];
        out[b].max_per_solve = h[4 * b + 2];
        out[b].unconverged = h[4 * b + 3];
    }
    return out;
}

template <class T> void BatchEngine<T>::set_threads(int threads) {
    threads_ = threads;
    for (BatchClass& c : cls_) c.threads = threads;
}

template <class T>
void BatchEngine<T>::step(T* X, T* V, T* XT, const T* DBCX, const BatchParams& p, hipStream_t stream) {
    SBS_REQUIRE(p.iterations >= 0 && p.pcg_max_iter >= 1 && p.dt > 0, "batched PD: invalid parameters");
    launch_step(X, V, XT, DBCX, p, stream, threads_);
}

template <class T>
void BatchEngine<T>::launch_step(T* X, T* V, T* XT, const T* DBCX, const BatchParams& p, hipStream_t s, int threads) {
    SBS_REQUIRE(threads >= 64 && threads <= 64 * kMaxWaves && threads % 64 == 0,
                "batched PD: workgroup size must be a multiple of 64 up to 1024");
    BatchArgs<T> a;
    a.vptr = vptr_.get();
    a.eptr = eptr_.get();
    a.ew = ew_.get();
    a.orig = orig_.get();
    a.vbody = vbody_.get();
    a.perm = perm_.get();
    a.ecol = ecol_.get();
    a.ecol_wide = ecol_wide_.get();
    a.eval = eval_.get();
    a.diagA = diagA_.get();
    a.dinv = dinv_.get();
    a.c0 = c0_.get();
    a.mass = mass_.get();
    a.dbc = dbc_.get();
    a.origin = origin_.get();
    a.nv = nv_;
    a.vent_ptr = vent_ptr_.get();
    a.partial = partial_.get();
    a.X = X;
    a.V = V;
    a.XT = XT;
    a.DBCX = DBCX;
    a.sn = sn_.get();
    a.sn_old = sn_old_.get();
    a.prev = prev_.get();
    a.x = x_.get();
    a.r = r_.get();
    a.p = p_.get();
    a.q = q_.get();
    a.stats = stats_.get();
    a.max_iter = p.pcg_max_iter;
    a.write_x = p.write_x ? 1 : 0;
    a.dt = (T)p.dt;
    a.gravity = (T)p.gravity;
    const T dt_inv = (T)1 / (T)p.dt;
    a.wdbc = (T)1e6 * (dt_inv * dt_inv);
    a.tol2 = (T)(p.pcg_tol * p.pcg_tol);
    a.floor2 = (T)(p.pcg_floor * p.pcg_floor);
    const unsigned vb = ceil_div((size_t)nv_, kTpbB);
    hipLaunchKernelGGL(batch_begin_kernel<T>, dim3(vb), dim3(kTpbB), 0, s, a);
    const T rho = (T)p.rho;
    T omega = 1;
    for (int i = 0; i < p.iterations; ++i) {
        if (chunks_ > 0)
            hipLaunchKernelGGL(batch_local_kernel<T>, dim3(chunks_), dim3(kChunkTets), local_lds_, s, nt_,
                               (const int*)chunk_tptr_.get(), lidx_.get(),
                               chunk_vptr_.get(), chunk_verts_.get(), entry_pos_.get(), inc_codes_.get(),
                               inc_end_.get(), dminv_.get(), w_.get(), (const T*)sn_.get(), partial_.get(),
                               p.polar ? kLocalPolar : 0);
        if (i <= 10) omega = 1;
        else if (i == 11) omega = (T)2 / ((T)2 - rho * rho);
        else omega = (T)4 / ((T)4 - rho * rho * omega);
        hipLaunchKernelGGL(batch_solve_kernel<T>, dim3(nb_), dim3(threads), solve_lds_, s, a,
                           (unsigned)(solve_lds_ / sizeof(T)), omega);
    }
    hipLaunchKernelGGL(batch_end_kernel<T>, dim3(vb), dim3(kTpbB), 0, s, a);
    SBS_HIP(hipGetLastError());
}

template <class T>
void BatchEngine<T>::autotune(const T* X, const T* V, const T* DBCX, const BatchParams& p, hipStream_t stream) {
    const size_t n3 = 3 * (size_t)nv_;
    DevBuf<T> xc(n3), vc(n3), tc(n3);
    hipEvent_t e0, e1;
    SBS_HIP(hipEventCreate(&e0));
    SBS_HIP(hipEventCreate(&e1));
    std::vector<std::pair<int, double>> tried;
    double best = 1e300;
    int best_t = threads_;
    for (int th : {64, 128, 256, 512, 1024}) {
        if (th > 64 && th / 2 >= round64(max_verts_)) continue;              // more threads than rows: no gain
        if (th < 1024 && (max_verts_ + th - 1) / th > 4) continue;           // rows would leave the registers
        double ms_best = 1e300;
        for (int rep = 0; rep < 3; ++rep) {  // one warm-up, then the faster of two
            SBS_HIP(hipMemcpyAsync(xc.get(), X, n3 * sizeof(T), hipMemcpyDeviceToDevice, stream));
            SBS_HIP(hipMemcpyAsync(vc.get(), V, n3 * sizeof(T), hipMemcpyDeviceToDevice, stream));
            SBS_HIP(hipMemcpyAsync(tc.get(), X, n3 * sizeof(T), hipMemcpyDeviceToDevice, stream));
            SBS_HIP(hipEventRecord(e0, stream));
            launch_step(xc.get(), vc.get(), tc.get(), DBCX, p, stream, th);
            SBS_HIP(hipEventRecord(e1, stream));
            SBS_HIP(hipEventSynchronize(e1));
            float ms = 0;
            SBS_HIP(hipEventElapsedTime(&ms, e0, e1));
            if (rep > 0) ms_best = std::min(ms_best, (double)ms);
        }
        tried.emplace_back(th, ms_best);
        if (ms_best < best) {
            best = ms_best;
            best_t = th;
        }
    }
    for (BatchClass& c : cls_) c.tried = tried;
    set_threads(best_t);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    reset_stats();
}

template class BatchEngine<float>;
template class BatchEngine<double>;

}  // namespace sbs
