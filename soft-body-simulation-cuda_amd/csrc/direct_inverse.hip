// Explicit inverse of the prefactored PD matrix: its columns from the FP64
// band factor, and the product that replaces the triangular solves.
#include "direct_inverse.hpp"

#include <algorithm>

namespace sbs {

namespace {

constexpr int kRowsPer = 8;       // rows of the inverse per workgroup of the product
constexpr int kThreads = 256;
constexpr int kStripCols = 64;    // columns of one inversion workgroup (one wavefront)
// The outer loop's decision is taken by the workgroup that passes a ticket last.
// Past kOneTicket workgroups the ticket is a tree of kStripes, since atomics on
// one word follow each other at 11 ns each; up to there the second level costs
// more (an iteration of one 125-row body 16.3 us with one ticket, 17.2 with the
// tree; 16 bodies of 729 rows 41 and 24; 1,024 of 64 rows about 130 and 40).
constexpr unsigned kOneTicket = 64;
constexpr unsigned kStripes = 32;
constexpr unsigned kTicketPitch = 32;  // words: a cache line of its own per ticket
constexpr int kPadTo = 4;         // rows are padded to whole 4-value loads
constexpr size_t kScratchBytes = (size_t)4 << 30;   // FP64 columns in flight while inverting

// One 64-column strip of a system's inverse, one column per lane.  Rows go in
// blocks of kBlkRows: each wavefront takes every kStripWaves-th of the rows
// the block depends on, loads that row's 64 values once and adds its product
// to all the block's rows (the factor entries are the same for every lane and
// consecutive: scalar loads), then wavefront 0 sums the wavefronts' parts and
// solves the block's own triangle in registers.  Rows above the strip's first
// column are 0 in the forward sweep and skipped.  `Lr` holds the factor by
// rows (entry d of row i: L[i][i-d]), `Uc` by columns (entry d of column i:
// L[i+d][i]), both zero past the band so a block reads kBlkRows entries
// unconditionally; rinv is 1 / L[i][i].  Run once per factorisation; one row
// at a time with one wavefront per strip took 75 ms for 3,360 rows of half
// bandwidth 225, this order 10.5 ms.
constexpr int kBlkRows = 16;
constexpr int kStripWaves = 4;
struct StripJob {
    int s0, n, col0, ld;
    long long y_off, out_off;
};
template <class T>
__global__ void __launch_bounds__(64 * kStripWaves) inverse_strip_kernel(
    const StripJob* __restrict__ jobs, int bw, int lw, const double* __restrict__ Lr, const double* __restrict__ Uc,
    const double* __restrict__ rinv, double* Y, T* __restrict__ out) {
    __shared__ double part[kStripWaves][kBlkRows][kStripCols];
    const StripJob j = jobs[blockIdx.x];
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), col = j.col0 + lane;
    double* y = Y + j.y_off + lane;
    double acc[kBlkRows], blk[kBlkRows];
    auto share = [&]() {
#pragma unroll
        for (int r = 0; r < kBlkRows; ++r) part[wid][r][lane] = acc[r];
        __syncthreads();
    };
    auto total = [&](int r) {
        double s = part[0][r][lane];
#pragma unroll
        for (int w = 1; w < kStripWaves; ++w) s += part[w][r][lane];
        return s;
    };
    for (int i0 = j.col0; i0 < j.n; i0 += kBlkRows) {
#pragma unroll
        for (int r = 0; r < kBlkRows; ++r) acc[r] = 0.0;
        for (int k = max(i0 - bw, j.col0) + wid; k < i0; k += kStripWaves) {
            const double yk = y[(size_t)k * kStripCols];
            const double* C = Uc + (size_t)(j.s0 + k) * lw + (i0 - k);
#pragma unroll
            for (int r = 0; r < kBlkRows; ++r) acc[r] -= C[r] * yk;
        }
        share();
        if (wid == 0) {
#pragma unroll
            for (int r = 0; r < kBlkRows; ++r) {
                double s = (i0 + r == col ? 1.0 : 0.0) + total(r);
#pragma unroll
                for (int q = 0; q < r; ++q) s -= Uc[(size_t)(j.s0 + i0 + q) * lw + (r - q)] * blk[q];
                blk[r] = s * rinv[j.s0 + i0 + r];
                if (i0 + r < j.n) y[(size_t)(i0 + r) * kStripCols] = blk[r];
            }
        }
        __syncthreads();
    }
    for (int i0 = (j.n - 1) / kBlkRows * kBlkRows; i0 >= 0; i0 -= kBlkRows) {
#pragma unroll
        for (int r = 0; r < kBlkRows; ++r) acc[r] = 0.0;
        for (int k = i0 + kBlkRows + wid; k <= min(j.n - 1, i0 + kBlkRows - 1 + bw); k += kStripWaves) {
            const double xk = y[(size_t)k * kStripCols];
            const double* C = Lr + (size_t)(j.s0 + k) * lw + (k - i0 - (kBlkRows - 1));
#pragma unroll
            for (int r = 0; r < kBlkRows; ++r) acc[r] -= C[kBlkRows - 1 - r] * xk;
        }
        share();
        if (wid == 0) {
#pragma unroll
            for (int r = kBlkRows - 1; r >= 0; --r) {
                const int i = i0 + r;
                double s = total(r);
                if (i >= j.col0 && i < j.n) s += y[(size_t)i * kStripCols];
#pragma unroll
                for (int q = r + 1; q < kBlkRows; ++q) s -= Lr[(size_t)(j.s0 + i0 + q) * lw + (q - r)] * blk[q];
                blk[r] = i < j.n ? s * rinv[j.s0 + i] : 0.0;
                if (i < j.n) {
                    y[(size_t)i * kStripCols] = blk[r];
                    if (col < j.ld) out[j.out_off + (long long)i * j.ld + col] = col < j.n ? (T)blk[r] : (T)0;
                }
            }
        }
        __syncthreads();
    }
}

template <class T>
__global__ void permute_rhs_kernel(int n, const T* __restrict__ b, const int* __restrict__ pos, int stride,
                                   T* __restrict__ out, const int* __restrict__ skip) {
    if (skip && *skip) return;
    const int v = blockIdx.x * kThreads + threadIdx.x;
    if (v >= n) return;
    const int p = pos[v];
#pragma unroll
    for (int c = 0; c < 3; ++c) out[(size_t)c * stride + p] = b[3 * (size_t)v + c];
}

// Sum over each row of 16 lanes, in the solve precision (DPP moves).
__device__ __forceinline__ float row16_sum(float v) {
#define SBS_DPP_ADD(CTRL) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true))
    SBS_DPP_ADD(0xB1);
    SBS_DPP_ADD(0x4E);
    SBS_DPP_ADD(0x141);
    SBS_DPP_ADD(0x140);
#undef SBS_DPP_ADD
    return v;
}
__device__ __forceinline__ double row16_sum(double v) { return row16_total(v); }

// Called by wavefront 0 of `members` workgroups: v (the same in every lane) into
// the slot; true in the workgroup that comes last, which may then read all
// slots.  The exchange's result is waited for, so the slot is written where all
// XCDs see it before the ticket counts it; a release fence in every workgroup
// instead writes back its XCD's L2 each time (32 bodies of 2,197 rows: 616 us
// an iteration, this form 146).
__device__ __forceinline__ bool passed_last(double v, double* slot, unsigned* ticket, unsigned members) {
    unsigned before = 0;
    if (threadIdx.x == 0) {
        double old = __hip_atomic_exchange(slot, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(old)::"memory");
        before = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (__builtin_amdgcn_readfirstlane(before) != members - 1) return false;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    if (threadIdx.x == 0) *ticket = 0;  // for the next launch
    return true;
}
// Sum of `members` slots, `pitch` apart, in every lane of the wavefront.
__device__ __forceinline__ double slot_sum(const double* slots, unsigned pitch, unsigned members) {
    double s = 0.0;
    for (unsigned k = threadIdx.x; k < members; k += 64)
        s += __hip_atomic_load(&slots[(size_t)k * pitch], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return wave_total(s);
}

// kRowsPer rows of a system's inverse times its three right-hand sides.  Each
// thread takes 4 consecutive columns of every 1,024: one 4-value load per
// row and right-hand side, kRowsPer + 3 of them in flight.  Per thread the
// products are summed in the solve precision (n / 1024 of them), then 16
// lanes, then the 16 row totals in double.  A launch that runs (not skipped by
// the early exit): 2.1 MB for 729 rows in 7.7 us, 45 MB for 3,360 rows in 13.7
// (3.3 TB/s), 1.9 GB for 21,952 rows in 340 (5.7 TB/s: HBM bound there, below
// it the launch, one round of loads and the ticket).  With the outer loop's
// error and decision taken along (two launches of 4 us each before), an
// iteration is three launches.
template <class T, bool kOuter>
__global__ void __launch_bounds__(kThreads) inverse_apply_kernel(
    const int4* __restrict__ job, const long long* __restrict__ job_off, const T* __restrict__ inv,
    const T* __restrict__ rhs, int stride, const int* __restrict__ vert, T* __restrict__ x, OuterStep<T> o,
    int nv, double* parts, unsigned* ticket, const int* __restrict__ skip) {
    if (skip && *skip) return;
    typedef T V4 __attribute__((ext_vector_type(4)));
    constexpr int kVals = 3 * kRowsPer, kRows16 = kThreads / 16;
    __shared__ double red[kVals][kRows16 + 1];
    const int4 j = job[blockIdx.x];  // first padded position of the system, its rows, ld, first row here
    const T* __restrict__ A = inv + job_off[blockIdx.x];
    const int ld = j.z, rows = min(kRowsPer, j.y - j.w);
    const T* __restrict__ b = rhs + j.x;
    T acc[kRowsPer][3];
#pragma unroll
    for (int r = 0; r < kRowsPer; ++r) acc[r][0] = acc[r][1] = acc[r][2] = (T)0;
    for (int k = 4 * threadIdx.x; k < ld; k += 4 * kThreads) {
        V4 a[kRowsPer], bv[3];
#pragma unroll
        for (int r = 0; r < kRowsPer; ++r)
            a[r] = *reinterpret_cast<const V4*>(A + (size_t)min(r, rows - 1) * ld + k);
#pragma unroll
        for (int c = 0; c < 3; ++c) bv[c] = *reinterpret_cast<const V4*>(b + (size_t)c * stride + k);
#pragma unroll
        for (int r = 0; r < kRowsPer; ++r)
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[r][c] += a[r][e] * bv[c][e];
    }
    const int tid = threadIdx.x;
#pragma unroll
    for (int r = 0; r < kRowsPer; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const T s = row16_sum(acc[r][c]);
            if ((tid & 15) == 0) red[3 * r + c][tid >> 4] = (double)s;
        }
    __syncthreads();
    if (tid >= 64) return;
    double sq = 0.0;
    if (tid < 3 * rows) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < kRows16; ++k) s += red[tid][k];
        const T xv = (T)s;
        const size_t i = 3 * (size_t)vert[j.x + j.w + tid / 3] + tid % 3;
        if constexpr (kOuter) {
            const T d = o.prev[i] - xv;
            sq = (double)(d * d);
            o.sn[i] = xv;
            o.prev[i] = xv;
        } else {
            x[i] = xv;
        }
    }
    if constexpr (kOuter) {
        const double total = wave_total(sq);
        // the workgroup that passes its stripe's ticket last adds the stripe's
        // sums, and the stripe that passes the common ticket last adds those
        // (one level up to kOneTicket workgroups), each in index order
        const unsigned groups = gridDim.x, stripes = groups <= kOneTicket ? 1u : kStripes;
        const unsigned st = blockIdx.x % stripes, members = (groups - st + stripes - 1) / stripes;
        double sum = total;
        if (!passed_last(sum, &parts[blockIdx.x], &ticket[kTicketPitch * (1 + st)], members)) return;
        sum = slot_sum(parts + st, stripes, members);
        if (stripes > 1) {
            if (!passed_last(sum, &parts[groups + st], ticket, stripes)) return;
            sum = slot_sum(parts + groups, 1, stripes);
        }
        if (tid == 0) {
            const double err = sum / (3.0 * (double)nv);
            *o.err = err;
            *o.done = !(sqrt(err) >= o.tol);
        }
    }
}

int padded(int n) { return (n + kPadTo - 1) / kPadTo * kPadTo; }

}  // namespace

// An iteration of the outer loop (local step, right-hand side, solve, error,
// decision) with the triangular solves and with the product, FP32, us: one
// body of 8 rows 20.1 and 13.3, of 1,000 rows 193 and 17.9, of 21,952 rows
// 10,891 and 359; 1,024 bodies of 64 rows 106 and 42, of 343 rows 437 and 214,
// of 729 rows 1,046 and 594; 128 bodies of 2,197 rows 619 and 547 (FP64: 22.3
// and 14.3, 227 and 20.2, 19,174 and 687; 187 and 69, 967 and 440, 2,318 and
// 1,263; 1,603 and 1,072).  The product was the faster one at every size that
// was measured, so the memory alone decides.
template <class T> bool InverseOperator<T>::fits(const std::vector<int>& sys, size_t most_bytes) {
    size_t bytes = 0;
    for (size_t s = 0; s + 1 < sys.size(); ++s) {
        const int n = sys[s + 1] - sys[s];
        bytes += (size_t)n * padded(n) * sizeof(T);
    }
    // never more than a quarter of what is free: the inverse of a large body is
    // 27 to 50 times its factor, and the caller's arrays come first
    size_t free_bytes = 0, total_bytes = 0;
    if (hipMemGetInfo(&free_bytes, &total_bytes) != hipSuccess) return false;
    return bytes <= std::min(most_bytes, free_bytes / 4);
}

template <class T>
void InverseOperator<T>::setup(const BandFactor& f, const std::vector<int>& sys, hipStream_t stream) {
    const int nsys = (int)sys.size() - 1;
    std::vector<int> pos(f.n), vert, job;
    std::vector<long long> off;
    std::vector<StripJob> strips;
    long long total = 0, y = 0;
    int npad = 0;
    for (int s = 0; s < nsys; ++s) {
        const int s0 = sys[s], n = sys[s + 1] - s0, ld = padded(n);
        for (int i = 0; i < ld; ++i) {
            if (i < n) pos[f.perm[s0 + i]] = npad + i;
            vert.push_back(i < n ? f.perm[s0 + i] : 0);
        }
        for (int r = 0; r < n; r += kRowsPer) {
            job.insert(job.end(), {npad, n, ld, r});
            off.push_back(total + (long long)r * ld);
        }
        for (int c = 0; c < ld; c += kStripCols) strips.push_back(StripJob{s0, n, c, ld, 0, total});
        total += (long long)n * ld;
        npad += ld;
    }
    // the factor by rows and by columns, kBlkRows zeros past the band and past the last row
    const int lw = f.bw + 1 + kBlkRows;
    std::vector<double> Lr((size_t)(f.n + kBlkRows) * lw, 0.0), Uc(Lr.size(), 0.0), ri(f.n + kBlkRows, 1.0);
    for (int i = 0; i < f.n; ++i) {
        const double* Li = &f.Lb[(size_t)i * (f.bw + 1)];
        ri[i] = 1.0 / Li[0];
        for (int d = 0; d <= std::min(f.bw, i); ++d) {
            Lr[(size_t)i * lw + d] = Li[d];
            Uc[(size_t)(i - d) * lw + d] = Li[d];
        }
    }
    // every allocation before the first copy: one that fails leaves nothing of the host's vectors in flight
    inv_.alloc((size_t)total);
    rhs_.alloc(3 * (size_t)npad);
    pos_.alloc(pos.size());
    vert_.alloc(vert.size());
    job_.alloc(job.size());
    job_off_.alloc(off.size());
    parts_.alloc(off.size() + kStripes);
    ticket_.alloc(kTicketPitch * (1 + kStripes));
    DevBuf<double> dLr(Lr.size()), dUc(Uc.size()), dri(ri.size());
    DevBuf<StripJob> dstrips(strips.size());
    // strips in runs whose columns fit the scratch, which takes a quarter of the free memory at most
    size_t free_bytes = 0, total_bytes = 0;
    SBS_HIP(hipMemGetInfo(&free_bytes, &total_bytes));
    const size_t most = std::min(kScratchBytes, free_bytes / 4) / sizeof(double);
    size_t scratch = 0;
    std::vector<size_t> runs = {0};
    for (size_t k = 0; k < strips.size(); ++k) {
        const long long need = (long long)strips[k].n * kStripCols;
        if (k > runs.back() && (size_t)(y + need) > most) {
            runs.push_back(k);
            y = 0;
        }
        strips[k].y_off = y;
        y += need;
        scratch = std::max(scratch, (size_t)y);
    }
    runs.push_back(strips.size());
    DevBuf<double> Y(scratch);
    SBS_HIP(hipMemsetAsync(rhs_.get(), 0, rhs_.bytes(), stream));
    SBS_HIP(hipMemsetAsync(ticket_.get(), 0, ticket_.bytes(), stream));
    SBS_HIP(hipMemcpyAsync(pos_.get(), pos.data(), pos_.bytes(), hipMemcpyHostToDevice, stream));
    SBS_HIP(hipMemcpyAsync(vert_.get(), vert.data(), vert_.bytes(), hipMemcpyHostToDevice, stream));
    SBS_HIP(hipMemcpyAsync(job_.get(), job.data(), job_.bytes(), hipMemcpyHostToDevice, stream));
    SBS_HIP(hipMemcpyAsync(job_off_.get(), off.data(), job_off_.bytes(), hipMemcpyHostToDevice, stream));
    SBS_HIP(hipMemcpyAsync(dLr.get(), Lr.data(), dLr.bytes(), hipMemcpyHostToDevice, stream));
    SBS_HIP(hipMemcpyAsync(dUc.get(), Uc.data(), dUc.bytes(), hipMemcpyHostToDevice, stream));
    SBS_HIP(hipMemcpyAsync(dri.get(), ri.data(), dri.bytes(), hipMemcpyHostToDevice, stream));
    SBS_HIP(hipMemcpyAsync(dstrips.get(), strips.data(), dstrips.bytes(), hipMemcpyHostToDevice, stream));
    for (size_t k = 0; k + 1 < runs.size(); ++k) {
        hipLaunchKernelGGL(inverse_strip_kernel<T>, dim3((unsigned)(runs[k + 1] - runs[k])), dim3(64 * kStripWaves), 0,
                           stream, (const StripJob*)dstrips.get() + runs[k], f.bw, lw, (const double*)dLr.get(),
                           (const double*)dUc.get(), (const double*)dri.get(), Y.get(), inv_.get());
        SBS_HIP(hipGetLastError());
    }
    SBS_HIP(hipStreamSynchronize(stream));  // the host vectors and the scratch end here
    n_ = f.n;
    npad_ = npad;
    groups_ = (unsigned)off.size();
}

template <class T> void InverseOperator<T>::load_rhs(const T* b, hipStream_t stream, const int* skip) const {
    hipLaunchKernelGGL(permute_rhs_kernel<T>, dim3(ceil_div((size_t)n_, kThreads)), dim3(kThreads), 0, stream, n_, b,
                       (const int*)pos_.get(), npad_, rhs_.get(), skip);
    SBS_HIP(hipGetLastError());
}

template <class T> void InverseOperator<T>::apply(T* x, hipStream_t stream, const int* skip) const {
    hipLaunchKernelGGL((inverse_apply_kernel<T, false>), dim3(groups_), dim3(kThreads), 0, stream,
                       (const int4*)job_.get(), (const long long*)job_off_.get(), (const T*)inv_.get(),
                       (const T*)rhs_.get(), npad_, (const int*)vert_.get(), x, OuterStep<T>{}, n_, parts_.get(),
                       (unsigned*)nullptr, skip);
    SBS_HIP(hipGetLastError());
}

template <class T>
void InverseOperator<T>::apply_outer(const OuterStep<T>& o, hipStream_t stream, const int* skip) const {
    hipLaunchKernelGGL((inverse_apply_kernel<T, true>), dim3(groups_), dim3(kThreads), 0, stream,
                       (const int4*)job_.get(), (const long long*)job_off_.get(), (const T*)inv_.get(),
                       (const T*)rhs_.get(), npad_, (const int*)vert_.get(), (T*)nullptr, o, n_, parts_.get(),
                       ticket_.get(), skip);
    SBS_HIP(hipGetLastError());
}

template class InverseOperator<float>;
template class InverseOperator<double>;

}  // namespace sbs
