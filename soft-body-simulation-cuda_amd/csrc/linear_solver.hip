// General COO linear solve (LinearSolver<T>::Solve with PCGJacobiSolver's
// algorithm): sort_coo on the GPU with hipCUB, CSR rows, Jacobi-PCG with the
// scalars on the device.  See linear_solver.hpp for the reference lines.
#include "linear_solver.hpp"

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <string>

namespace sbs {
namespace {

constexpr int kTpbL = 256;

struct LinCtl {
    double rho[2];   // r.z of iteration k, by parity of k
    int done;        // 1 once a stop test held
    int iters;       // iterations completed (the reference's k at its break)
    int bad_index;   // a triplet index outside [0, N)
    int pad;
    long long nnz;   // entries after summing repeats
};

unsigned nblk(size_t n) { return (unsigned)std::max<size_t>(1, (n + kTpbL - 1) / kTpbL); }

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Block sum of a double into parts[blockIdx.x] (fixed order inside the block).
__device__ __forceinline__ void block_sum_to(double v, double* parts) {
    __shared__ double red[kTpbL / 64];
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int w = 0; w < kTpbL / 64; ++w) s += red[w];
        parts[blockIdx.x] = s;
    }
}

// Sums of NQ arrays of nb partials: every block of a launch forms the same
// values (thread t adds partials t, t + kTpbL, ..., then the wavefronts'
// totals in index order).  The loads can be issued ahead of the sums.
template <int NQ> __device__ __forceinline__ void load_partials(const double* const (&parts)[NQ], int nb, double (&s)[NQ]) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) s[q] = 0.0;
    for (int i = threadIdx.x; i < nb; i += kTpbL)
#pragma unroll
        for (int q = 0; q < NQ; ++q) s[q] += parts[q][i];
}
template <int NQ> __device__ __forceinline__ void totals_of(double (&s)[NQ]) {
    __shared__ double red[NQ][kTpbL / 64];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const double w = wave_total(s[q]);
        if ((threadIdx.x & 63) == 0) red[q][threadIdx.x >> 6] = w;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        s[q] = 0.0;
#pragma unroll
        for (int w = 0; w < kTpbL / 64; ++w) s[q] += red[q][w];
    }
}

__global__ void ctl_reset_kernel(LinCtl* ctl, long long* nruns) {
    if (threadIdx.x == 0) {
        ctl->rho[0] = ctl->rho[1] = 0.0;
        ctl->done = 0;
        ctl->iters = 0;
        ctl->bad_index = 0;
        ctl->nnz = 0;
        *nruns = 0;
    }
}

// The solve's done flag as one value for the whole block (thread 0 reads it).
__device__ __forceinline__ bool block_done(const LinCtl* ctl) {
    __shared__ int s_done;
    if (threadIdx.x == 0) s_done = ctl->done;
    __syncthreads();
    return s_done != 0;
}

// key = row * N + col; indices outside [0, N) flag the control block.
__global__ void coo_keys_kernel(long long nz, const int* row, const int* col, int n, unsigned long long* keys,
                                LinCtl* ctl) {
    const long long i = (long long)blockIdx.x * kTpbL + threadIdx.x;
    if (i >= nz) return;
    const int r = row[i], c = col[i];
    if (r < 0 || r >= n || c < 0 || c >= n) {
        ctl->bad_index = 1;
        keys[i] = 0;
        return;
    }
    keys[i] = (unsigned long long)r * (unsigned long long)n + (unsigned long long)c;
}

// CSR from the sorted unique keys: column of each entry, and rowptr[r] = the
// first entry of row r (rows without entries point at the next row's first).
__global__ void csr_kernel(long long nz_bound, const long long* nruns, const unsigned long long* ukeys, int n,
                           int* rowptr, int* colidx, LinCtl* ctl) {
    const long long i = (long long)blockIdx.x * kTpbL + threadIdx.x;
    const long long m = *nruns;
    if (i == 0) ctl->nnz = m;
    if (m == 0) {
        for (long long r = i; r <= n; r += (long long)gridDim.x * kTpbL) rowptr[r] = 0;
        return;
    }
    if (i >= m || i >= nz_bound) return;
    const unsigned long long k = ukeys[i];
    const long long r = (long long)(k / (unsigned long long)n);
    colidx[i] = (int)(k - (unsigned long long)r * (unsigned long long)n);
    const long long prev = i == 0 ? -1 : (long long)(ukeys[i - 1] / (unsigned long long)n);
    for (long long rr = prev + 1; rr <= r; ++rr) rowptr[rr] = (int)i;
    if (i == m - 1)
        for (long long rr = r + 1; rr <= n; ++rr) rowptr[rr] = (int)m;
}

// ExtractInverseDiagonalKernel (pcgJacobi.cu:6-24): 1 / the row's diagonal
// entry, 1 where it is missing or |d| < 1e-9.
template <class T>
__global__ void inv_diag_kernel(int n, const int* rowptr, const int* colidx, const T* val, T* dinv) {
    const int r = blockIdx.x * kTpbL + threadIdx.x;
    if (r >= n) return;
    T d = (T)1;
    for (int e = rowptr[r]; e < rowptr[r + 1]; ++e)
        if (colidx[e] == r) {
            d = val[e];
            break;
        }
    if (fabs((double)d) < 1e-9) d = (T)1;
    dinv[r] = (T)1 / d;
}

// Rows are shared by kLanes lanes: lane l of a row takes its entries l,
// l + kLanes, ... (consecutive lanes read consecutive entries), and the lanes'
// sums are added as a tree.  A block holds kTpbL / kLanes rows.
template <int kLanes, class T> __device__ __forceinline__ T lane_sum(T v) {
#pragma unroll
    for (int o = 1; o < kLanes; o <<= 1) v += __shfl_xor(v, o);
    return v;
}
constexpr int kRowBatch = 4;  // entries of a lane whose loads are in flight together
template <class T> struct RowPart {
    int c[kRowBatch];
    T m[kRowBatch];  // 0 past the row's end
};
template <int kLanes, class T>
__device__ __forceinline__ void load_part(const int* __restrict__ colidx, const T* __restrict__ val, int e, int e1,
                                          RowPart<T>& p) {
#pragma unroll
    for (int j = 0; j < kRowBatch; ++j) {
        const int k = e + j * kLanes, kc = k < e1 ? k : e1 - 1;
        p.c[j] = colidx[kc];
        const T m = val[kc];
        p.m[j] = k < e1 ? m : (T)0;
    }
}

// x0 = guess (r = b - A x0) or 0 (r = b); z = D^-1 r; partials of r.r, r.z
// for iteration 0 (parity 0).
template <class T>
__global__ void pcg_start_kernel(int n, const T* b, const T* guess, T* x, T* r, T* z, const T* dinv, const int* rowptr,
                                 const int* colidx, const T* val, double* prr, double* prz) {
    const int i = blockIdx.x * kTpbL + threadIdx.x;
    double rr = 0.0, rz = 0.0;
    if (i < n) {
        T ri = b[i];
        if (guess) {
            T acc = 0;
            for (int e = rowptr[i]; e < rowptr[i + 1]; ++e) acc += val[e] * guess[colidx[e]];
            ri -= acc;
        }
        const T zi = dinv[i] * ri;
        x[i] = guess ? guess[i] : (T)0;
        r[i] = ri;
        z[i] = zi;
        rr = (double)ri * (double)ri;
        rz = (double)ri * (double)zi;
    }
    block_sum_to(rr, prr);
    block_sum_to(rz, prz);
}

// The stop tests of iteration k (||r|| < tol, then |r.z| < 1e-15) and beta =
// rho_k / rho_{k-1}, formed by every block from the totals rr = r.r and rho =
// r.z of the update launch; block 0 records them.  Returns true when the solve
// stops here.
__device__ __forceinline__ bool pcg_direction(int k, double tol, double rr, double rho, LinCtl* ctl, double& beta) {
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    if (sqrt(rr) < tol || fabs(rho) < 1e-15) {
        if (lead) {
            ctl->done = 1;
            ctl->iters = k;
        }
        return true;
    }
    beta = k == 0 ? 0.0 : rho / ctl->rho[(k - 1) & 1];
    if (lead) ctl->rho[k & 1] = rho;
    return false;
}

// Iteration k, part 1 when there is no room for a second direction: p = z +
// beta p in place (p = z at k = 0).
template <class T>
__global__ void pcg_dir_kernel(int n, int k, int nb, double tol, const double* prr, const double* prz, const T* z,
                               T* p, LinCtl* ctl) {
    if (block_done(ctl)) return;
    double s[2];
    load_partials<2>({prr, prz}, nb, s);
    totals_of<2>(s);
    double beta;
    if (pcg_direction(k, tol, s[0], s[1], ctl, beta)) return;
    const int i = blockIdx.x * kTpbL + threadIdx.x;
    if (i < n) p[i] = k == 0 ? z[i] : z[i] + (T)beta * p[i];
}

// Iteration k, part 2: q = A p and the partials of p.q.  With kForm the
// direction is formed here too: p_k = z + beta p_{k-1} by one expression
// wherever it is read (the row's own entry, stored to pnew, and the columns),
// so an iteration is two launches.  A launch is a chain of memory round trips
// (row bounds, entries, the columns' values; the stop word; the partials), so
// all but the last of them are requested before the stop word is looked at.
// With one thread per row the entries of neighbouring threads lie a row
// apart: 16,416 rows of 41 entries in FP64 took 17.9 us (and 4.4 us for the
// direction), this form 6.0 us.
template <int kLanes, bool kForm, class T>
__global__ void __launch_bounds__(kTpbL) pcg_spmv_kernel(int n, int k, int nb, double tol, const double* prr,
                                                         const double* prz, const int* __restrict__ rowptr,
                                                         const int* __restrict__ colidx, const T* __restrict__ val,
                                                         const T* __restrict__ z, const T* __restrict__ pold,
                                                         T* __restrict__ pnew, T* __restrict__ q, double* ppq,
                                                         LinCtl* ctl) {
    const bool first = k == 0;
    const int i = (blockIdx.x * kTpbL + threadIdx.x) / kLanes, l = threadIdx.x % kLanes;
    const bool live = i < n;
    const int e0 = live ? rowptr[i] : 0, e1 = live ? rowptr[i + 1] : 0;
    double tot[2];
    if (kForm) load_partials<2>({prr, prz}, nb, tot);
    T zi = 0, pi = 0;
    if (live && l == 0) {
        if (kForm) zi = z[i];
        if (!kForm || !first) pi = pold[i];
    }
    RowPart<T> part;
    T zc[kRowBatch], pc[kRowBatch];
    auto fetch = [&](int e) {
        load_part<kLanes>(colidx, val, e, e1, part);
#pragma unroll
        for (int j = 0; j < kRowBatch; ++j) {
            if (kForm) zc[j] = z[part.c[j]];
            pc[j] = kForm && first ? (T)0 : pold[part.c[j]];
        }
    };
    const bool any = e0 + l < e1;
    if (any) fetch(e0 + l);
    if (block_done(ctl)) return;
    double bt = 0.0;
    if (kForm) {
        totals_of<2>(tot);
        if (pcg_direction(k, tol, tot[0], tot[1], ctl, bt)) return;
    }
    const T beta = (T)bt;
    auto dir = [&](T zv, T pv) -> T { return !kForm ? pv : first ? zv : zv + beta * pv; };
    T acc = 0;
    if (any)
        for (int e = e0 + l;;) {
#pragma unroll
            for (int j = 0; j < kRowBatch; ++j)
                if (e + j * kLanes < e1) acc += part.m[j] * dir(zc[j], pc[j]);
            e += kLanes * kRowBatch;
            if (e >= e1) break;
            fetch(e);
        }
    acc = lane_sum<kLanes>(acc);
    double pq = 0.0;
    if (live && l == 0) {
        const T pv = dir(zi, pi);
        if (kForm) pnew[i] = pv;
        q[i] = acc;
        pq = (double)pv * (double)acc;
    }
    block_sum_to(pq, ppq);
}

// Iteration k, part 3: alpha = rho / p.q, x += alpha p, r -= alpha q, then
// z = D^-1 r and the partials of iteration k+1 (other parity).
template <class T>
__global__ void pcg_update_kernel(int n, int k, int nb_prod, const double* ppq, const T* p, const T* q, T* x, T* r, T* z,
                                  const T* dinv, double* prr_next, double* prz_next, LinCtl* ctl) {
    double tot[1];
    load_partials<1>({ppq}, nb_prod, tot);
    const int i = blockIdx.x * kTpbL + threadIdx.x;
    T xi = 0, pi = 0, ri = 0, qi = 0, di = 0;
    if (i < n) {
        xi = x[i];
        pi = p[i];
        ri = r[i];
        qi = q[i];
        di = dinv[i];
    }
    if (block_done(ctl)) return;
    totals_of<1>(tot);
    const T alpha = (T)(ctl->rho[k & 1] / tot[0]);
    double rr = 0.0, rz = 0.0;
    if (i < n) {
        x[i] = xi + alpha * pi;
        ri -= alpha * qi;
        const T zi = di * ri;
        r[i] = ri;
        z[i] = zi;
        rr = (double)ri * (double)ri;
        rz = (double)ri * (double)zi;
    }
    block_sum_to(rr, prr_next);
    block_sum_to(rz, prz_next);
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl->iters = k + 1;
}

constexpr int kMaxLanes = 32;  // lanes per row of the product at most
// Lanes per row: a lane keeps 4 to 8 entries of a mean row (an elasticity row
// of 41 entries, 152 iterations of 16,416 rows: 4 lanes 2,175 us a solve, 8
// 2,185, 16 2,223; with one thread per row 4,700).
int lanes_for(int n, long long nnz) {
    int l = 1;
    while (l < kMaxLanes && 8ll * l * n <= nnz) l *= 2;
    return l;
}

// Workspace layout (each piece 256-byte aligned).
template <class T> struct Layout {
    unsigned long long *keys, *keys_sorted, *ukeys;
    T *vals_sorted, *uvals;
    long long* nruns;
    int *rowptr, *colidx;
    T *dinv, *r, *z, *p, *q;
    double *prr, *prz, *ppq;  // prr, prz: two parities of nb partials
    LinCtl* ctl;
    void* tmp;
    size_t tmp_bytes;
    size_t total;
    // The sort's arrays (keys to vals_sorted, contiguous) are free once the
    // rows stand: the second direction and the product's partials live there
    // where they fit, so the workspace is no larger for them.
    T* p2 = nullptr;
    double* ppq_rows = nullptr;

    Layout(char* base, int n, long long nz, size_t tmp_b) {
        size_t off = 0;
        auto take = [&](size_t bytes) {
            char* ptr = base ? base + off : nullptr;
            off += align256(std::max<size_t>(bytes, 1));
            return ptr;
        };
        const size_t z1 = (size_t)std::max<long long>(nz, 1);
        const int nb = (int)nblk(n);
        keys = (unsigned long long*)take(z1 * 8);
        keys_sorted = (unsigned long long*)take(z1 * 8);
        ukeys = (unsigned long long*)take(z1 * 8);
        vals_sorted = (T*)take(z1 * sizeof(T));
        uvals = (T*)take(z1 * sizeof(T));
        nruns = (long long*)take(8);
        rowptr = (int*)take(((size_t)n + 1) * 4);
        colidx = (int*)take(z1 * 4);
        dinv = (T*)take((size_t)n * sizeof(T));
        r = (T*)take((size_t)n * sizeof(T));
        z = (T*)take((size_t)n * sizeof(T));
        p = (T*)take((size_t)n * sizeof(T));
        q = (T*)take((size_t)n * sizeof(T));
        prr = (double*)take(2 * (size_t)nb * 8);
        prz = (double*)take(2 * (size_t)nb * 8);
        ppq = (double*)take((size_t)nb * 8);
        ctl = (LinCtl*)take(sizeof(LinCtl));
        tmp = take(tmp_b);
        tmp_bytes = tmp_b;
        total = off;
        const size_t second = align256((size_t)n * sizeof(T));
        const size_t partials = align256((size_t)nblk((size_t)n * kMaxLanes) * sizeof(double));
        if (base && second + partials <= (size_t)((char*)uvals - base)) {
            p2 = (T*)base;
            ppq_rows = (double*)(base + second);
        }
    }
};

}  // namespace

// Workspace of the allocation-free solve (solve_no_alloc): one array per GPU,
// held until the process ends.  Host code never passes the array's name to a
// kernel or a copy (on the host it is only a stand-in for the symbol): it
// uses the device address hipGetSymbolAddress returns for the current GPU.
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The current GPU's address of `scratch`, looked up once per device.
void* scratch_ptr() {
    int dev = 0;
    SBS_HIP(hipGetDevice(&dev));
    SBS_REQUIRE(dev >= 0 && dev < kMaxDevices, "allocation-free solve: device index out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        SBS_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        SBS_REQUIRE(p != nullptr, "allocation-free solve: no device address for the workspace");
        g_scratch_ptr[dev] = p;
    }
    return g_scratch_ptr[dev];
}
}  // namespace

template <class T>
int CooPcgSolver<T>::solve_no_alloc(int n, const T* b, T* x, const T* A, long long nz, const int* row,
                                    const int* col, const T* guess, hipStream_t stream) {
    SBS_REQUIRE(n >= 0 && nz >= 0, "LinearSolver::Solve: negative size");
    const size_t need = CooWorkspace::bytes(n, nz, sizeof(T), sort_tmp_bytes(nz, n));
    if (need > kNoAllocScratchBytes)
        throw Error(kInvalidArgument, "allocation-free solve: N = " + std::to_string(n) + ", nz = " +
                                          std::to_string(nz) + " needs " + std::to_string(need) +
                                          " bytes of workspace; its fixed workspace holds " +
                                          std::to_string(kNoAllocScratchBytes));
    return solve_in(n, b, x, A, nz, row, col, guess, stream, scratch_ptr(), kNoAllocScratchBytes);
}

template <class T> size_t CooPcgSolver<T>::sort_tmp_bytes(long long nz, int n) {
    const int items = (int)std::max<long long>(nz, 1);
    size_t a = 0, b = 0;
    unsigned long long* k = nullptr;
    T* v = nullptr;
    long long* nr = nullptr;
    SBS_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, a, k, k, v, v, items, 0, 64, nullptr));
    SBS_HIP(hipcub::DeviceReduce::ReduceByKey(nullptr, b, k, k, v, v, nr, hipcub::Sum(), items, nullptr));
    (void)n;
    return std::max(a, b);
}

size_t CooWorkspace::bytes(int n, long long nz, size_t elem, size_t sort_tmp) {
    if (elem == 4) return Layout<float>(nullptr, n, nz, sort_tmp).total;
    return Layout<double>(nullptr, n, nz, sort_tmp).total;
}

template <class T>
int CooPcgSolver<T>::solve(int n, const T* b, T* x, const T* A, long long nz, const int* row, const int* col,
                           const T* guess, hipStream_t stream) {
    SBS_REQUIRE(n >= 0 && nz >= 0, "LinearSolver::Solve: negative size");
    const size_t need = CooWorkspace::bytes(n, nz, sizeof(T), sort_tmp_bytes(nz, n));
    if (ws_.bytes() < need) ws_.alloc(need);
    return solve_in(n, b, x, A, nz, row, col, guess, stream, ws_.get(), ws_.bytes());
}

template <class T>
int CooPcgSolver<T>::solve_in(int n, const T* b, T* x, const T* A, long long nz, const int* row, const int* col,
                              const T* guess, hipStream_t stream, void* ws, size_t ws_bytes) {
    SBS_REQUIRE(n >= 0 && nz >= 0, "LinearSolver::Solve: negative size");
    SBS_REQUIRE(nz < (1ll << 31), "LinearSolver::Solve: more than 2^31 - 1 triplets");
    if (n == 0) return 0;
    SBS_REQUIRE(b && x, "LinearSolver::Solve: null b or x");
    SBS_REQUIRE(nz == 0 || (A && row && col), "LinearSolver::Solve: null triplet array");
    const size_t tmp_b = sort_tmp_bytes(nz, n);
    Layout<T> L(static_cast<char*>(ws), n, nz, tmp_b);
    SBS_REQUIRE(ws != nullptr && L.total <= ws_bytes, "LinearSolver::Solve: workspace too small for this system");
    LinCtl hc{};  // host copy of the control word (a plain copy: nothing is allocated)
    const int nb = (int)nblk(n);
    hipLaunchKernelGGL(ctl_reset_kernel, dim3(1), dim3(64), 0, stream, L.ctl, L.nruns);
    // sort_coo (linear.cu:7-40): sort by (row, column), sum repeated entries
    const int items = (int)nz;
    int end_bit = 1;
    while (end_bit < 64 && ((unsigned long long)n * (unsigned long long)n) > (1ull << end_bit)) ++end_bit;
    if (nz > 0) {
        hipLaunchKernelGGL(coo_keys_kernel, dim3(nblk(nz)), dim3(kTpbL), 0, stream, (long long)nz, row, col, n, L.keys,
                           L.ctl);
        size_t tb = L.tmp_bytes;
        SBS_HIP(hipcub::DeviceRadixSort::SortPairs(L.tmp, tb, L.keys, L.keys_sorted, A, L.vals_sorted, items, 0,
                                                   end_bit, stream));
        tb = L.tmp_bytes;
        SBS_HIP(hipcub::DeviceReduce::ReduceByKey(L.tmp, tb, L.keys_sorted, L.ukeys, L.vals_sorted, L.uvals, L.nruns,
                                                  hipcub::Sum(), items, stream));
    }
    hipLaunchKernelGGL(csr_kernel, dim3(nblk(std::max<long long>(nz, 1))), dim3(kTpbL), 0, stream,
                       (long long)std::max<long long>(nz, 1), (const long long*)L.nruns,
                       (const unsigned long long*)L.ukeys, n, L.rowptr, L.colidx, L.ctl);
    hipLaunchKernelGGL(inv_diag_kernel<T>, dim3(nb), dim3(kTpbL), 0, stream, n, (const int*)L.rowptr,
                       (const int*)L.colidx, (const T*)L.uvals, L.dinv);
    hipLaunchKernelGGL(pcg_start_kernel<T>, dim3(nb), dim3(kTpbL), 0, stream, n, b, guess, x, L.r, L.z,
                       (const T*)L.dinv, (const int*)L.rowptr, (const int*)L.colidx, (const T*)L.uvals, L.prr, L.prz);
    SBS_HIP(hipGetLastError());
    SBS_HIP(hipMemcpyAsync(&hc, L.ctl, sizeof(LinCtl), hipMemcpyDeviceToHost, stream));
    SBS_HIP(hipStreamSynchronize(stream));
    SBS_REQUIRE(!hc.bad_index, "LinearSolver::Solve: a row or column index is outside [0, N)");
    nnz_ = hc.nnz;
    const int lanes = L.p2 ? lanes_for(n, hc.nnz) : 1;
    const int nbp = (int)nblk((size_t)n * lanes);
    double* ppq = L.p2 ? L.ppq_rows : L.ppq;
    const bool form = L.p2 != nullptr;
    T* dir[2] = {L.p, form ? L.p2 : L.p};
    // product of iteration k: reads the direction of k - 1 (or, without room
    // for two, the direction that pcg_dir_kernel has just formed)
    auto product = [&](int k, const double* prr, const double* prz) {
        auto launch = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(nbp), dim3(kTpbL), 0, stream, n, k, nb, tol_, prr, prz,
                               (const int*)L.rowptr, (const int*)L.colidx, (const T*)L.uvals, (const T*)L.z,
                               (const T*)dir[(k + 1) & 1], dir[k & 1], L.q, ppq, L.ctl);
        };
        if (!form) {
            hipLaunchKernelGGL(pcg_dir_kernel<T>, dim3(nb), dim3(kTpbL), 0, stream, n, k, nb, tol_, prr, prz,
                               (const T*)L.z, L.p, L.ctl);
            launch(pcg_spmv_kernel<1, false, T>);
            return;
        }
        switch (lanes) {
            case 1: launch(pcg_spmv_kernel<1, true, T>); break;
            case 2: launch(pcg_spmv_kernel<2, true, T>); break;
            case 4: launch(pcg_spmv_kernel<4, true, T>); break;
            case 8: launch(pcg_spmv_kernel<8, true, T>); break;
            case 16: launch(pcg_spmv_kernel<16, true, T>); break;
            default: launch(pcg_spmv_kernel<32, true, T>); break;
        }
    };
    looks_.begin(n, nz, guess != nullptr);
    int k = 0;
    while (k < max_iter_) {
        const int chunk = std::min(looks_.next(k), max_iter_ - k);
        for (int j = 0; j < chunk; ++j, ++k) {
            const int par = k & 1;
            product(k, L.prr + par * nb, L.prz + par * nb);
            hipLaunchKernelGGL(pcg_update_kernel<T>, dim3(nb), dim3(kTpbL), 0, stream, n, k, nbp, (const double*)ppq,
                               (const T*)dir[k & 1], (const T*)L.q, x, L.r, L.z, (const T*)L.dinv,
                               L.prr + (1 - par) * nb, L.prz + (1 - par) * nb, L.ctl);
        }
        SBS_HIP(hipGetLastError());
        SBS_HIP(hipMemcpyAsync(&hc, L.ctl, sizeof(LinCtl), hipMemcpyDeviceToHost, stream));
        SBS_HIP(hipStreamSynchronize(stream));
        if (hc.done) break;
    }
    looks_.end(hc.iters, hc.done != 0);
    return hc.iters;
}

template class CooPcgSolver<float>;
template class CooPcgSolver<double>;

}  // namespace sbs
