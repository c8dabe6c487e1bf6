// oc_solver_matrices.hip -- the solver system of an equations set on the
// device: the equations matrix (Laplace) or the Jacobian (Mooney-Rivlin)
// restricted to the free DOFs, and the matching vector.
//
// The reference builds its solver system from the equations matrices through
// the solver mapping (SOLVER_MATRICES_STATIC_ASSEMBLE, solver_routines.f90:
// 13745-14771; SOLVER_MATRIX_JACOBIAN_MATRIX_ADD, solver_matrices_routines.f90:
// 1258-1483, and its equations-matrix counterpart):
//  * an equations row or column enters the solver system only when its DOF is
//    free (INCLUDE_ROW / INCLUDE_COLUMN, solver_mapping_routines.f90:434-520);
//  * solver rows and columns number the free DOFs in ascending order (one
//    equations set on one rank);
//  * the coupling coefficients of a single equations set are 1 and the solver
//    matrix starts at zero, so each solver entry is 0 + J(r, c);
//  * the solver vector of a linear set is the RHS with the fixed columns moved
//    over: for solver row r, in ascending column order, RHS(r) at c = r and
//    -K(r, c) u_c for every fixed column c, where u_c is the DOF's current
//    value and terms with |u_c| or |K(r, c)| below ZERO_TOLERANCE are skipped
//    (solver_routines.f90:14380-14620);
//  * the solver vector of a nonlinear set is the residual of the free rows.
//
// Layout: index[d] is the solver number of DOF d (-1 when fixed), rows[i] the
// equations row of solver row i.  One wavefront per solver row compacts the
// row: lane k takes entry k of a 64-entry chunk, whose free-column bits give
// every free entry its place, so the solver CSR is written once, in order, with
// no scan pass over the nonzeros.
#include "oc_internal.h"

#include <algorithm>

namespace oc {

namespace {

constexpr double kZeroTolerance = 5.0 * 2.220446049250313e-16;  // ZERO_TOLERANCE, constants.f90:68
constexpr int kRowsPerBlock = 4;                                // wavefronts
constexpr int kWaveRows = 2;                                    // solver rows each

// keep: bit k of the equations matrix's entries tells a free column, 64 entries
// a word (structure, made with the numbering): a values pass then reads one bit
// an entry where the columns and their solver numbers are 4 bytes and a
// dependent lookup
__global__ void __launch_bounds__(256)
solver_keep_kernel(int64_t nnz, const int *__restrict__ col_idx, const int *__restrict__ index,
                   uint64_t *__restrict__ keep)
{
    const int lane = threadIdx.x & 63;
    const int64_t words = nnz / 64 + 2;  // two past the last entry: keep_bits reads the next word
    for (int64_t w = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6); w < words;
         w += static_cast<int64_t>(gridDim.x) * 4) {
        const int64_t k = 64 * w + lane;
        const uint64_t m = __ballot(k < nnz && index[col_idx[min(k, nnz - 1)]] >= 0);
        if (lane == 0) keep[w] = m;
    }
}

// the bits of entries k0 .. k0 + n - 1 (n <= 64)
__device__ __forceinline__ uint64_t keep_bits(const uint64_t *__restrict__ keep, int64_t k0, int n)
{
    const uint64_t lo = keep[k0 >> 6], hi = keep[(k0 >> 6) + 1];
    const int s = static_cast<int>(k0 & 63);
    const uint64_t m = s ? lo >> s | hi << (64 - s) : lo;
    return n >= 64 ? m : m & ((uint64_t(1) << max(n, 0)) - 1);
}

// free columns of every solver row
__global__ void __launch_bounds__(256)
solver_count_kernel(int n, const int *__restrict__ rows, const int64_t *__restrict__ row_ptr,
                    const uint64_t *__restrict__ keep, int *__restrict__ counts)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int64_t k1 = row_ptr[rows[i] + 1];
    int c = 0;
    for (int64_t k = row_ptr[rows[i]]; k < k1; k += 64)
        c += __popcll(keep_bits(keep, k, static_cast<int>(min(k1 - k, int64_t(64)))));
    counts[i] = c;
}

// solver row i = equations row rows[i] without its fixed columns; with
// kStructure the solver column numbers are written as well.  A wavefront takes two
// rows by four 64-entry chunks, all of most Mooney-Rivlin rows: its loads are issued
// together (lanes past the end repeat the last entry), and the chunks' bits are
// scalars.  113,000 rows of an FP32 Jacobian: 85 us with the columns read
// and looked up, 55 us from the bits (62 with one row a wavefront).
template <typename T, bool kStructure>
__global__ void __launch_bounds__(64 * kRowsPerBlock)
solver_matrix_kernel(int n, const int *__restrict__ rows, const int64_t *__restrict__ row_ptr,
                     const int *__restrict__ col_idx, const int *__restrict__ index, const uint64_t *__restrict__ keep,
                     const int64_t *__restrict__ s_row_ptr, const T *__restrict__ values, T *__restrict__ s_values,
                     int *__restrict__ s_col_idx)
{
    constexpr int kChunks = 4;
    const int i0 = kWaveRows * (blockIdx.x * kRowsPerBlock + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    if (i0 >= n) return;  // whole wavefronts
    int64_t k0[kWaveRows], out[kWaveRows];
    int len[kWaveRows];
#pragma unroll
    for (int q = 0; q < kWaveRows; ++q) {
        const int i = min(i0 + q, n - 1), r = rows[i];
        k0[q] = row_ptr[r];
        len[q] = i0 + q < n ? static_cast<int>(row_ptr[r + 1] - k0[q]) : 0;
        out[q] = s_row_ptr[i];
    }
    T v[kWaveRows][kChunks];
#pragma unroll
    for (int q = 0; q < kWaveRows; ++q)
        if (len[q] > 0)  // a free DOF of no element has an empty row, which may stand at the end of the values
#pragma unroll
            for (int u = 0; u < kChunks; ++u) v[q][u] = values[k0[q] + min(64 * u + lane, len[q] - 1)];
#pragma unroll
    for (int q = 0; q < kWaveRows; ++q)
        for (int base = 0; base < len[q]; base += 64 * kChunks) {
            if (base > 0)
#pragma unroll
                for (int u = 0; u < kChunks; ++u) v[q][u] = values[k0[q] + min(base + 64 * u + lane, len[q] - 1)];
#pragma unroll
            for (int u = 0; u < kChunks; ++u) {
                const int left = len[q] - base - 64 * u;
                if (left <= 0) break;
                const uint64_t m = keep_bits(keep, k0[q] + base + 64 * u, left);
                if (__builtin_amdgcn_inverse_ballot_w64(m)) {
                    const int64_t p = out[q] + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                                                         __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0));
                    s_values[p] = T(0) + v[q][u];  // the solver matrix starts at zero
                    if (kStructure) s_col_idx[p] = index[col_idx[k0[q] + base + 64 * u + lane]];
                }
                out[q] += __popcll(m);
            }
        }
}

// Solver vector: with `lift` (linear sets) RHS(r) and the fixed columns in
// ascending column order, one thread per solver row; otherwise the residual.
__global__ void __launch_bounds__(256)
solver_vector_kernel(int n, const int *__restrict__ rows, const int64_t *__restrict__ row_ptr,
                     const int *__restrict__ col_idx, const int *__restrict__ index,
                     const double *__restrict__ values, const double *__restrict__ rhs,
                     const double *__restrict__ dofs, bool lift, double *__restrict__ out)
{
#pragma clang fp contract(off)  // each product rounded before its add, as the reference
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int r = rows[i];
    double acc = 0.0;
    if (!lift) {
        acc = acc + rhs[r];
    } else {
        for (int64_t k = row_ptr[r]; k < row_ptr[r + 1]; ++k) {
            const int c = col_idx[k];
            if (c == r) {
                acc = acc + rhs[r];
            } else if (index[c] < 0) {
                const double u = dofs[c], K = values[k];
                if (fabs(u) >= kZeroTolerance && fabs(K) >= kZeroTolerance) acc = acc + (-1.0 * K) * u;
            }
        }
    }
    out[i] = acc;
}

}  // namespace

// Free-DOF numbering and the solver CSR structure, rebuilt when the
// boundary conditions change.
static int solver_structure(EquationsSet &s)
{
    SolverSystem &S = s.solver;
    if (S.built && S.bc_version == s.bc_version) return OC_NO_ERROR;
    Runtime &rt = runtime();
    std::vector<uint8_t> mask(static_cast<size_t>(s.n_rows), 1);
    if (s.n_bc > 0) {
        OC_HIP_CHECK(hipMemcpyAsync(mask.data(), s.free_mask.ptr, mask.size(), hipMemcpyDeviceToHost, rt.stream));
        OC_HIP_CHECK(hipStreamSynchronize(rt.stream));
    }
    std::vector<int32_t> index(mask.size()), rows;
    rows.reserve(mask.size());
    for (int d = 0; d < s.n_rows; ++d) {
        index[d] = mask[d] ? static_cast<int32_t>(rows.size()) : -1;
        if (mask[d]) rows.push_back(d);
    }
    S.n = static_cast<int>(rows.size());
    OC_CHECK(S.index.upload(index.data(), index.size()));
    OC_CHECK(S.rows.upload(rows.data(), rows.size()));
    std::vector<int64_t> ptr(static_cast<size_t>(S.n) + 1, 0);
    if (S.n > 0) {
        DevBuf<int> counts;
        OC_CHECK(counts.alloc(static_cast<size_t>(S.n)));
        OC_CHECK(S.keep.alloc(static_cast<size_t>(s.nnz / 64 + 2)));
        solver_keep_kernel<<<static_cast<unsigned>(std::min<int64_t>(s.nnz / 256 + 1, 65536)), 256, 0, rt.stream>>>(
            s.nnz, s.col_idx.ptr, S.index.ptr, S.keep.ptr);
        solver_count_kernel<<<static_cast<unsigned>((S.n + 255) / 256), 256, 0, rt.stream>>>(
            S.n, S.rows.ptr, s.row_ptr.ptr, S.keep.ptr, counts.ptr);
        OC_HIP_CHECK(hipGetLastError());
        std::vector<int> h(static_cast<size_t>(S.n));
        OC_HIP_CHECK(hipMemcpyAsync(h.data(), counts.ptr, h.size() * sizeof(int), hipMemcpyDeviceToHost, rt.stream));
        OC_HIP_CHECK(hipStreamSynchronize(rt.stream));
        for (int i = 0; i < S.n; ++i) ptr[i + 1] = ptr[i] + h[i];
    }
    S.nnz = ptr.back();
    OC_CHECK(S.row_ptr.upload(ptr.data(), ptr.size()));
    OC_CHECK(S.col_idx.alloc(static_cast<size_t>(S.nnz)));
    S.values.release();
    S.values_sp.release();
    OC_CHECK(S.vector.alloc(static_cast<size_t>(S.n)));
    S.columns_written = false;
    S.built = true;
    S.bc_version = s.bc_version;
    return OC_NO_ERROR;
}

template <typename T>
static int solver_values(EquationsSet &s, const T *values, DevBuf<T> &out)
{
    SolverSystem &S = s.solver;
    if (!out.ptr) OC_CHECK(out.alloc(static_cast<size_t>(S.nnz)));
    if (S.n == 0) return OC_NO_ERROR;
    Runtime &rt = runtime();
    const unsigned blocks =
        static_cast<unsigned>((S.n + kWaveRows * kRowsPerBlock - 1) / (kWaveRows * kRowsPerBlock));
    if (!S.columns_written) {
        solver_matrix_kernel<T, true><<<blocks, 64 * kRowsPerBlock, 0, rt.stream>>>(
            S.n, S.rows.ptr, s.row_ptr.ptr, s.col_idx.ptr, S.index.ptr, S.keep.ptr, S.row_ptr.ptr, values, out.ptr,
            S.col_idx.ptr);
        S.columns_written = true;
    } else {
        solver_matrix_kernel<T, false><<<blocks, 64 * kRowsPerBlock, 0, rt.stream>>>(
            S.n, S.rows.ptr, s.row_ptr.ptr, s.col_idx.ptr, S.index.ptr, S.keep.ptr, S.row_ptr.ptr, values, out.ptr,
            nullptr);
    }
    OC_HIP_CHECK(hipGetLastError());
    return OC_NO_ERROR;
}

int solver_matrices_assemble(EquationsSet &s, int precision)
{
    const bool linear = s.cls == OC_EQUATIONS_SET_LAPLACE;
    if (precision != OC_FP64 && precision != OC_FP32)
        return set_error(OC_ERR_INVALID_ARGUMENT, "precision must be OC_FP64 or OC_FP32");
    if (linear && precision != OC_FP64)
        return set_error(OC_ERR_INVALID_ARGUMENT, "a linear equations matrix is FP64 only");
    if (precision == OC_FP64 && !s.values.ptr)
        return set_error(OC_ERR_INVALID_ARGUMENT, "no FP64 matrix has been assembled");
    if (precision == OC_FP32 && !s.values_sp.ptr)
        return set_error(OC_ERR_INVALID_ARGUMENT, "no FP32 Jacobian has been assembled");
    OC_CHECK(solver_structure(s));
    SolverSystem &S = s.solver;
    KernelTimer timer(precision == OC_FP64 ? "solver_matrix_fp64" : "solver_matrix_fp32");
    if (precision == OC_FP64) OC_CHECK(solver_values<double>(s, s.values.ptr, S.values));
    else OC_CHECK(solver_values<float>(s, s.values_sp.ptr, S.values_sp));
    if (S.n > 0) {
        const double *vec = linear ? s.rhs.ptr : s.residual.ptr;
        solver_vector_kernel<<<static_cast<unsigned>((S.n + 255) / 256), 256, 0, runtime().stream>>>(
            S.n, S.rows.ptr, s.row_ptr.ptr, s.col_idx.ptr, S.index.ptr, s.values.ptr, vec, s.dofs.ptr, linear,
            S.vector.ptr);
        OC_HIP_CHECK(hipGetLastError());
    }
    S.precision = precision;
    return OC_NO_ERROR;
}

}  // namespace oc
