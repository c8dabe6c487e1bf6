// oc_elasticity.hip -- gfx950 Mooney-Rivlin finite elasticity assembly:
// residual and analytic Jacobian (finite_elasticity_routines.f90:842-1175,
// 1260-1640) scattered deterministically into the CSR equations matrix.
//
// Jacobian: mr_gauss_kernel (one thread per element Gauss point, all
// elements) evaluates the FP64 kinematics and tangent into Gauss-point
// records (see GpField); mr_element_matrix_f64_kernel (FP64) or
// mr_element_matrix_f32_kernel (FP32) contracts the records of every
// element into its 89x89 element matrix on MFMA; and csr_row_gather_kernel
// assembles each CSR row from the element rows that touch it in ascending
// element order (deterministic, write-once), placing them through the
// neighbour-rank scatter map.
// Residual: mr_residual_element_kernel evaluates element residuals of all
// elements into a buffer and dof_gather_kernel sums them per DOF in
// ascending element order.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>
#include <vector>

#include "oc_fe_device.h"
#include "oc_internal.h"

namespace oc {

// Gauss-point record fields.  Field f of Gauss point g of element e is at
// rec[(e * GP_NFIELDS + f) * 27 + g]: an element's records are contiguous, so the
// element-matrix kernels take them without address arithmetic.
enum GpField : int {
    GP_DXIDZ = 0,   // 9: DXI_DX of the deformed metrics, column-major
    GP_JGW = 9,     // J_z * w_g
    GP_C = 10,      // 36: spatial elasticity tensor (Voigt, column-major)
    GP_SIGJ = 46,   // 6: Cauchy stress from the elasticity routine
    GP_NFIELDS = 52
};

constexpr int kGaussElemsPerBlock = 9;  // 9 elements x 27 Gauss points = 243 threads

constexpr int kGaussThreads = 256;

// The interpolation of nine elements at their Gauss points, one direction at a
// time: a thread takes a field's 9 nodal values of one zeta plane of an element
// to the 9 (xi, eta) points (value and both derivatives, in registers, with the
// 1D functions as constants), then each Gauss point adds the three planes: 99
// multiply-adds and 36 LDS reads a field and point row where the 27-node sums
// of every point took 486 and 243 for all six fields.  Those reads bound both
// kernels that use it (32,768 elements: residual 252 -> 63 us, records 120 -> 109
// us of which the 368 MB they write take 70).
struct ElementLds {
    double nodal[kGaussElemsPerBlock * 6][27];      // X then z, by component
    double plane[kGaussElemsPerBlock * 6 * 3][27];  // [.. 3 f + plane][kind * 9 + xi + 3 eta]: d/dxi, d/deta, value
    double p[kGaussElemsPerBlock][8];
};

// Thread t = 27 le + g: kinematics and pressure of Gauss point g of the block's
// element le; false where there is none.  With kFD launch element v is the pair
// (v / 89, v % 89) and the column's DOF is raised by delta.
template <bool kFD>
__device__ __forceinline__ bool element_points(int n_elements, int e0, const int *__restrict__ conn_q,
                                               const int *__restrict__ conn_l, const double *__restrict__ coords,
                                               int nq, const double *__restrict__ dofs, double delta, ElementLds &s,
                                               GaussKinematics &k, double *P)
{
    constexpr int kNodePer = (kGaussElemsPerBlock * 81 + kGaussThreads - 1) / kGaussThreads;
    const int t = threadIdx.x;
    // all global loads are issued before the LDS writes: the connectivity,
    // then the nodal values it indexes
    int node[kNodePer];
#pragma unroll
    for (int i = 0; i < kNodePer; ++i) {
        const int j = t + kGaussThreads * i;
        const int v = e0 + j / 81;
        node[i] = (j < kGaussElemsPerBlock * 81 && v < n_elements) ? conn_q[(kFD ? v / 89 : v) * 27 + j % 27] : -1;
    }
    const int pv = e0 + t / 8;
    const int pnode = (t < kGaussElemsPerBlock * 8 && pv < n_elements) ? conn_l[(kFD ? pv / 89 : pv) * 8 + t % 8] : -1;
    double xv[kNodePer], zv[kNodePer];
#pragma unroll
    for (int i = 0; i < kNodePer; ++i) {
        const int c = ((t + kGaussThreads * i) % 81) / 27;
        xv[i] = node[i] >= 0 ? coords[static_cast<int64_t>(c) * nq + node[i]] : 0.0;
        zv[i] = node[i] >= 0 ? dofs[static_cast<int64_t>(c) * nq + node[i]] : 0.0;
    }
    const double pval = pnode >= 0 ? dofs[static_cast<int64_t>(3) * nq + pnode] : 0.0;
#pragma unroll
    for (int i = 0; i < kNodePer; ++i) {
        const int j = t + kGaussThreads * i;
        const int le = j / 81, r = j % 81;
        if (node[i] >= 0) {
            s.nodal[6 * le + r / 27][r % 27] = xv[i];
            s.nodal[6 * le + 3 + r / 27][r % 27] = zv[i] + ((kFD && (e0 + le) % 89 == r) ? delta : 0.0);
        }
    }
    if (pnode >= 0) s.p[t / 8][t % 8] = pval + ((kFD && pv % 89 == 81 + t % 8) ? delta : 0.0);
    __syncthreads();
    if (t < kGaussElemsPerBlock * 18) {
        // only derivatives leave the planes: taken from the element's centre
        // node the sums round with the element's size, not its distance from
        // the origin
        const double *u = s.nodal[t / 3] + 9 * (t % 3), centre = s.nodal[t / 3][13];
        double v[3][3], d[3][3];  // [eta row][xi]: value, derivative
#pragma unroll
        for (int y = 0; y < 3; ++y) {
            const double u0 = u[3 * y] - centre, u1 = u[3 * y + 1] - centre, u2 = u[3 * y + 2] - centre;
#pragma unroll
            for (int g = 0; g < 3; ++g) {
                v[y][g] = kQuad[g][0] * u0 + kQuad[g][1] * u1 + kQuad[g][2] * u2;
                d[y][g] = kQuadD[g][0] * u0 + kQuadD[g][1] * u1 + kQuadD[g][2] * u2;
            }
        }
        double *o = s.plane[t];
#pragma unroll
        for (int h = 0; h < 3; ++h)
#pragma unroll
            for (int g = 0; g < 3; ++g) {
                o[g + 3 * h] = kQuad[h][0] * d[0][g] + kQuad[h][1] * d[1][g] + kQuad[h][2] * d[2][g];
                o[9 + g + 3 * h] = kQuadD[h][0] * v[0][g] + kQuadD[h][1] * v[1][g] + kQuadD[h][2] * v[2][g];
                o[18 + g + 3 * h] = kQuad[h][0] * v[0][g] + kQuad[h][1] * v[1][g] + kQuad[h][2] * v[2][g];
            }
    }
    __syncthreads();
    const int le = t / 27, g = t % 27;
    if (t >= kGaussElemsPerBlock * 27 || e0 + le >= n_elements) return false;
    const int xy = g % 9, gz = g / 9;
    double q[3], qd[3];
#pragma unroll
    for (int z = 0; z < 3; ++z) {
        q[z] = pick3(gz, kQuad[0][z], kQuad[1][z], kQuad[2][z]);
        qd[z] = pick3(gz, kQuadD[0][z], kQuadD[1][z], kQuadD[2][z]);
    }
    double dX[9], dz[9];
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        const double(*pl)[27] = s.plane + (6 * le + f) * 3;
        double *o = (f < 3 ? dX : dz) + f % 3;
        o[0] = q[0] * pl[0][xy] + q[1] * pl[1][xy] + q[2] * pl[2][xy];
        o[3] = q[0] * pl[0][9 + xy] + q[1] * pl[1][9 + xy] + q[2] * pl[2][9 + xy];
        o[6] = qd[0] * pl[0][18 + xy] + qd[1] * pl[1][18 + xy] + qd[2] * pl[2][18 + xy];
    }
    gauss_kinematics(dz, dX, k);
    const double x1 = pick3(g % 3, kXi[0], kXi[1], kXi[2]), y1 = pick3(xy / 3, kXi[0], kXi[1], kXi[2]),
                 z1 = pick3(gz, kXi[0], kXi[1], kXi[2]), x0 = 1.0 - x1, y0 = 1.0 - y1;
    const double *p = s.p[le];
    *P = (1.0 - z1) * (y0 * (x0 * p[0] + x1 * p[1]) + y1 * (x0 * p[2] + x1 * p[3])) +
         z1 * (y0 * (x0 * p[4] + x1 * p[5]) + y1 * (x0 * p[6] + x1 * p[7]));
    return true;
}

// Restates, per Gauss point, the interpolation/metrics/F/J block of the
// Jacobian routine (:954-989) and FINITE_ELASTICITY_GAUSS_ELASTICITY_TENSOR
// (:609-740).
__global__ void __launch_bounds__(kGaussThreads)
mr_gauss_kernel(int n_elements, const int *__restrict__ conn_q, const int *__restrict__ conn_l,
                const double *__restrict__ coords, int nq, const double *__restrict__ dofs,
                const double *__restrict__ mat, const BasisTables *__restrict__ T, double *__restrict__ rec)
{
    __shared__ ElementLds s;
    const int e0 = xcd_block(blockIdx.x, gridDim.x) * kGaussElemsPerBlock;
    const int e = e0 + static_cast<int>(threadIdx.x) / 27, g = threadIdx.x % 27;
    GaussKinematics k;
    double P;
    if (!element_points<false>(n_elements, e0, conn_q, conn_l, coords, nq, dofs, 0.0, s, k, &P)) return;
    rec += static_cast<int64_t>(e) * GP_NFIELDS * 27 + g;
#pragma unroll
    for (int i = 0; i < 9; ++i) rec[(GP_DXIDZ + i) * 27] = k.dxidz[i];
    rec[GP_JGW * 27] = k.jz * T->w27[g];
    double c[36], sigma[6];
    mr_elasticity_tensor(k.F, k.Jznu, P, mat[2 * e], mat[2 * e + 1], c, sigma);
#pragma unroll
    for (int i = 0; i < 36; ++i) rec[(GP_C + i) * 27] = c[i];
#pragma unroll
    for (int i = 0; i < 6; ++i) rec[(GP_SIGJ + i) * 27] = sigma[i];
}

// Scatter map.  A CSR row of node n (any of its three displacement rows, or
// a pressure row) holds, in ascending DOF order, the component-0 block of its
// nb displacement-node neighbours, the component-1 and component-2 blocks of
// the same nodes, then its pressure-node neighbours.  Element column j of
// row dof_i therefore sits at
//   (j / 27) * nb + rank[e][k][j % 27]           (j < 81)
//   3 * nb + rank[e][k][27 + j - 81]             (j >= 81),
// where k is the element node of row i (0..26 displacement, 27..34 pressure)
// and rank[e][k][m] is the position of element node m among the neighbours of
// node k: 35 x 35 bytes per element instead of 89 x 89 offsets, shared by the
// three displacement rows of a node.  nb is stored per row.
constexpr int kRankNodes = 35;

// nb of every row: the number of its columns below nq (component-0 block)
__global__ void __launch_bounds__(256)
row_neighbours_kernel(int n_rows, int nq, const int64_t *__restrict__ row_ptr, const int *__restrict__ col_idx,
                      uint16_t *__restrict__ nb)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n_rows) return;
    int64_t lo = row_ptr[r], hi = row_ptr[r + 1];  // first column >= nq
    const int64_t start = lo;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (col_idx[mid] < nq) lo = mid + 1;
        else hi = mid;
    }
    nb[r] = static_cast<uint16_t>(lo - start);
}

// rank[e][k][m], checked by bisection against every component pair it stands for
__global__ void __launch_bounds__(256)
column_rank_kernel(int n_elements, const int *__restrict__ conn_q, const int *__restrict__ conn_l, int nq,
                   const int64_t *__restrict__ row_ptr, const int *__restrict__ col_idx,
                   const uint16_t *__restrict__ nb, uint8_t *__restrict__ rank, int *__restrict__ n_bad)
{
    const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (gid >= static_cast<int64_t>(n_elements) * kRankNodes * kRankNodes) return;
    const int e = static_cast<int>(gid / (kRankNodes * kRankNodes));
    const int k = static_cast<int>((gid / kRankNodes) % kRankNodes), m = static_cast<int>(gid % kRankNodes);
    const bool qrow = k < 27, qcol = m < 27;
    const int rnode = qrow ? conn_q[e * 27 + k] : conn_l[e * 8 + k - 27];
    const int cnode = qcol ? conn_q[e * 27 + m] : conn_l[e * 8 + m - 27];
    const int row0 = qrow ? rnode : 3 * nq + rnode;
    const int col0 = qcol ? cnode : 3 * nq + cnode;
    const int64_t slot0 = csr_slot(row_ptr, col_idx, row0, col0);
    const int64_t rk = slot0 - row_ptr[row0] - (qcol ? 0 : 3 * static_cast<int64_t>(nb[row0]));
    bool ok = slot0 >= 0 && rk >= 0 && rk < 256;
    for (int c = 0; c < (qrow ? 3 : 1) && ok; ++c) {
        const int row = qrow ? c * nq + rnode : row0;
        for (int cc = 0; cc < (qcol ? 3 : 1) && ok; ++cc) {
            const int col = qcol ? cc * nq + cnode : col0;
            const int64_t want = row_ptr[row] + (qcol ? cc : 3) * static_cast<int64_t>(nb[row]) + rk;
            ok = csr_slot(row_ptr, col_idx, row, col) == want;
        }
    }
    if (!ok) atomicAdd(n_bad, 1);
    rank[gid] = ok ? static_cast<uint8_t>(rk) : 0;
}

// Row of the element buffer that holds element matrix row i (0..80: component i
// / 27 of node i % 27; pressure rows after them): a node's three rows lie next
// to each other, as the row gather reads them.
__device__ __forceinline__ int kbuf_row(int i) { return i < 81 ? 3 * (i % 27) + i / 27 : i; }

// The row gather's lists, from the DOF -> element-entry lists: entry p < 27 E of
// the component-0 rows (node m of element e) holds the element-buffer row of the
// node's first component and the row of the rank table; the entries of the
// pressure rows follow.
__global__ void __launch_bounds__(256) row_lists_kernel(int n_elements, const int *__restrict__ gidx, int2 *__restrict__ lists)
{
    const int64_t q = static_cast<int64_t>(n_elements) * 27;
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= static_cast<int64_t>(n_elements) * 35) return;
    const int ei = gidx[t < q ? t : t + 2 * q], e = ei / 89, i = ei % 89;
    lists[t] = make_int2(e * 89 + kbuf_row(i), e * kRankNodes + (i < 81 ? i : i - 54));
}

int mr_prepare(EquationsSet &s)
{
    if (s.col_rank.ptr) return OC_NO_ERROR;
    int64_t max_row = 0;
    for (int r = 0; r < s.n_rows; ++r) max_row = std::max(max_row, s.h_row_ptr[r + 1] - s.h_row_ptr[r]);
    if (max_row > 8192)
        return set_error(OC_ERR_UNSUPPORTED, "CSR row of %lld entries exceeds the row-gather capacity",
                         static_cast<long long>(max_row));
    if (static_cast<int64_t>(s.n_elements) * 89 >= INT32_MAX)
        return set_error(OC_ERR_UNSUPPORTED, "%d elements exceed the int32 element-entry gather lists", s.n_elements);
    s.max_row_len = static_cast<int>(max_row);
    Runtime &rt = runtime();
    OC_CHECK(s.row_nb.alloc(static_cast<size_t>(s.n_rows)));
    row_neighbours_kernel<<<static_cast<unsigned>((s.n_rows + 255) / 256), 256, 0, rt.stream>>>(
        s.n_rows, s.n_nodes, s.row_ptr.ptr, s.col_idx.ptr, s.row_nb.ptr);
    OC_HIP_CHECK(hipGetLastError());
    const int64_t nranks = static_cast<int64_t>(s.n_elements) * kRankNodes * kRankNodes;
    OC_CHECK(s.col_rank.alloc(static_cast<size_t>(nranks)));
    DevBuf<int> bad;
    OC_CHECK(bad.alloc(1));
    OC_HIP_CHECK(hipMemsetAsync(bad.ptr, 0, sizeof(int), rt.stream));
    column_rank_kernel<<<static_cast<unsigned>((nranks + 255) / 256), 256, 0, rt.stream>>>(
        s.n_elements, s.conn.ptr, s.conn_l.ptr, s.n_nodes, s.row_ptr.ptr, s.col_idx.ptr, s.row_nb.ptr,
        s.col_rank.ptr, bad.ptr);
    OC_HIP_CHECK(hipGetLastError());
    int h_bad = 0;
    OC_HIP_CHECK(hipMemcpyAsync(&h_bad, bad.ptr, sizeof(int), hipMemcpyDeviceToHost, rt.stream));
    OC_HIP_CHECK(hipStreamSynchronize(rt.stream));
    if (h_bad) {
        s.col_rank.release();
        return set_error(OC_ERR_PATTERN,
                         "%d element entries missing from the CSR structure, not in its component-block layout or past 255 neighbour nodes",
                         h_bad);
    }
    OC_CHECK(s.gp_records.alloc(static_cast<size_t>(s.n_elements) * 27 * GP_NFIELDS));
    OC_CHECK(s.relem.alloc(static_cast<size_t>(s.n_elements) * 89));
    // DOF -> element entries, ascending element order
    std::vector<int32_t> hconn(static_cast<size_t>(s.n_elements) * 27), hconn_l(static_cast<size_t>(s.n_elements) * 8);
    OC_HIP_CHECK(hipMemcpy(hconn.data(), s.conn.ptr, hconn.size() * sizeof(int32_t), hipMemcpyDeviceToHost));
    OC_HIP_CHECK(hipMemcpy(hconn_l.data(), s.conn_l.ptr, hconn_l.size() * sizeof(int32_t), hipMemcpyDeviceToHost));
    std::vector<int32_t> ptr(static_cast<size_t>(s.n_rows) + 1, 0), idx(static_cast<size_t>(s.n_elements) * 89);
    // element DOF i of element e (component -> node order of the reference
    // element matrix, equations_matrices_routines.f90:684-941): 0..80
    // displacement, 81..88 pressure
    auto dof_of = [&](int64_t e, int i) {
        return i < 81 ? (i / 27) * s.n_nodes + hconn[e * 27 + i % 27] : 3 * s.n_nodes + hconn_l[e * 8 + i - 81];
    };
    for (int64_t e = 0; e < s.n_elements; ++e)
        for (int i = 0; i < 89; ++i) ptr[dof_of(e, i) + 1]++;
    for (int d = 0; d < s.n_rows; ++d) ptr[d + 1] += ptr[d];
    std::vector<int32_t> fillp(ptr.begin(), ptr.end() - 1);
    for (int64_t e = 0; e < s.n_elements; ++e)
        for (int i = 0; i < 89; ++i) idx[fillp[dof_of(e, i)]++] = static_cast<int32_t>(e * 89 + i);
    OC_CHECK(s.gather_ptr.upload(ptr.data(), ptr.size()));
    OC_CHECK(s.gather_idx.upload(idx.data(), idx.size()));
    const int64_t nlist = static_cast<int64_t>(s.n_elements) * 35;
    OC_CHECK(s.row_lists.alloc(static_cast<size_t>(2 * nlist)));
    row_lists_kernel<<<static_cast<unsigned>((nlist + 255) / 256), 256, 0, rt.stream>>>(
        s.n_elements, s.gather_idx.ptr, reinterpret_cast<int2 *>(s.row_lists.ptr));
    OC_HIP_CHECK(hipGetLastError());
    return OC_NO_ERROR;
}

int launch_mr_gauss(EquationsSet &s)
{
    const BasisTables *T = nullptr;
    OC_CHECK(ensure_tables(&T));
    Runtime &rt = runtime();
    const unsigned blocks = static_cast<unsigned>((s.n_elements + kGaussElemsPerBlock - 1) / kGaussElemsPerBlock);
    KernelTimer timer("mr_gauss_jacobian");
    mr_gauss_kernel<<<blocks, kGaussThreads, 0, rt.stream>>>(s.n_elements, s.conn.ptr, s.conn_l.ptr, s.coords.ptr, s.n_nodes,
                                                   s.dofs.ptr, s.mat.ptr, T, s.gp_records.ptr);
    OC_HIP_CHECK(hipGetLastError());
    return OC_NO_ERROR;
}

// ---------------------------------------------------------------------------
// Residual (:1491-1574), fused with the Gauss-point evaluation: one block of
// 9 elements x 27 Gauss points evaluates kinematics and the stress routine,
// then sums each element residual entry
//   R_(a,m) += sum_i DPHIDZ(i,m) JGW sigma(i,a),  R_(p,m) += J_X w (J-1) psi_m
// over the Gauss points in order into a per-element buffer.  With
// DPHIDZ(i,m) = sum_j dphi_m/dxi_j DXI_DX(j,i), each Gauss point keeps in LDS
// only T(j,a) = sum_i DXI_DX(j,i) JGW sigma(i,a), and the entry sums
// dphi_m/dxi_j T(j,a) over j and the Gauss points.  A gather kernel
// then adds the element contributions of every DOF in ascending element order
// (the reference's element-loop order, equations_set_routines.f90:5535-5568).
//
// With kFD, "element" v of the launch is the pair (e = v / 89, column col =
// v % 89): element e's residual with its DOF col raised by delta, written as
// column col of e's element matrix (R(x + delta e_col) - R(x)) / delta, R(x)
// from relem (EquationsSet_FiniteElementJacobianEvaluateFD,
// equations_set_routines.f90:3032-3150).
// The sums over the Gauss points run one direction at a time as well: a thread
// per (element, component, xi point, zeta node) adds the nine points of its xi
// plane into the three eta nodes, one per (element, component, zeta and eta
// node) adds the xi points; a thread per pressure entry.  48 LDS reads and 72
// multiply-adds for three entries, where each entry's 27 terms took 12 and 9
// apiece.
template <bool kFD, int kSub>
__global__ void __launch_bounds__(kGaussThreads)
mr_residual_element_kernel(int n_elements, const int *__restrict__ conn_q, const int *__restrict__ conn_l,
                           const double *__restrict__ coords, int nq, const double *__restrict__ dofs,
                           const double *__restrict__ mat, const BasisTables *__restrict__ T,
                           double *__restrict__ relem, double delta, double *__restrict__ kfd)
{
    __shared__ ElementLds s;
    // the Gauss points' results take the place of the planes they have read
    double(*s_T)[27] = s.plane;                                    // [9 le + 3 a + j][g]
    double(*s_rp)[27] = s.plane + kGaussElemsPerBlock * 9;         // [le][g]
    double(*s_PQ)[6] = reinterpret_cast<double(*)[6]>(s.plane + kGaussElemsPerBlock * 10);
    static_assert(kGaussElemsPerBlock * (10 * 27 + 27 * 6) <= kGaussElemsPerBlock * 18 * 27, "results fit the planes");
    const int t = threadIdx.x;
    const int e0 = xcd_block(blockIdx.x, gridDim.x) * kGaussElemsPerBlock;
    const int le = t / 27, g = t % 27, v = e0 + le;
    {
        GaussKinematics k;
        double P;
        const bool active = element_points<kFD>(n_elements, e0, conn_q, conn_l, coords, nq, dofs, delta, s, k, &P);
        double rT[9], rrp = 0.0;
        if (active) {
            const int e = kFD ? v / 89 : v;
            double sigma[6], jgw, J;
            if (kSub == OC_INCOMPRESSIBLE_MOONEY_RIVLIN_SUBTYPE) {
                // the 4-component residual loop of the subtype (:1654-1761):
                // weight w Jxxi Jznu, Jznu from the stress routine
                J = imr_cauchy_stress(k.F, P, mat[2 * e], mat[2 * e + 1], sigma);
                jgw = T->w27[g] * k.jx * J;
            } else {
                mr_cauchy_stress(k.F, k.Jznu, P, mat[2 * e], mat[2 * e + 1], sigma);
                jgw = k.jz * T->w27[g];
                J = k.Jznu;
            }
            // dxidz[j + 3 i] = DXI_DX(j, i)
            for (int a = 0; a < 3; ++a)
                for (int j = 0; j < 3; ++j) {
                    double acc = 0.0;
                    for (int i = 0; i < 3; ++i) acc = fma(k.dxidz[j + 3 * i], jgw * sigma[t2v(i, a)], acc);
                    rT[3 * a + j] = acc;
                }
            rrp = k.jx * T->w27[g] * (J - 1.0);
        }
        __syncthreads();
        if (active) {
#pragma unroll
            for (int i = 0; i < 9; ++i) s_T[9 * le + i][g] = rT[i];
            s_rp[le][g] = rrp;
        }
    }
    __syncthreads();
    const bool mine = t < kGaussElemsPerBlock * 27 && v < n_elements;
    const int a = g / 9;
    if (mine) {  // xi point g / 3 % 3, zeta node g % 3
        const int gx = (g / 3) % 3, mz = g % 3;
        const double q[3] = {pick3(mz, kQuad[0][0], kQuad[0][1], kQuad[0][2]),
                             pick3(mz, kQuad[1][0], kQuad[1][1], kQuad[1][2]),
                             pick3(mz, kQuad[2][0], kQuad[2][1], kQuad[2][2])};
        const double qd[3] = {pick3(mz, kQuadD[0][0], kQuadD[0][1], kQuadD[0][2]),
                              pick3(mz, kQuadD[1][0], kQuadD[1][1], kQuadD[1][2]),
                              pick3(mz, kQuadD[2][0], kQuadD[2][1], kQuadD[2][2])};
        const double(*T3)[27] = s_T + 9 * le + 3 * a;
        double pq[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int h = 0; h < 3; ++h) {
            const int i = gx + 3 * h;
            const double ax = q[0] * T3[0][i] + q[1] * T3[0][i + 9] + q[2] * T3[0][i + 18];
            const double ay = q[0] * T3[1][i] + q[1] * T3[1][i + 9] + q[2] * T3[1][i + 18];
            const double az = qd[0] * T3[2][i] + qd[1] * T3[2][i + 9] + qd[2] * T3[2][i + 18];
#pragma unroll
            for (int my = 0; my < 3; ++my) {
                pq[my] += kQuad[h][my] * az + kQuadD[h][my] * ay;
                pq[3 + my] += kQuad[h][my] * ax;
            }
        }
#pragma unroll
        for (int i = 0; i < 6; ++i) s_PQ[t][i] = pq[i];
    }
    __syncthreads();
    const auto put = [&](int u, int r, double value) {
        if (kFD) {
            const int64_t e = u / 89, col = u % 89;
            kfd[(e * 89 + kbuf_row(r)) * 89 + col] = (value - relem[e * 89 + r]) / delta;
        } else {
            relem[static_cast<int64_t>(u) * 89 + r] = value;
        }
    };
    if (mine) {  // zeta node g / 3 % 3, eta node g % 3
        const int mz = (g / 3) % 3, my = g % 3;
        double p[3], q[3];
#pragma unroll
        for (int gx = 0; gx < 3; ++gx) {
            const double *pq = s_PQ[27 * le + 9 * a + 3 * gx + mz];
            p[gx] = pq[my];
            q[gx] = pq[3 + my];
        }
#pragma unroll
        for (int mx = 0; mx < 3; ++mx) {
            double r = 0.0;
#pragma unroll
            for (int gx = 0; gx < 3; ++gx) r += kQuad[gx][mx] * p[gx] + kQuadD[gx][mx] * q[gx];
            put(v, 27 * a + mx + 3 * my + 9 * mz, r);
        }
    }
    // pressure entries, by the last threads first: they have less to do above
    const int w = kGaussThreads - 1 - t;
    if (w < kGaussElemsPerBlock * 8 && e0 + w / 8 < n_elements) {
        const int m = w % 8;
        double lx[3], ly[3], lz[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            lx[i] = (m & 1) ? kXi[i] : 1.0 - kXi[i];
            ly[i] = (m & 2) ? kXi[i] : 1.0 - kXi[i];
            lz[i] = (m & 4) ? kXi[i] : 1.0 - kXi[i];
        }
        const double *rp = s_rp[w / 8];
        double r = 0.0;
#pragma unroll
        for (int z = 0; z < 3; ++z)
#pragma unroll
            for (int y = 0; y < 3; ++y) {
                const double *row = rp + 3 * y + 9 * z;
                r += lz[z] * ly[y] * (lx[0] * row[0] + lx[1] * row[1] + lx[2] * row[2]);
            }
        put(e0 + w / 8, 81 + m, r);
    }
}

// Schur-complement estimate of the pressure block, S = B K^-1 B^T ~ M_p / mu
// (the pressure mass matrix over the shear modulus, as for Stokes flow):
// lumped, in the current configuration, each element's part divided by its
// linearised shear modulus mu = 2 (c10 + c01).  One thread per pressure node
// sums its elements' integrals of psi_m J_z w (its gather list: entries
// e*89 + 81 + m, ascending elements); inv_p = -1 / S.
__global__ void __launch_bounds__(256)
schur_mass_kernel(int nl, const int *__restrict__ gptr, const int *__restrict__ gidx,
                  const double *__restrict__ rec, const BasisTables *__restrict__ T, const double *__restrict__ mat,
                  double *__restrict__ inv_p)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nl) return;
    double sum = 0.0;
    for (int k = gptr[p]; k < gptr[p + 1]; ++k) {
        const int64_t e = gidx[k] / 89;
        const int m = gidx[k] % 89 - 81;
        double acc = 0.0;
        for (int g = 0; g < 27; ++g) acc += T->lin27[(g * 8 + m) * 4] * rec[(e * GP_NFIELDS + GP_JGW) * 27 + g];
        sum += acc / (2.0 * (mat[2 * e] + mat[2 * e + 1]));
    }
    inv_p[p] = sum > 0.0 ? -1.0 / sum : -1.0;
}

// residual[d] = sum over the element entries of DOF d, ascending elements: four
// indices and then four entries on their way (those past the end repeat the
// last), where a loop of single ones waited twice for each.  859,000 DOFs 28 ->
// 20 us.
__global__ void __launch_bounds__(256)
dof_gather_kernel(int n_rows, const int *__restrict__ ptr, const int *__restrict__ idx,
                  const double *__restrict__ relem, double *__restrict__ out)
{
    const int d = blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= n_rows) return;
    constexpr int kFlight = 4;
    const int k1 = ptr[d + 1];
    double acc = 0.0;
    for (int k = ptr[d]; k < k1; k += kFlight) {
        int j[kFlight];
        double v[kFlight];
#pragma unroll
        for (int u = 0; u < kFlight; ++u) j[u] = idx[min(k + u, k1 - 1)];
#pragma unroll
        for (int u = 0; u < kFlight; ++u) v[u] = relem[j[u]];
#pragma unroll
        for (int u = 0; u < kFlight; ++u)
            if (k + u < k1) acc = acc + v[u];
    }
    out[d] = acc;
}

// element residuals of the set's subtype into relem (kFD: the forward-
// difference columns, `blocks` covering every (element, column) pair)
template <bool kFD>
static int launch_residual_elements(const EquationsSet &s, unsigned blocks, const double *dofs,
                                    const BasisTables *T, double *relem, double delta, double *kfd)
{
    Runtime &rt = runtime();
    const int nv = kFD ? s.n_elements * 89 : s.n_elements;
    if (s.subtype == OC_INCOMPRESSIBLE_MOONEY_RIVLIN_SUBTYPE)
        mr_residual_element_kernel<kFD, OC_INCOMPRESSIBLE_MOONEY_RIVLIN_SUBTYPE><<<blocks, kGaussThreads, 0, rt.stream>>>(
            nv, s.conn.ptr, s.conn_l.ptr, s.coords.ptr, s.n_nodes, dofs, s.mat.ptr, T, relem, delta, kfd);
    else
        mr_residual_element_kernel<kFD, OC_MOONEY_RIVLIN_SUBTYPE><<<blocks, kGaussThreads, 0, rt.stream>>>(
            nv, s.conn.ptr, s.conn_l.ptr, s.coords.ptr, s.n_nodes, dofs, s.mat.ptr, T, relem, delta, kfd);
    OC_HIP_CHECK(hipGetLastError());
    return OC_NO_ERROR;
}

int launch_mr_residual(EquationsSet &s)
{
    OC_CHECK(mr_prepare(s));
    const BasisTables *T = nullptr;
    OC_CHECK(ensure_tables(&T));
    Runtime &rt = runtime();
    const unsigned blocks = static_cast<unsigned>((s.n_elements + kGaussElemsPerBlock - 1) / kGaussElemsPerBlock);
    {
        KernelTimer timer("mr_residual");
        OC_CHECK(launch_residual_elements<false>(s, blocks, s.dofs.ptr, T, s.relem.ptr, 0.0, nullptr));
    }
    {
        KernelTimer timer("dof_gather");
        dof_gather_kernel<<<static_cast<unsigned>((s.n_rows + 255) / 256), 256, 0, rt.stream>>>(
            s.n_rows, s.gather_ptr.ptr, s.gather_idx.ptr, s.relem.ptr, s.residual.ptr);
        OC_HIP_CHECK(hipGetLastError());
    }
    return OC_NO_ERROR;
}

// ---------------------------------------------------------------------------
// Analytic Jacobian (FiniteElasticity_FiniteElementJacobianEvaluate,
// finite_elasticity_routines.f90:842-1175) in two phases.
//
// Phase A (mr_element_matrix_f64_kernel for FP64, mr_element_matrix_f32_kernel
// for FP32; all elements, no colours): for each of the six lower displacement
// blocks (a, b), b <= a,
//   K_(a,m),(b,n) = sum_(g,j) U_g^{ab}[m][j] D_g[j][n],
//   U_g^{ab}[m][j] = sum_i D_g[i][m] W_g[(a,i),(b,j)],
//   W_g[(a,i),(b,j)] = J_z w_g (c(V(i,a),V(j,b)) + delta_ab sigma_ij),
// i.e. the reference's TEMPVEC / DOT_PRODUCT contraction (:1001-1037)
// re-associated as a 27x81 by 81x27 GEMM on MFMA; pressure rows
// K_(p,m),(b,n) = sum_g (J_z w_g psi_m) D_g[b][n] (:1039-1054) as an 8x27 by
// 27x81 GEMM.  U is formed in registers from D and W and never stored.  Lower
// triangle kept, mirrored (:1149-1153); the element matrix goes to an HBM
// buffer, its rows by nodes (kbuf_row).
// Phase B (csr_row_gather_kernel<Real>): one wavefront per node (its three
// displacement rows) or pressure row adds the element rows that touch it, in
// ascending element order, into an LDS copy of the rows and writes them once (no
// zero fill, no read-modify-write).
typedef float mfma_f32x4 __attribute__((ext_vector_type(4)));

// Both element-matrix kernels are persistent (one block of twelve waves per CU)
// and run their elements through a three-stage pipeline.  In slot s
//   * the producers, waves 4..7, build the operands D, W and the pressure
//     operand of element s in one half of double-buffered LDS and load the
//     Gauss-point records of element s + 2;
//   * the consumers, waves 0..3, run the MFMA contraction of element s - 1 from
//     the other half;
//   * the storers, waves 8..11, copy the staged tiles of element s - 2 to its
//     place in the element buffer.
// Between the slot's two barriers the consumers put their accumulators into the
// staging area and the producers the records of element s + 1 into theirs.
//
// The staging area holds the lower blocks and the pressure rows only, as the
// MFMA tiles give them; a storer thread keeps the LDS places of its entries (the
// same for every element), so the mirror image costs no writes, and stores two
// entries of consecutive addresses: the element matrix leaves in contiguous
// kilobytes.  Stored tile by tile from the accumulators it left in requests of 29
// bytes on average (73 million for 32,768 elements), which alone took 620 us.
// 32,768 elements: FP64 805 -> 713 us, where MFMAs and vector instructions take
// turns (see f64_units); 13,100 elements in FP32 307 -> 229 us.
constexpr int kElementThreads = 768;
constexpr int kRoleThreads = 256;  // threads of each of the three roles

// Staging area: lower block q = a (a + 1) / 2 + b as 27 rows of 29 (an odd
// stride: a column read is free of bank conflicts), the pressure rows, a zero
constexpr int kStageRow = 29, kStageBlock = 27 * kStageRow, kStagePRow = 83;
constexpr int kStageP = 6 * kStageBlock, kStageZero = kStageP + 8 * kStagePRow, kStageSize = kStageZero + 1;
constexpr int kEntries = 89 * 89;
constexpr int kStorePairs = ((kEntries + 1) / 2 + kRoleThreads - 1) / kRoleThreads;  // pairs of entries per storer thread

// staging place of entry idx of the 89x89 element buffer: blocks above the
// diagonal mirror those below (:1149-1153), the p-p block is zero
__device__ __forceinline__ int stage_place(int idx)
{
    const int br = idx / 89, j = idx % 89;
    const int r = br < 81 ? (br % 3) * 27 + br / 3 : br;  // the inverse of kbuf_row
    const int hi = max(r, j), lo = min(r, j);
    if (lo >= 81) return kStageZero;
    if (hi >= 81) return kStageP + (hi - 81) * kStagePRow + lo;
    // (a, m) row and (b, n) column of the lower block
    int a = r / 27, m = r % 27, b = j / 27, n = j % 27;
    if (a < b || (a == b && m < n)) {
        int x = a;
        a = b;
        b = x;
        x = m;
        m = n;
        n = x;
    }
    return (a * (a + 1) / 2 + b) * kStageBlock + m * kStageRow + n;
}

// The stores go through a buffer resource over the 89x89 block of one element:
// the lane part of an offset is one register and the rest a constant, so a
// store costs no address arithmetic.
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void store_pair(__amdgpu_buffer_rsrc_t rs, double v0, double v1, int voff, int soff)
{
    const u32x2 a = __builtin_bit_cast(u32x2, v0), b = __builtin_bit_cast(u32x2, v1);
    __builtin_amdgcn_raw_buffer_store_b128(u32x4{a.x, a.y, b.x, b.y}, rs, voff, soff, 0);
}
__device__ __forceinline__ void store_pair(__amdgpu_buffer_rsrc_t rs, float v0, float v1, int voff, int soff)
{
    __builtin_amdgcn_raw_buffer_store_b64(u32x2{__builtin_bit_cast(unsigned, v0), __builtin_bit_cast(unsigned, v1)}, rs,
                                          voff, soff, 0);
}

// the storers' slots: thread st copies the pairs of entries st + 256 i
template <typename Real>
__device__ __forceinline__ void element_storer(int st, int n_mine, int e0, int step, const Real *s_stage,
                                               Real *__restrict__ kbuf)
{
    constexpr int kR = static_cast<int>(sizeof(Real));
    int place[2 * kStorePairs];
#pragma unroll
    for (int i = 0; i < 2 * kStorePairs; ++i)
        place[i] = stage_place(min(2 * (st + kRoleThreads * (i >> 1)) + (i & 1), kEntries - 1));
    const int last = 2 * (st + kRoleThreads * (kStorePairs - 1));
    for (int s = 0; s < n_mine + 2; ++s) {
        if (s >= 2) {
            Real *Ke = kbuf + (e0 + static_cast<int64_t>(s - 2) * step) * kEntries;
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(Ke, 0, kEntries * kR, 0x00020000);
#pragma unroll
            for (int i = 0; i < kStorePairs; ++i) {
                const Real v0 = s_stage[place[2 * i]], v1 = s_stage[place[2 * i + 1]];
                if (i + 1 < kStorePairs || last + 1 < kEntries) store_pair(rs, v0, v1, 2 * kR * st, 2 * kR * kRoleThreads * i);
                else if (last < kEntries) Ke[last] = v0;
            }
        }
        __syncthreads();
        __syncthreads();
    }
}

// The records of one element on their way to LDS: loaded two elements ahead
constexpr int kRec = GP_NFIELDS * 27, kRecPerThread = (kRec + kRoleThreads - 1) / kRoleThreads;
__device__ __forceinline__ void load_records(const double *__restrict__ rec, int64_t e, bool valid, int pt,
                                             double (&v)[kRecPerThread])
{
    const double *r = rec + e * kRec;
#pragma unroll
    for (int i = 0; i < kRecPerThread; ++i)
        v[i] = (valid && (i + 1 < kRecPerThread || pt + kRoleThreads * i < kRec)) ? r[pt + kRoleThreads * i] : 0.0;
}
__device__ __forceinline__ void put_records(double (*s_rec)[27], int pt, const double (&v)[kRecPerThread])
{
    double *r = &s_rec[0][0];
#pragma unroll
    for (int i = 0; i < kRecPerThread; ++i)
        if (i + 1 < kRecPerThread || pt + kRoleThreads * i < kRec) r[pt + kRoleThreads * i] = v[i];
}

// Producer thread pt < 243 owns (j, n) = (rq / 27, rq % 27) of D_g, rq = pt % 81,
// for g = pg + 3k, pg = pt / 81: D_g[j][n] = sum_mi DXI_DX(mi, j) dphi_n/dxi_mi
// (:974-986).  Its table values dphi_n/dxi_mi at those g stay in registers.
struct ProducerTable {
    double d[9][3];
};
__device__ __forceinline__ ProducerTable producer_table(const BasisTables *__restrict__ T, int pt)
{
    const int n = (pt % 81) % 27, pg = pt / 81;
    ProducerTable t;
#pragma unroll
    for (int k = 0; k < 9; ++k)
#pragma unroll
        for (int mi = 0; mi < 3; ++mi) t.d[k][mi] = pt < 243 ? T->quad27[((pg + 3 * k) * 27 + n) * 4 + 1 + mi] : 0.0;
    return t;
}
__device__ __forceinline__ double producer_d(const double (*R)[27], const ProducerTable &t, int dj, int g, int k)
{
    return R[GP_DXIDZ + 0 + 3 * dj][g] * t.d[k][0] + R[GP_DXIDZ + 1 + 3 * dj][g] * t.d[k][1] +
           R[GP_DXIDZ + 2 + 3 * dj][g] * t.d[k][2];
}

// ---- FP32 element matrices: v_mfma_f32_16x16x4f32 -----------------------------
// Per-lane operand slices of D_g[j][n] = sum_mi DXI_DX(mi, j) dphi_n/dxi_mi
// (:974-986).  The contraction index is k = (j, g) with g padded to 28, so
// MFMA k-step ks covers j = ks / 7 and g = 4 (ks % 7) + kk (kk = lane / 16).
// Lane (kk, l) keeps D_g[j][16 t + l] for its seven Gauss points g = 4 g' + kk
// and j = 0..2 in D[t][g'][j] (t = 0, 1: the two 16-wide tiles of the 27 basis
// functions).  These registers are the B operand of every displacement block
// and, contracted with W, form its A operand
//   U^{ab}_g[m][j] = sum_i D_g[i][m] W_g[(a,i),(b,j)]
// on the fly, so U never goes through LDS.
struct DSlice {
    float v[2][7][3];
};

// One displacement block (A, B), row tile MT, column tiles 0 (and 1 if TWO)
template <int A, int B, int MT, bool TWO>
struct F32Unit {
    static constexpr int a = A, b = B, mt = MT;
    static constexpr bool two = TWO;
};

// accumulator register r of a lane holds row 4 (lane / 16) + r, column lane % 16
template <typename U>
__device__ __forceinline__ void f32_unit(int lane, const DSlice &D, const float (*s_W)[81], mfma_f32x4 (&acc)[2])
{
    const int kk = lane >> 4;
    acc[0] = acc[1] = mfma_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // k-step s = 7 j + gp; software pipeline: the W loads of step s + 2 and
    // the A operand of step s + 1 are issued behind the MFMAs of step s, and a
    // scheduling barrier per step keeps that order (and the register count)
    const float *wbase = &s_W[kk][U::a * 27 + U::b * 3];
    auto load_w = [&](int st, float *w) {
        const float *p = wbase + (4 * (st % 7)) * 81 + st / 7;
        w[0] = p[0];
        w[1] = p[9];
        w[2] = p[18];
    };
    auto a_operand = [&](int st, const float *w) {
        const int gp = st % 7;
        return D.v[U::mt][gp][0] * w[0] + D.v[U::mt][gp][1] * w[1] + D.v[U::mt][gp][2] * w[2];
    };
    float wq[2][3];
    load_w(0, wq[0]);
    load_w(1, wq[1]);
    float u = a_operand(0, wq[0]);
#pragma unroll
    for (int st = 0; st < 21; ++st) {
        const int j = st / 7, gp = st % 7;
        if (st + 2 < 21) load_w(st + 2, wq[st & 1]);
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(u, D.v[0][gp][j], acc[0], 0, 0, 0);
        if (U::two) acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(u, D.v[1][gp][j], acc[1], 0, 0, 0);
        if (st + 1 < 21) u = a_operand(st + 1, wq[(st + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// entry (m, n), m = MT*16 + 4 (lane / 16) + r, n = nt*16 + lane % 16, of a
// unit's tiles into the staging area
template <typename U>
__device__ __forceinline__ void f32_unit_stage(int lane, const mfma_f32x4 (&acc)[2], float *s_stage)
{
    const int l = lane & 15, row0 = U::mt * 16 + 4 * (lane >> 4);
    float *o = s_stage + (U::a * (U::a + 1) / 2 + U::b) * kStageBlock + row0 * kStageRow + l;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (row0 + r >= 27) continue;
#pragma unroll
        for (int nt = 0; nt < (U::two ? 2 : 1); ++nt)
            if (nt == 0 || 16 + l < 27) o[r * kStageRow + 16 * nt] = acc[nt][r];
    }
}

// Pressure rows K_(p,m),(b,n) = sum_g (J_z w_g psi_m(g)) D_g[b][n]
// (:1039-1054): k = g only, so k-step ks is g = 4 ks + kk and the B operand
// is D[t][ks][b]; six 16x16 tiles acc[b][t], rows 8..15 padding
__device__ __forceinline__ void f32_pressure(int lane, const DSlice &D, const float *s_Pa, mfma_f32x4 (&acc)[3][2])
{
    const int kk = lane >> 4, l = lane & 15;
#pragma unroll
    for (int b = 0; b < 3; ++b) acc[b][0] = acc[b][1] = mfma_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ks = 0; ks < 7; ++ks) {
        const float pa = s_Pa[(4 * ks + kk) * 16 + l];
#pragma unroll
        for (int b = 0; b < 3; ++b)
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa, D.v[t][ks][b], acc[b][t], 0, 0, 0);
    }
}

__device__ __forceinline__ void f32_pressure_stage(int lane, const mfma_f32x4 (&acc)[3][2], float *s_stage)
{
    const int l = lane & 15, row0 = 4 * (lane >> 4);
    if (row0 >= 8) return;
    float *o = s_stage + kStageP + row0 * kStagePRow + l;
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (t == 0 || 16 + l < 27) o[r * kStagePRow + b * 27 + t * 16] = acc[b][t][r];
}

// the slots of consumer wave kWave (0..3)
template <int kWave>
__device__ __forceinline__ void f32_consumer(int lane, int n_mine, const float (*s_D)[28][3][32], const float (*s_W)[28][81],
                                             const float (*s_Pa)[28 * 16], float *s_stage)
{
    // 483 MFMA k-steps per element over four waves (126/126/126/105)
    using U0 = std::conditional_t<kWave == 0, F32Unit<1, 0, 0, true>, std::conditional_t<kWave == 1, F32Unit<2, 0, 0, true>,
               std::conditional_t<kWave == 2, F32Unit<2, 1, 0, true>, F32Unit<0, 0, 0, false>>>>;
    using U1 = std::conditional_t<kWave == 0, F32Unit<1, 0, 1, true>, std::conditional_t<kWave == 1, F32Unit<2, 0, 1, true>,
               std::conditional_t<kWave == 2, F32Unit<2, 1, 1, true>, F32Unit<1, 1, 0, false>>>>;
    using U2 = std::conditional_t<kWave == 0, F32Unit<0, 0, 1, true>, std::conditional_t<kWave == 1, F32Unit<1, 1, 1, true>,
               std::conditional_t<kWave == 2, F32Unit<2, 2, 1, true>, F32Unit<2, 2, 0, false>>>>;
    for (int s = 0; s < n_mine + 2; ++s) {
        // the lane index is made opaque per element so that the offsets
        // derived from it are recomputed here rather than held across the loop
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const bool work = s >= 1 && s - 1 < n_mine;
        mfma_f32x4 acc[3][2], accp[3][2];
        if (work) {
            const int p = (s - 1) & 1, kk = ln >> 4, l = ln & 15;
            DSlice D;
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int gp = 0; gp < 7; ++gp)
#pragma unroll
                    for (int j = 0; j < 3; ++j) D.v[tt][gp][j] = s_D[p][4 * gp + kk][j][16 * tt + l];
            const float(*W)[81] = s_W[p];
            if (kWave == 3) f32_pressure(ln, D, s_Pa[p], accp);
            __builtin_amdgcn_sched_barrier(0);
            f32_unit<U0>(ln, D, W, acc[0]);
            f32_unit<U1>(ln, D, W, acc[1]);
            f32_unit<U2>(ln, D, W, acc[2]);
        }
        __syncthreads();
        if (work) {
            if (kWave == 3) f32_pressure_stage(ln, accp, s_stage);
            f32_unit_stage<U0>(ln, acc[0], s_stage);
            f32_unit_stage<U1>(ln, acc[1], s_stage);
            f32_unit_stage<U2>(ln, acc[2], s_stage);
        }
        __syncthreads();
    }
}

__global__ void __launch_bounds__(kElementThreads)
mr_element_matrix_f32_kernel(int n_elements, const double *__restrict__ rec, const BasisTables *__restrict__ T,
                             float *__restrict__ kbuf)
{
    __shared__ double s_rec[52][27];     // Gauss-point records
    __shared__ float s_D[2][28][3][32];  // D_g[j][n]; g = 27 and n >= 27 zero
    __shared__ float s_W[2][28][81];     // W_g[(a,i),(b,j)] at [g][(3a+i)*9 + 3b+j]; g = 27 zero
    __shared__ float s_Pa[2][28 * 16];   // J_z w_g psi_m(g) at [g*16 + m]; m >= 8 and g = 27 zero
    __shared__ float s_stage[kStageSize];
    const int t = threadIdx.x, lane = t & 63;
    const int role = __builtin_amdgcn_readfirstlane(t >> 6);
    const int e0 = static_cast<int>(blockIdx.x), step = static_cast<int>(gridDim.x);
    const int n_mine = e0 < n_elements ? (n_elements - 1 - e0) / step + 1 : 0;
    for (int k = t; k < 2 * 28 * 3 * 32; k += kElementThreads) (&s_D[0][0][0][0])[k] = 0.0f;
    for (int k = t; k < 2 * 28 * 81; k += kElementThreads) (&s_W[0][0][0])[k] = 0.0f;
    for (int k = t; k < 2 * 28 * 16; k += kElementThreads) (&s_Pa[0][0])[k] = 0.0f;
    if (t == 0) s_stage[kStageZero] = 0.0f;
    // every wave passes the barriers of each slot in a loop of its own role
    if (role < 4 || role >= 8) {
        __syncthreads();
        switch (role) {
        case 0: f32_consumer<0>(lane, n_mine, s_D, s_W, s_Pa, s_stage); break;
        case 1: f32_consumer<1>(lane, n_mine, s_D, s_W, s_Pa, s_stage); break;
        case 2: f32_consumer<2>(lane, n_mine, s_D, s_W, s_Pa, s_stage); break;
        case 3: f32_consumer<3>(lane, n_mine, s_D, s_W, s_Pa, s_stage); break;
        default: element_storer<float>(t - 2 * kRoleThreads, n_mine, e0, step, s_stage, kbuf); break;
        }
        return;
    }
    const int pt = t - kRoleThreads;
    const ProducerTable tab = producer_table(T, pt);
    const double psi = pt < 27 * 8 ? T->lin27[pt * 4] : 0.0;  // psi_m(g) at g = pt / 8, m = pt % 8
    // thread pt < 243 also owns column rq of W_g (row (a,i), column (b,j))
    const int rq = pt % 81, pg = pt / 81, dj = rq / 27, dn = rq % 27;
    const int wa = rq / 27, wi = (rq / 9) % 3, wb = (rq % 9) / 3, wj = rq % 3;
    const int wf1 = GP_C + t2v(wi, wa) + 6 * t2v(wj, wb), wf2 = GP_SIGJ + t2v(wi, wj);
    const bool wdiag = wa == wb;
    double pre[kRecPerThread];
    load_records(rec, e0, n_mine > 0, pt, pre);
    put_records(s_rec, pt, pre);
    load_records(rec, e0 + step, n_mine > 1, pt, pre);
    __syncthreads();
    for (int s = 0; s < n_mine + 2; ++s) {
        double nxt[kRecPerThread];
        load_records(rec, e0 + static_cast<int64_t>(s + 2) * step, s + 2 < n_mine, pt, nxt);
        if (s < n_mine) {
            const int p = s & 1;
            const double(*R)[27] = s_rec;
            // all LDS reads of a phase before its writes: one round trip
            if (pt < 243) {  // g = pg + 3k
                float dv[9], wv[9];
#pragma unroll
                for (int k = 0; k < 9; ++k) dv[k] = static_cast<float>(producer_d(R, tab, dj, pg + 3 * k, k));
#pragma unroll
                for (int k = 0; k < 9; ++k) s_D[p][pg + 3 * k][dj][dn] = dv[k];
#pragma unroll
                for (int k = 0; k < 9; ++k) {
                    const int g = pg + 3 * k;
                    double v = R[wf1][g];
                    if (wdiag) v = v + R[wf2][g];
                    wv[k] = static_cast<float>(R[GP_JGW][g] * v);
                }
#pragma unroll
                for (int k = 0; k < 9; ++k) s_W[p][pg + 3 * k][rq] = wv[k];
            }
            if (pt < 27 * 8) s_Pa[p][pt / 8 * 16 + pt % 8] = static_cast<float>(R[GP_JGW][pt / 8] * psi);
        }
        __syncthreads();
        put_records(s_rec, pt, pre);
#pragma unroll
        for (int i = 0; i < kRecPerThread; ++i) pre[i] = nxt[i];
        __syncthreads();
    }
}

// ---- FP64 element matrices: v_mfma_f64_4x4x4f64 ---------------------------------
// Four 4x4x4 blocks per instruction; lane = c + 4 blk + 16 h holds A_blk[c][h],
// B_blk[h][c] and the result D_blk[h][c].  The FP64 16x16x4 instruction runs at
// about 60% of the 4x4x4 rate here, and the 4-wide tiles also pad 27 to 28
// instead of 32.  A consumer instruction covers the row tiles I = 4t + blk of one
// displacement block (rows m = 16t + 4blk + i) against one column tile J
// (n = 4J + j):
//   A = U^{ab}_g[16t + l][j_dim] from D and W (l = c + 4 blk),
//   B = D_g[j_dim][4J + c], shared by the four row tiles, read from LDS;
// k-step s covers g = 4 (s / 3) + h and j_dim = s % 3.  Lower block (a, b) is
// numbered q = a (a + 1) / 2 + b (F64Unit).
// An FP64 MFMA and a vector instruction do not overlap here, not even from two
// wavefronts of a SIMD (16 of the one and 64 of the other take the sum of their
// times), and alternating them costs 13 cycles a switch: so the SIMD's time is
// that of its MFMAs plus that of all its wavefronts' vector instructions, and
// the kernel keeps those few and together.
__device__ __forceinline__ double2 lds_pair(const double *p) { return *reinterpret_cast<const double2 *>(p); }

template <int Q, int T, int NJ>
struct F64Unit {
    static constexpr int q = Q, t = T, nj = NJ;
    static constexpr int a = Q == 0 ? 0 : (Q <= 2 ? 1 : 2);
    static constexpr int b = Q - (a * (a + 1)) / 2;
};

// the tiles of one unit into the staging area: acc[J] at m = 16T + 4blk + h,
// n = 4J + c
template <typename U>
__device__ __forceinline__ void f64_unit_stage(int lane, const double *acc, double *s_stage)
{
    const int c = lane & 3, m = 16 * U::t + (lane & 12) + (lane >> 4);
    if (m >= 27) return;
    double *o = s_stage + U::q * kStageBlock + m * kStageRow + c;
#pragma unroll
    for (int J = 0; J < U::nj; ++J)
        if (J < 6 || c < 3) o[4 * J] = acc[J];
}

// LDS layouts.  D_g[j][n] at [g][j][n % 4][n / 4], the Gauss points 98 doubles
// apart: the four g of a 16-byte read then fall on different banks.  W_g[(a,i),
// (b,j)] of lower block q at [g][q][j][i], i padded to 4.
constexpr int kDStride = 98, kWStride = 72;

// three units of one wave, all on row half T, sharing the B reads of every
// k-step; the operands of step s + 1 are loaded and formed while the MFMAs of
// step s run
template <int T, typename U0, typename U1, typename U2>
__device__ __forceinline__ void f64_units(int lane, const double *sD, const double *sW, double (&acc)[3][7])
{
    const int c = lane & 3, blk = (lane >> 2) & 3, h = lane >> 4;
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
        for (int J = 0; J < 7; ++J) acc[x][J] = 0.0;
    double B[2][7], W[2][3][3], DT[2][3], u[2][3];  // DT: D_g[i][16t + 4blk + c]
    auto load_b = [&](int st, double (&b)[7]) {
        const double *bp = sD + (4 * (st / 3) + h) * kDStride + (st % 3 * 4 + c) * 8;  // D_g[jd][4J + c], J = 0..6
        const double2 b01 = lds_pair(bp), b23 = lds_pair(bp + 2), b45 = lds_pair(bp + 4);
        b[0] = b01.x; b[1] = b01.y; b[2] = b23.x; b[3] = b23.y; b[4] = b45.x; b[5] = b45.y; b[6] = bp[6];
    };
    auto load_w = [&](int st, double (&w)[3][3]) {
        const int qs[3] = {U0::q, U1::q, U2::q};
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            const double *wp = sW + (4 * (st / 3) + h) * kWStride + (qs[x] * 3 + st % 3) * 4;  // W_g[(a,i),(b,jd)], i = 0..2
            const double2 w01 = lds_pair(wp);
            w[x][0] = w01.x; w[x][1] = w01.y; w[x][2] = wp[2];
        }
    };
    auto load_dt = [&](int gp, double (&d)[3]) {
        const double *dp = sD + (4 * gp + h) * kDStride + c * 8 + 4 * T + blk;
#pragma unroll
        for (int i = 0; i < 3; ++i) d[i] = dp[i * 32];
    };
    auto a_operands = [](const double (&d)[3], const double (&w)[3][3], double (&o)[3]) {
#pragma unroll
        for (int x = 0; x < 3; ++x) o[x] = d[0] * w[x][0] + d[1] * w[x][1] + d[2] * w[x][2];
    };
    load_dt(0, DT[0]);
    load_w(0, W[0]);
    load_w(1, W[1]);
    load_b(0, B[0]);
    a_operands(DT[0], W[0], u[0]);
#pragma unroll
    for (int st = 0; st < 21; ++st) {
        const int cur = st & 1;
        if (st + 1 < 21) a_operands(DT[((st + 1) / 3) & 1], W[cur ^ 1], u[cur ^ 1]);
        if (st + 1 < 21) load_b(st + 1, B[cur ^ 1]);
        if (st + 2 < 21) load_w(st + 2, W[cur]);
        if (st % 3 == 0 && st / 3 + 1 < 7) load_dt(st / 3 + 1, DT[(st / 3 + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int J = 0; J < 7; ++J) {
            if (J < U0::nj) acc[0][J] = __builtin_amdgcn_mfma_f64_4x4x4f64(u[cur][0], B[cur][J], acc[0][J], 0, 0, 0);
            if (J < U1::nj) acc[1][J] = __builtin_amdgcn_mfma_f64_4x4x4f64(u[cur][1], B[cur][J], acc[1][J], 0, 0, 0);
            if (J < U2::nj) acc[2][J] = __builtin_amdgcn_mfma_f64_4x4x4f64(u[cur][2], B[cur][J], acc[2][J], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// pressure rows K_(p,m),(b,n): acc[b][I][t] at m = 4I + h, n = 16t + 4blk + c; the
// B operand D_g[b][n] comes from LDS
__device__ __forceinline__ void f64_pressure(int lane, const double *sD, const double *sPa, double (&acc)[3][2][2])
{
    const int c = lane & 3, blk = (lane >> 2) & 3, h = lane >> 4;
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        acc[b][0][0] = acc[b][0][1] = acc[b][1][0] = acc[b][1][1] = 0.0;
#pragma unroll
        for (int gp = 0; gp < 7; ++gp) {
            const int g = 4 * gp + h;
            const double *pp = sPa + g * 8 + c;
            const double a0 = pp[0], a1 = pp[4];
            const double *bp = sD + g * kDStride + (b * 4 + c) * 8 + blk;  // D_g[b][16t + 4blk + c] at +4t
            const double b0 = bp[0], b1 = bp[4];
            acc[b][0][0] = __builtin_amdgcn_mfma_f64_4x4x4f64(a0, b0, acc[b][0][0], 0, 0, 0);
            acc[b][1][0] = __builtin_amdgcn_mfma_f64_4x4x4f64(a1, b0, acc[b][1][0], 0, 0, 0);
            acc[b][0][1] = __builtin_amdgcn_mfma_f64_4x4x4f64(a0, b1, acc[b][0][1], 0, 0, 0);
            acc[b][1][1] = __builtin_amdgcn_mfma_f64_4x4x4f64(a1, b1, acc[b][1][1], 0, 0, 0);
        }
    }
}

__device__ __forceinline__ void f64_pressure_stage(int lane, const double (&acc)[3][2][2], double *s_stage)
{
    const int n0 = lane & 15, h = lane >> 4;
    double *o = s_stage + kStageP + h * kStagePRow + n0;
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
        for (int I = 0; I < 2; ++I)
#pragma unroll
            for (int t = 0; t < 2; ++t)
                if (t == 0 || 16 + n0 < 27) o[4 * I * kStagePRow + b * 27 + 16 * t] = acc[b][I][t];
}

// the slots of consumer wave kWave (0..3): waves 0, 1 take row half t = 0 (and
// the pressure rows), waves 2, 3 t = 1; 1659 k-steps per element: 378 / 399 /
// 441 / 441
template <int kWave>
__device__ __forceinline__ void f64_consumer(int lane, int n_mine, const double (*s_D)[28 * kDStride],
                                             const double (*s_W)[28 * kWStride], const double (*s_Pa)[28][8],
                                             double *s_stage)
{
    constexpr int kT = kWave >> 1;
    using U0 = F64Unit<(kWave & 1) ? 4 : 1, kT, 7>;
    using U1 = F64Unit<(kWave & 1) ? 2 : 3, kT, kWave == 1 ? 4 : 7>;
    using U2 = F64Unit<(kWave & 1) ? 5 : 0, kT, kT == 0 ? 4 : 7>;
    for (int s = 0; s < n_mine + 2; ++s) {
        // the lane index is made opaque per element so that offsets derived
        // from it are recomputed here rather than held across the loop
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const bool work = s >= 1 && s - 1 < n_mine;
        double acc[3][7], accp[3][2][2];
        if (work) {
            const int p = (s - 1) & 1;
            if (kWave == 1) f64_pressure(ln, s_D[p], &s_Pa[p][0][0], accp);
            f64_units<kT, U0, U1, U2>(ln, s_D[p], s_W[p], acc);
        }
        __syncthreads();
        if (work) {
            if (kWave == 1) f64_pressure_stage(ln, accp, s_stage);
            f64_unit_stage<U0>(ln, acc[0], s_stage);
            f64_unit_stage<U1>(ln, acc[1], s_stage);
            f64_unit_stage<U2>(ln, acc[2], s_stage);
        }
        __syncthreads();
    }
}

__global__ void __launch_bounds__(kElementThreads)
mr_element_matrix_f64_kernel(int n_elements, const double *__restrict__ rec, const BasisTables *__restrict__ T,
                             double *__restrict__ kbuf)
{
    __shared__ double s_rec[52][27];                        // Gauss-point records
    __shared__ __align__(16) double s_D[2][28 * kDStride];  // padding zero
    __shared__ __align__(16) double s_W[2][28 * kWStride];  // padding zero
    __shared__ double s_Pa[2][28][8];                       // J_z w_g psi_m(g); g = 27 zero
    __shared__ double s_stage[kStageSize];
    const int t = threadIdx.x, lane = t & 63;
    const int role = __builtin_amdgcn_readfirstlane(t >> 6);
    const int e0 = static_cast<int>(blockIdx.x), step = static_cast<int>(gridDim.x);
    const int n_mine = e0 < n_elements ? (n_elements - 1 - e0) / step + 1 : 0;
    for (int k = t; k < 2 * 28 * kDStride; k += kElementThreads) (&s_D[0][0])[k] = 0.0;
    for (int k = t; k < 2 * 28 * kWStride; k += kElementThreads) (&s_W[0][0])[k] = 0.0;
    for (int k = t; k < 2 * 28 * 8; k += kElementThreads) (&s_Pa[0][0][0])[k] = 0.0;
    if (t == 0) s_stage[kStageZero] = 0.0;
    // every wave passes the barriers of each slot in a loop of its own role
    if (role < 4 || role >= 8) {
        __syncthreads();
        switch (role) {
        case 0: f64_consumer<0>(lane, n_mine, s_D, s_W, s_Pa, s_stage); break;
        case 1: f64_consumer<1>(lane, n_mine, s_D, s_W, s_Pa, s_stage); break;
        case 2: f64_consumer<2>(lane, n_mine, s_D, s_W, s_Pa, s_stage); break;
        case 3: f64_consumer<3>(lane, n_mine, s_D, s_W, s_Pa, s_stage); break;
        default: element_storer<double>(t - 2 * kRoleThreads, n_mine, e0, step, s_stage, kbuf); break;
        }
        return;
    }
    const int pt = t - kRoleThreads;
    const ProducerTable tab = producer_table(T, pt);
    const double psi = pt < 27 * 8 ? T->lin27[pt * 4] : 0.0;  // psi_m(g) at g = pt / 8, m = pt % 8
    const int rq = pt % 81, pg = pt / 81, dj = rq / 27, dn = rq % 27;
    // pt < 216 owns (q, j, i) = wq of W_g for g = pw (mod 4)
    const int wq = pt % 54, pw = pt / 54;
    const int wqq = wq / 9, wj = (wq / 3) % 3, wi = wq % 3;
    const int wa = wqq == 0 ? 0 : (wqq <= 2 ? 1 : 2), wb = wqq - (wa * (wa + 1)) / 2;
    const int wf1 = GP_C + t2v(wi, wa) + 6 * t2v(wj, wb), wf2 = GP_SIGJ + t2v(wi, wj);
    const bool wdiag = wa == wb;
    double pre[kRecPerThread];
    load_records(rec, e0, n_mine > 0, pt, pre);
    put_records(s_rec, pt, pre);
    load_records(rec, e0 + step, n_mine > 1, pt, pre);
    __syncthreads();
    for (int s = 0; s < n_mine + 2; ++s) {
        double nxt[kRecPerThread];
        load_records(rec, e0 + static_cast<int64_t>(s + 2) * step, s + 2 < n_mine, pt, nxt);
        if (s < n_mine) {
            const int p = s & 1;
            const double(*R)[27] = s_rec;
            // every LDS read of a phase is issued before its writes (which
            // the compiler may not move reads across), so a phase waits
            // for one LDS round trip rather than one per Gauss point
            if (pt < 243) {  // g = pg + 3k
                double dv[9];
#pragma unroll
                for (int k = 0; k < 9; ++k) dv[k] = producer_d(R, tab, dj, pg + 3 * k, k);
#pragma unroll
                for (int k = 0; k < 9; ++k) s_D[p][(pg + 3 * k) * kDStride + (dj * 4 + dn % 4) * 8 + dn / 4] = dv[k];
            }
            if (pt < 216) {  // W_g[(a,i),(b,j)] = J_z w_g (c + delta_ab sigma_ij), g = pw + 4k < 27
                double wv[7];
#pragma unroll
                for (int k = 0; k < 7; ++k) {
                    const int g = min(pw + 4 * k, 26);
                    double v = R[wf1][g];
                    if (wdiag) v = v + R[wf2][g];
                    wv[k] = R[GP_JGW][g] * v;
                }
                const double pa = R[GP_JGW][pt / 8] * psi;
#pragma unroll
                for (int k = 0; k < 7; ++k)
                    if (pw + 4 * k < 27) s_W[p][(pw + 4 * k) * kWStride + (wqq * 3 + wj) * 4 + wi] = wv[k];
                s_Pa[p][pt / 8][pt % 8] = pa;
            }
        }
        __syncthreads();
        put_records(s_rec, pt, pre);
#pragma unroll
        for (int i = 0; i < kRecPerThread; ++i) pre[i] = nxt[i];
        __syncthreads();
    }
}

// kN element rows of one pressure row: every global load before the LDS adds.  The
// addresses are uniform and advance by scalar multiplies.
template <int kN, typename Real>
__device__ __forceinline__ void gather_rows(const int2 *__restrict__ list, int lane, bool hi, int m0, int m1,
                                            int blk0, int blk1, const Real *__restrict__ kbuf,
                                            const uint8_t *__restrict__ rank, Real *s_row)
{
    Real v0[kN], v1[kN];
    int o0[kN], o1[kN];
#pragma unroll
    for (int c = 0; c < kN; ++c) {
        const int2 at = list[c];
        const Real *k = kbuf + static_cast<int64_t>(at.x) * 89;
        const uint8_t *rk = rank + static_cast<int64_t>(at.y) * kRankNodes;
        v0[c] = k[lane];
        o0[c] = rk[m0];
        if (hi) {
            v1[c] = k[lane + 64];
            o1[c] = rk[m1];
        }
    }
    // the adds of one element row complete before the next one's: a
    // wavefront's LDS instructions run in order, and the barrier (no
    // instruction) keeps all lanes together, so that the compiler does not
    // take the lanes with and without a second column one after the other
#pragma unroll
    for (int c = 0; c < kN; ++c) {
        s_row[blk0 + o0[c]] += v0[c];
        if (hi) s_row[blk1 + o1[c]] += v1[c];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// The same for a displacement node's three rows, 267 consecutive entries of each
// of its elements: lane l takes entries l + 64 u; pos[u] is an entry's LDS row
// and component block, m[u] the element node whose rank places it.  The 35
// ranks are loaded once, a lane a node, and handed round.
constexpr int kNodeEntries = 3 * 89, kNodeLoads = (kNodeEntries + 63) / 64, kNodeLast = kNodeEntries - 64 * (kNodeLoads - 1);
template <int kN, typename Real>
__device__ __forceinline__ void gather_node(const int2 *__restrict__ list, int lane, const int (&pos)[kNodeLoads],
                                            const int (&m)[kNodeLoads], const Real *__restrict__ kbuf,
                                            const uint8_t *__restrict__ rank, Real *s_rows)
{
    Real v[kN][kNodeLoads];
    int rk[kN];
#pragma unroll
    for (int c = 0; c < kN; ++c) {
        const int2 at = list[c];
        const Real *k = kbuf + static_cast<int64_t>(at.x) * 89;
        rk[c] = rank[static_cast<int64_t>(at.y) * kRankNodes + min(lane, kRankNodes - 1)];
#pragma unroll
        for (int u = 0; u < kNodeLoads; ++u) v[c][u] = k[64 * u + (u + 1 < kNodeLoads ? lane : min(lane, kNodeLast - 1))];
    }
    // an element's entries have places of their own, so its reads all go before
    // its writes: one LDS latency an element
#pragma unroll
    for (int c = 0; c < kN; ++c) {
        int o[kNodeLoads];
#pragma unroll
        for (int u = 0; u < kNodeLoads; ++u) o[u] = pos[u] + __shfl(rk[c], m[u]);
        Real t[kNodeLoads];
#pragma unroll
        for (int u = 0; u < kNodeLoads; ++u) t[u] = s_rows[o[u]];
#pragma unroll
        for (int u = 0; u < kNodeLoads; ++u)
            if (u + 1 < kNodeLoads || lane < kNodeLast) s_rows[o[u]] = t[u] + v[c][u];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// One wavefront per displacement node (its three CSR rows) and per pressure row,
// kGatherWaves to a block.  A node's element rows lie next to each other in the
// element buffer and share the lists and the neighbour ranks.  Requests waiting
// for lines that others have on their way bounded one wavefront a row (73% of
// its time in FP32): its two loads of an element row and its two rank loads met
// in the same lines, as did the three rows'.  The element rows are taken in
// groups of kMax, ..., 2, 1: with a test per row the scalar instructions took
// three times the vector ones' issue slots.
// 32,768 elements FP64: 788 -> 721 us (3.8 GB); 13,100 elements FP32 293 -> 185 us,
// 4,301 elements 77 -> 54 us.  Two wavefronts a block: 769 us with four, 779 with one.
constexpr int kGatherWaves = 2;

template <typename Real, int kMax>
__global__ void __launch_bounds__(64 * kGatherWaves)
csr_row_gather_kernel(int nq, int nl, int n_elements, int max_row, const int64_t *__restrict__ row_ptr,
                      const int *__restrict__ gptr, const int2 *__restrict__ lists, const Real *__restrict__ kbuf,
                      const uint8_t *__restrict__ rank, const uint16_t *__restrict__ row_nb, Real *__restrict__ values)
{
    extern __shared__ unsigned char s_raw[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    Real *s_rows = reinterpret_cast<Real *>(s_raw) + wave * 3 * max_row;  // a wavefront's own: no block barriers
    const int b = blockIdx.x * kGatherWaves + wave;
    if (b >= nq + nl) return;
    const bool disp = b < nq;
    const int r = disp ? b : 3 * nq + (b - nq);
    const int g0 = gptr[r], n = gptr[r + 1] - g0;
    const int2 *list = lists + (disp ? g0 : g0 - 54 * n_elements);
    const int64_t r0 = row_ptr[r];
    const int len = static_cast<int>(row_ptr[r + 1] - r0);
    const int nb = row_nb[r];
    const auto block = [&](int j) { return j < 81 ? (j / 27) * nb : 3 * nb; };
    const auto node = [&](int j) { return j < 81 ? j % 27 : 27 + j - 81; };
    int c = 0;
    if (!disp) {
        for (int k = lane; k < len; k += 64) s_rows[k] = Real(0);
        __builtin_amdgcn_wave_barrier();
        // lane j holds element columns j and j + 64: component block and rank slot
        const bool hi = lane + 64 < 89;
        const int blk0 = block(lane), m0 = node(lane), blk1 = block(min(lane + 64, 88)), m1 = node(min(lane + 64, 88));
        for (; c + 4 <= n; c += 4) gather_rows<4>(list + c, lane, hi, m0, m1, blk0, blk1, kbuf, rank, s_rows);
        if (n - c >= 2) {
            gather_rows<2>(list + c, lane, hi, m0, m1, blk0, blk1, kbuf, rank, s_rows);
            c += 2;
        }
        if (n - c >= 1) gather_rows<1>(list + c, lane, hi, m0, m1, blk0, blk1, kbuf, rank, s_rows);
        for (int k = lane; k < len; k += 64) values[r0 + k] = s_rows[k];
        return;
    }
    const int64_t r1 = row_ptr[nq + b], r2 = row_ptr[2 * static_cast<int64_t>(nq) + b];
    for (int k = lane; k < len; k += 64) s_rows[k] = s_rows[max_row + k] = s_rows[2 * max_row + k] = Real(0);
    __builtin_amdgcn_wave_barrier();
    int pos[kNodeLoads], m[kNodeLoads];
#pragma unroll
    for (int u = 0; u < kNodeLoads; ++u) {
        const int k = min(64 * u + lane, kNodeEntries - 1);
        pos[u] = (k / 89) * max_row + block(k % 89);
        m[u] = node(k % 89);
    }
    for (; c + kMax <= n; c += kMax) gather_node<kMax>(list + c, lane, pos, m, kbuf, rank, s_rows);
    if (kMax > 8 && n - c >= 8) {
        gather_node<8>(list + c, lane, pos, m, kbuf, rank, s_rows);
        c += 8;
    }
    if (kMax > 4 && n - c >= 4) {
        gather_node<4>(list + c, lane, pos, m, kbuf, rank, s_rows);
        c += 4;
    }
    if (kMax > 2 && n - c >= 2) {
        gather_node<2>(list + c, lane, pos, m, kbuf, rank, s_rows);
        c += 2;
    }
    if (n - c >= 1) gather_node<1>(list + c, lane, pos, m, kbuf, rank, s_rows);
    for (int k = lane; k < len; k += 64) {
        values[r0 + k] = s_rows[k];
        values[r1 + k] = s_rows[max_row + k];
        values[r2 + k] = s_rows[2 * max_row + k];
    }
}

// The element rows a wavefront gathers at once: eight where the mesh leaves
// wavefronts of the GPU idle, as the round trips are all there is to wait for
// then, else four
int row_gather_default(const EquationsSet &s) { return s.n_nodes + s.n_nodes_l <= 8 * runtime().num_cus ? 8 : 4; }

template <typename Real>
static int launch_row_gather(EquationsSet &s, const Real *kbuf, Real *values, int chunk)
{
    Runtime &rt = runtime();
    const size_t lds = static_cast<size_t>(3 * kGatherWaves) * s.max_row_len * sizeof(Real);
    const unsigned grid = static_cast<unsigned>((static_cast<int64_t>(s.n_nodes) + s.n_nodes_l + kGatherWaves - 1) / kGatherWaves);
#define OC_ROW_GATHER(C)                                                                                            \
    csr_row_gather_kernel<Real, C><<<grid, 64 * kGatherWaves, lds, rt.stream>>>(                                   \
        s.n_nodes, s.n_nodes_l, s.n_elements, s.max_row_len, s.row_ptr.ptr, s.gather_ptr.ptr,                      \
        reinterpret_cast<const int2 *>(s.row_lists.ptr), kbuf, s.col_rank.ptr, s.row_nb.ptr, values)
    switch (chunk > 0 ? chunk : row_gather_default(s)) {
    case 8: OC_ROW_GATHER(8); break;
    case 16: OC_ROW_GATHER(16); break;
    default: OC_ROW_GATHER(4); break;
    }
#undef OC_ROW_GATHER
    OC_HIP_CHECK(hipGetLastError());
    return OC_NO_ERROR;
}

int launch_schur_mass(EquationsSet &s, double *inv_p)
{
    if (!s.gp_records.ptr || s.subtype != OC_MOONEY_RIVLIN_SUBTYPE)
        return set_error(OC_ERR_UNSUPPORTED, "the pressure-mass Schur estimate needs the analytic Jacobian's Gauss records");
    const BasisTables *T = nullptr;
    OC_CHECK(ensure_tables(&T));
    const int nl = s.n_nodes_l;
    schur_mass_kernel<<<static_cast<unsigned>((nl + 255) / 256), 256, 0, runtime().stream>>>(
        nl, s.gather_ptr.ptr + 3 * static_cast<int64_t>(s.n_nodes), s.gather_idx.ptr, s.gp_records.ptr, T,
        s.mat.ptr, inv_p);
    OC_HIP_CHECK(hipGetLastError());
    return OC_NO_ERROR;
}

int mr_jacobian_buffers(EquationsSet &s, int precision)
{
    OC_CHECK(mr_prepare(s));
    const BasisTables *T = nullptr;
    OC_CHECK(ensure_tables(&T));
    const size_t kn = static_cast<size_t>(s.n_elements) * 89 * 89;
    if (precision == OC_FP64) {
        if (!s.kbuf64.ptr) OC_CHECK(s.kbuf64.alloc(kn));
        if (!s.values.ptr) OC_CHECK(s.values.alloc(s.nnz));
    } else {
        if (!s.kbuf32.ptr) OC_CHECK(s.kbuf32.alloc(kn));
        if (!s.values_sp.ptr) OC_CHECK(s.values_sp.alloc(s.nnz));
    }
    return OC_NO_ERROR;
}

// Element-matrix phase alone (the autotuner times it per launch shape).
int launch_mr_element_matrices(EquationsSet &s, int precision, int blocks_per_cu)
{
    const BasisTables *T = nullptr;
    OC_CHECK(ensure_tables(&T));
    Runtime &rt = runtime();
    // default: one resident block of twelve waves per CU
    const int bpc = blocks_per_cu > 0 ? blocks_per_cu : 1;
    const unsigned blocks = static_cast<unsigned>(std::min(s.n_elements, rt.num_cus * bpc));
    if (precision == OC_FP64) {
        KernelTimer timer("mr_element_matrix_fp64");
        mr_element_matrix_f64_kernel<<<blocks, kElementThreads, 0, rt.stream>>>(s.n_elements, s.gp_records.ptr, T, s.kbuf64.ptr);
    } else {
        KernelTimer timer("mr_element_matrix_fp32");
        mr_element_matrix_f32_kernel<<<blocks, kElementThreads, 0, rt.stream>>>(s.n_elements, s.gp_records.ptr, T,
                                                                               s.kbuf32.ptr);
    }
    OC_HIP_CHECK(hipGetLastError());
    return OC_NO_ERROR;
}

int launch_mr_row_gather(EquationsSet &s, int precision, int chunk)
{
    if (precision == OC_FP64) {
        KernelTimer timer("csr_row_gather_fp64");
        return launch_row_gather<double>(s, s.kbuf64.ptr, s.values.ptr, chunk);
    }
    KernelTimer timer("csr_row_gather_fp32");
    return launch_row_gather<float>(s, s.kbuf32.ptr, s.values_sp.ptr, chunk);
}

// Forward-difference Jacobian: element residuals at x, then one launch over
// all (element, column) pairs, then the same ordered CSR row gather.
int launch_mr_jacobian_fd(EquationsSet &s)
{
    OC_CHECK(mr_jacobian_buffers(s, OC_FP64));
    const BasisTables *T = nullptr;
    OC_CHECK(ensure_tables(&T));
    Runtime &rt = runtime();
    // delta = (1 + ||x||_2) 1e-7 over the whole dependent vector (:3086-3087)
    std::vector<double> x(s.n_rows);
    OC_HIP_CHECK(hipMemcpyAsync(x.data(), s.dofs.ptr, sizeof(double) * x.size(), hipMemcpyDeviceToHost, rt.stream));
    OC_HIP_CHECK(hipStreamSynchronize(rt.stream));
    double ss = 0.0;
    for (double v : x) ss += v * v;
    const double delta = (1.0 + std::sqrt(ss)) * 1e-7;
    const unsigned blocks = static_cast<unsigned>((s.n_elements + kGaussElemsPerBlock - 1) / kGaussElemsPerBlock);
    OC_CHECK(launch_residual_elements<false>(s, blocks, s.dofs.ptr, T, s.relem.ptr, 0.0, nullptr));
    const int64_t nv = static_cast<int64_t>(s.n_elements) * 89;
    if (nv >= INT32_MAX) return set_error(OC_ERR_UNSUPPORTED, "too many elements for the finite-difference launch");
    {
        KernelTimer timer("mr_fd_columns");
        const unsigned fb = static_cast<unsigned>((nv + kGaussElemsPerBlock - 1) / kGaussElemsPerBlock);
        OC_CHECK(launch_residual_elements<true>(s, fb, s.dofs.ptr, T, s.relem.ptr, delta, s.kbuf64.ptr));
    }
    return launch_mr_row_gather(s, OC_FP64, s.tuned[OC_FP64].gather_chunk);
}

int launch_mr_jacobian(EquationsSet &s, int precision)
{
    if (s.subtype == OC_INCOMPRESSIBLE_MOONEY_RIVLIN_SUBTYPE) {
        // the reference evaluates this subtype's Jacobian by forward differences
        if (precision != OC_FP64)
            return set_error(OC_ERR_UNSUPPORTED, "the incompressible Mooney-Rivlin subtype has FP64 "
                                                 "forward-difference Jacobians only");
        return launch_mr_jacobian_fd(s);
    }
    OC_CHECK(mr_jacobian_buffers(s, precision));
    OC_CHECK(launch_mr_gauss(s));
    OC_CHECK(launch_mr_element_matrices(s, precision, s.tuned[precision].element_blocks_per_cu));
    return launch_mr_row_gather(s, precision, s.tuned[precision].gather_chunk);
}

// ---------------------------------------------------------------------------
// Allocation-free residual evaluation (oc_residual_evaluate_noalloc): the
// element residuals go through `scratch`, a fixed array in device memory (one
// copy per GPU, held until the process ends) instead of the set's buffer.
// Host code never passes the symbol itself to a kernel (on the host it only
// stands for the device variable): it uses the address hipGetSymbolAddress
// returned for the device, kept in g_scratch_ptr.  Every element residual
// entry is written before the DOF gather reads it, so nothing is cleared
// between calls; calls that overlap on one GPU share the array and race.
constexpr int kMaxDevices = 64;
static __device__ __align__(256) double scratch[static_cast<size_t>(OC_NOALLOC_MAX_ELEMENTS) * 89];
static double *g_scratch_ptr[kMaxDevices] = {};

int noalloc_scratch_init(int device)
{
    if (device < 0 || device >= kMaxDevices)
        return set_error(OC_ERR_UNSUPPORTED, "device %d beyond the %d devices of the scratch table", device, kMaxDevices);
    if (g_scratch_ptr[device]) return OC_NO_ERROR;
    void *p = nullptr;
    OC_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return set_error(OC_ERR_HIP, "hipGetSymbolAddress returned no address for the scratch array");
    g_scratch_ptr[device] = static_cast<double *>(p);
    return OC_NO_ERROR;
}

// (c10, c01) of every quadratic node from its elements (all elements around
// a node belong to one mesh, so every writer of an entry writes the same pair)
__global__ void __launch_bounds__(256) node_materials_kernel(int n_elements, const int *__restrict__ conn_q,
                                                            const double *__restrict__ mat,
                                                            double *__restrict__ node_mat)
{
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n_elements * 27; t += gridDim.x * blockDim.x) {
        const int e = t / 27, node = conn_q[t];
        node_mat[2 * node] = mat[2 * e];
        node_mat[2 * node + 1] = mat[2 * e + 1];
    }
}

int mr_node_materials(EquationsSet &s)
{
    if (!s.node_mat.ptr) OC_CHECK(s.node_mat.alloc(static_cast<size_t>(2) * s.n_nodes));
    const int64_t n = static_cast<int64_t>(s.n_elements) * 27;
    const unsigned blocks = static_cast<unsigned>(std::min<int64_t>((n + 255) / 256, 8192));
    node_materials_kernel<<<blocks, 256, 0, runtime().stream>>>(s.n_elements, s.conn.ptr, s.mat.ptr, s.node_mat.ptr);
    OC_HIP_CHECK(hipGetLastError());
    return OC_NO_ERROR;
}

}  // namespace oc

using namespace oc;

extern "C" int oc_residual_evaluate_noalloc(oc_equations_set h, const double *dofs_device, double *residual_device)
{
    OC_CHECK(require_runtime());
    if (!h) return set_error(OC_ERR_INVALID_HANDLE, "equations set handle is NULL");
    if (!dofs_device || !residual_device)
        return set_error(OC_ERR_INVALID_ARGUMENT, "oc_residual_evaluate_noalloc: NULL device array");
    EquationsSet &s = h->s;
    if (s.cls != OC_EQUATIONS_SET_MOONEY_RIVLIN)
        return set_error(OC_ERR_INVALID_ARGUMENT, "oc_residual_evaluate_noalloc is defined for Mooney-Rivlin sets");
    if (s.n_elements > OC_NOALLOC_MAX_ELEMENTS)
        return set_error(OC_ERR_UNSUPPORTED,
                         "%d elements exceed the %d elements of the allocation-free residual's scratch; use "
                         "oc_equations_set_residual_evaluate",
                         s.n_elements, OC_NOALLOC_MAX_ELEMENTS);
    Runtime &rt = runtime();
    const BasisTables *T = device_basis_tables();
    double *scr = (rt.device >= 0 && rt.device < kMaxDevices) ? g_scratch_ptr[rt.device] : nullptr;
    if (!T || !scr || !s.gather_ptr.ptr)
        return set_error(OC_ERR_NOT_INITIALISED, "device tables, scratch or the set's gather lists are not set up");
    const unsigned blocks = static_cast<unsigned>((s.n_elements + kGaussElemsPerBlock - 1) / kGaussElemsPerBlock);
    OC_CHECK(launch_residual_elements<false>(s, blocks, dofs_device, T, scr, 0.0, nullptr));
    dof_gather_kernel<<<static_cast<unsigned>((s.n_rows + 255) / 256), 256, 0, rt.stream>>>(
        s.n_rows, s.gather_ptr.ptr, s.gather_idx.ptr, scr, residual_device);
    OC_HIP_CHECK(hipGetLastError());
    return OC_NO_ERROR;
}
