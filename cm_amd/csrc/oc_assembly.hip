// oc_assembly.hip -- basis tables, fill kernel and the gfx950 Laplace
// linear-matrix assembly: element matrices, then a deterministic write-once
// CSR row gather in ascending element order.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "oc_fe_device.h"
#include "oc_internal.h"

namespace oc {

// ---------------------------------------------------------------------------
// Basis tables (host).  GAUSS_LEGENDRE closed forms on [0,1]
// (basis_routines.f90:5826-5875); Lagrange 1-D polynomials (:7015-7137);
// tensor products with xi1 fastest for both Gauss points (:2863-2890) and
// basis nodes (:1594-1630).
static double lagrange_1d(int order, int node, bool deriv, double xi)
{
    if (order == 1) {
        if (!deriv) return node == 0 ? 1.0 - xi : xi;
        return node == 0 ? -1.0 : 1.0;
    }
    if (!deriv) {
        if (node == 0) return 1.0 - 3.0 * xi + 2.0 * xi * xi;
        if (node == 1) return 4.0 * xi * (1.0 - xi);
        return xi * (xi + xi - 1.0);
    }
    if (node == 0) return 4.0 * xi - 3.0;
    if (node == 1) return 4.0 - 8.0 * xi;
    return 4.0 * xi - 1.0;
}

static void gauss_1d(int n, double *x, double *w)
{
    if (n == 2) {
        const double s = 1.0 / std::sqrt(3.0);
        x[0] = (-s + 1.0) / 2.0;
        x[1] = (s + 1.0) / 2.0;
        w[0] = w[1] = 0.5;
    } else {  // n == 3
        const double s = std::sqrt(0.6);
        x[0] = (-s + 1.0) / 2.0;
        x[1] = 0.5;
        x[2] = (s + 1.0) / 2.0;
        w[0] = 2.5 / 9.0;
        w[1] = 4.0 / 9.0;
        w[2] = 2.5 / 9.0;
    }
}

static void tabulate(int order, int ng1, double *w, double *fns)
{
    double gx[3], gw[3];
    gauss_1d(ng1, gx, gw);
    const int nx = order + 1, ns = nx * nx * nx;
    int g = 0;
    for (int k = 0; k < ng1; ++k)
        for (int j = 0; j < ng1; ++j)
            for (int i = 0; i < ng1; ++i, ++g) {
                const double xi[3] = {gx[i], gx[j], gx[k]};
                w[g] = gw[i] * gw[j] * gw[k];
                int s = 0;
                for (int n3 = 0; n3 < nx; ++n3)
                    for (int n2 = 0; n2 < nx; ++n2)
                        for (int n1 = 0; n1 < nx; ++n1, ++s) {
                            const int pos[3] = {n1, n2, n3};
                            for (int nu = 0; nu < 4; ++nu) {
                                double v = 1.0;
                                for (int d = 0; d < 3; ++d) v *= lagrange_1d(order, pos[d], nu == d + 1, xi[d]);
                                fns[(g * ns + s) * 4 + nu] = v;
                            }
                        }
            }
}

void build_basis_tables(BasisTables &t)
{
    double wtmp[27];
    tabulate(2, 3, t.w27, t.quad27);
    tabulate(1, 3, wtmp, t.lin27);
    tabulate(1, 2, t.w8, t.lin8);
}

static BasisTables *g_device_tables = nullptr;
static int g_tables_device = -1;

int ensure_tables(const BasisTables **out)
{
    Runtime &rt = runtime();
    if (g_device_tables == nullptr || g_tables_device != rt.device) {
        static BasisTables host;
        build_basis_tables(host);
        void *p = nullptr;
        OC_HIP_CHECK(hipMalloc(&p, sizeof(BasisTables)));
        OC_HIP_CHECK(hipMemcpy(p, &host, sizeof(BasisTables), hipMemcpyHostToDevice));
        g_device_tables = static_cast<BasisTables *>(p);
        g_tables_device = rt.device;
    }
    *out = g_device_tables;
    return OC_NO_ERROR;
}

const BasisTables *device_basis_tables() { return g_device_tables; }

// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256) fill_kernel(T *__restrict__ p, int64_t n, T v)
{
    const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

template <typename T>
int fill(T *p, int64_t n, T v)
{
    if (n <= 0) return OC_NO_ERROR;
    Runtime &rt = runtime();
    const int64_t blocks = std::min<int64_t>((n + 255) / 256, static_cast<int64_t>(rt.num_cus) * 16);
    KernelTimer timer("fill");
    fill_kernel<T><<<static_cast<unsigned>(blocks), 256, 0, rt.stream>>>(p, n, v);
    OC_HIP_CHECK(hipGetLastError());
    return OC_NO_ERROR;
}
template int fill<double>(double *, int64_t, double);
template int fill<float>(float *, int64_t, float);

// ---------------------------------------------------------------------------
// Laplace, standard subtype (Laplace_equations_routines.f90:474-571):
// K_e(ms,ns) += sum_{mi,ni} dphi_ms/dxi_mi GU(mi,ni) dphi_ns/dxi_ni * J w.
// Two phases, as the Jacobian: laplace_element_kernel writes every element
// matrix to a buffer (one thread per element); laplace_row_gather_kernel
// gives each CSR row eight lanes, which add the element rows touching it in
// ascending element order (the reference's element-loop order) into an LDS
// copy of its block's rows, and the block writes its contiguous CSR segment
// once: no zero fill, no read-modify-write, no colours.
__global__ void __launch_bounds__(256)
laplace_slot_offsets_kernel(int n_elements, const int *__restrict__ conn, const int64_t *__restrict__ row_ptr,
                            const int *__restrict__ col_idx, uint8_t *__restrict__ offs, int *__restrict__ n_bad)
{
    const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (gid >= static_cast<int64_t>(n_elements) * 8) return;
    const int64_t e = gid / 8;
    const int row = conn[gid];
    const int64_t base = row_ptr[row];
    for (int j = 0; j < 8; ++j) {
        const int64_t slot = csr_slot(row_ptr, col_idx, row, conn[e * 8 + j]);
        if (slot < 0 || slot - base > 255) {
            atomicAdd(n_bad, 1);
            offs[gid * 8 + j] = 0;
        } else {
            offs[gid * 8 + j] = static_cast<uint8_t>(slot - base);
        }
    }
}

// The 36 upper-triangle entries K[ms*(15-ms)/2 + ns] (ms <= ns) of one
// trilinear element matrix from its node coordinates x[c][n]
// (Laplace_equations_routines.f90:474-571).  Restated for the tensor-product
// structure of the trilinear basis at the 2x2x2 Gauss points:
//   * dX/dxi by sum factorisation: along xi_d a trilinear map's derivative is
//     the bilinear interpolant, in the other two coordinates, of its four edge
//     differences along d, so 36 values serve all eight Gauss points;
//   * the basis derivatives are products of the 1-D factors 1 - xi, xi at
//     the Gauss abscissae, compile-time constants;
//   * GU J w = adj(GL) w / sqrt(det GL) =: A, since J = sqrt(det GL) and
//     GU = adj(GL) / det GL (COORDINATE_METRICS_CALCULATE and
//     INVERT_FULL_DP, whose zero-tolerance rule it keeps);
//   * K by sum factorisation as well: the part of A_ij is a sum over the Gauss
//     points of A_ij times one 1-D factor (or a product of two) per direction,
//     so each A_ij is contracted one direction at a time into 9 (i = j) or 12
//     values, and an entry of K adds nine of those with signs;
//   * the basis derivatives sum to zero at every point, so each row of K_e
//     sums to zero: the 28 entries among local nodes 0-6 are formed and the
//     entries of node 7 follow as negated row sums.
// 920 FP64 operations an element against 1,850 with K summed over the Gauss
// points entry by entry.  Everything unrolls, so every index is a constant.
__device__ __forceinline__ constexpr int lap_upper(int ms, int ns) { return ms * (15 - ms) / 2 + ns; }

// The 1-D factors 1 - xi and xi at the two Gauss abscissae (1 -+ 1/sqrt 3) / 2
// are kLapP = (3 + sqrt 3) / 6 and 1 - kLapP, kLapR their ratio 2 - sqrt 3.
// Every sum below leaves one kLapP per factor out, so that a weighted sum of
// two values is one fma: a slope of x lacks kLapP^2, so A = adj(GL) w /
// sqrt(det GL) lacks kLapP^2 as well, and a contracted A lacks one kLapP for
// each of its four factors.  The weight w = 1/8 takes the six of them.
constexpr double kLapP = 0x1.93cd3a2c8198ep-1, kLapR = 0x1.126145e9ecd56p-2;
constexpr double kLapP2 = kLapP * kLapP, kLapP6 = kLapP2 * kLapP2 * kLapP2;

// sums over the two abscissae of one direction, from the values at each:
// against the factor of node 0 and 1, or against the products of two nodes'
// factors (0: nodes 0 0, 1: nodes 0 1, 2: nodes 1 1)
__device__ __forceinline__ void lap_single(double x0, double x1, double (&o)[2])
{
    o[0] = fma(kLapR, x1, x0);
    o[1] = fma(kLapR, x0, x1);
}
__device__ __forceinline__ void lap_pair(double x0, double x1, double (&o)[3])
{
    o[0] = fma(kLapR * kLapR, x1, x0);
    o[1] = kLapR * (x0 + x1);
    o[2] = fma(kLapR * kLapR, x0, x1);
}

// ready() runs before the first store(index, value); every value is stored once
template <typename Ready, typename Store>
__device__ __forceinline__ void laplace_element_upper(const double (&x)[3][8], Ready ready, Store store)
{
    // every multiply-add is an explicit fma (contraction is off here), so the
    // rounding is the same wherever the function is compiled: the fused and
    // the two-pass assembly write bit-identical values
#pragma clang fp contract(off)
    // dX_c/dxi_d at abscissae (ga, gb) of the other two directions (ascending)
    auto edges = [&](int c, int d, double (&e)[2][2]) {
        const int sd = 1 << d, sa = d == 0 ? 2 : 1, sb = d == 2 ? 2 : 4;
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
            for (int na = 0; na < 2; ++na) e[nb][na] = x[c][sd + sa * na + sb * nb] - x[c][sa * na + sb * nb];
    };
    // the interpolant of a and b at abscissa g
    auto between = [](double a, double b, int g) { return g ? fma(kLapR, a, b) : fma(kLapR, b, a); };
    auto slope = [&](const double (&e)[2][2], int ga, int gb) {
        return between(between(e[0][0], e[0][1], ga), between(e[1][0], e[1][1], ga), gb);
    };
    double Dz[3][2][2];  // dX_c/dxi_3 at [g2][g1]: the same in both Gauss layers
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        double e[2][2];
        edges(c, 2, e);
#pragma unroll
        for (int g2 = 0; g2 < 2; ++g2)
#pragma unroll
            for (int g1 = 0; g1 < 2; ++g1) Dz[c][g2][g1] = slope(e, g1, g2);
    }
    // the two Gauss layers g3, contracted over g1 and g2: A_00 (y pair), A_11
    // (x pair), A_22 (x pair, y pair), A_01 (x node, y node), A_02 (x node, y
    // pair), A_12 (x pair, y node).  The scheduling barriers keep one row of
    // Gauss points at a time in registers.
    double t00[2][3], t11[2][3], t22[2][3][3], t01[2][2][2], t02[2][2][3], t12[2][3][2];
#pragma unroll
    for (int g3 = 0; g3 < 2; ++g3) {
        double Dy[3][2];  // dX_c/dxi_2 at g1
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            double e[2][2];
            edges(c, 1, e);
            Dy[c][0] = slope(e, 0, g3);
            Dy[c][1] = slope(e, 1, g3);
        }
        double s00[2], s11[2][2], s22[2][3], s01[2][2], s02[2][2], s12[2][3];  // contracted over g1, at g2
#pragma unroll
        for (int g2 = 0; g2 < 2; ++g2) {
            double Dx[3];  // dX_c/dxi_1
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                double e[2][2];
                edges(c, 0, e);
                Dx[c] = slope(e, g2, g3);
            }
            double A[6][2];  // 00 11 22 01 02 12 at g1
#pragma unroll
            for (int g1 = 0; g1 < 2; ++g1) {
                double dx[9];  // dx[c + 3 mi] = dX_c/dxi_mi
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    dx[c] = Dx[c];
                    dx[c + 3] = Dy[c][g1];
                    dx[c + 6] = Dz[c][g2][g1];
                }
                double gl[6];  // GL = dX^T dX: 00 11 22 01 02 12
                auto dot3 = [](double a0, double b0, double a1, double b1, double a2, double b2) {
                    return fma(a2, b2, fma(a1, b1, a0 * b0));
                };
                gl[0] = dot3(dx[0], dx[0], dx[1], dx[1], dx[2], dx[2]);
                gl[1] = dot3(dx[3], dx[3], dx[4], dx[4], dx[5], dx[5]);
                gl[2] = dot3(dx[6], dx[6], dx[7], dx[7], dx[8], dx[8]);
                gl[3] = dot3(dx[0], dx[3], dx[1], dx[4], dx[2], dx[5]);
                gl[4] = dot3(dx[0], dx[6], dx[1], dx[7], dx[2], dx[8]);
                gl[5] = dot3(dx[3], dx[6], dx[4], dx[7], dx[5], dx[8]);
                auto diff2 = [](double a, double b, double c, double d) { return fma(a, b, -(c * d)); };  // ab - cd
                const double c00 = diff2(gl[1], gl[2], gl[5], gl[5]), c11 = diff2(gl[0], gl[2], gl[4], gl[4]);
                const double c22 = diff2(gl[0], gl[1], gl[3], gl[3]), c01 = diff2(gl[4], gl[5], gl[3], gl[2]);
                const double c02 = diff2(gl[3], gl[5], gl[4], gl[1]), c12 = diff2(gl[3], gl[4], gl[0], gl[5]);
                const double det = dot3(gl[0], c00, gl[3], c01, gl[4], c02);  // det GL = det(dX)^2
                // weight 1/8 of the 2x2x2 rule on [0, 1]^3; the root is opaque
                // so that it stays out of a branch, which would keep the Gauss
                // points from overlapping
                double rs = rsqrt(fabs(det));
                asm("" : "+v"(rs));
                const double sc = fabs(det) > 5.0 * 2.220446049250313e-16 / (kLapP6 * kLapP6) ? copysign(0.125 * kLapP6 * rs, det) : 0.0;
                A[0][g1] = c00 * sc;
                A[1][g1] = c11 * sc;
                A[2][g1] = c22 * sc;
                A[3][g1] = c01 * sc;
                A[4][g1] = c02 * sc;
                A[5][g1] = c12 * sc;
            }
            s00[g2] = A[0][0] + A[0][1];
            s11[g2][0] = A[1][0];
            s11[g2][1] = A[1][1];
            lap_pair(A[2][0], A[2][1], s22[g2]);
            lap_single(A[3][0], A[3][1], s01[g2]);
            lap_single(A[4][0], A[4][1], s02[g2]);
            lap_pair(A[5][0], A[5][1], s12[g2]);
            __builtin_amdgcn_sched_barrier(0);
        }
        lap_pair(s00[0], s00[1], t00[g3]);
        lap_pair(s11[0][0] + s11[1][0], s11[0][1] + s11[1][1], t11[g3]);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            lap_pair(s22[0][k], s22[1][k], t22[g3][k]);
            lap_single(s12[0][k], s12[1][k], t12[g3][k]);
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            lap_single(s01[0][k], s01[1][k], t01[g3][k]);
            lap_pair(s02[0][k], s02[1][k], t02[g3][k]);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // over g3: z pairs for 00, 11 and 01, z nodes for 02 and 12
    double T00[3][3], T11[3][3], T22[3][3], T01[2][2][3], T02[2][3][2], T12[3][2][2];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        lap_pair(t00[0][k], t00[1][k], T00[k]);
        lap_pair(t11[0][k], t11[1][k], T11[k]);
#pragma unroll
        for (int q = 0; q < 3; ++q) T22[k][q] = t22[0][k][q] + t22[1][k][q];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            lap_single(t02[0][q][k], t02[1][q][k], T02[q][k]);
            lap_single(t12[0][k][q], t12[1][k][q], T12[k][q]);
        }
    }
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int q = 0; q < 2; ++q) lap_pair(t01[0][k][q], t01[1][k][q], T01[k][q]);
    ready();
    double row[7] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    auto sgn = [](int a, int b, double t) { return a == b ? t : -t; };
#pragma unroll
    for (int ms = 0; ms < 7; ++ms)
#pragma unroll
        for (int ns = ms; ns < 7; ++ns) {
            const int m0 = ms & 1, m1 = (ms >> 1) & 1, m2 = ms >> 2, n0 = ns & 1, n1 = (ns >> 1) & 1, n2 = ns >> 2;
            const int p0 = m0 + n0, p1 = m1 + n1, p2 = m2 + n2;  // the nodes' pair per direction
            double k = sgn(m0, n0, T00[p1][p2]) + sgn(m1, n1, T11[p0][p2]) + sgn(m2, n2, T22[p0][p1]);
            k = k + (sgn(m0, n1, T01[n0][m1][p2]) + sgn(n0, m1, T01[m0][n1][p2]));
            k = k + (sgn(m0, n2, T02[n0][p1][m2]) + sgn(n0, m2, T02[m0][p1][n2]));
            k = k + (sgn(m1, n2, T12[p0][n1][m2]) + sgn(n1, m2, T12[p0][m1][n2]));
            store(lap_upper(ms, ns), k);
            row[ms] += k;
            if (ns != ms) row[ns] += k;
        }
    double k77 = 0.0;
#pragma unroll
    for (int ms = 0; ms < 7; ++ms) {
        store(lap_upper(ms, 7), -row[ms]);
        k77 += row[ms];
    }
    store(lap_upper(7, 7), k77);
}

// the coordinates of one node of an (x, y, z, -) list: two 16-byte loads of one
// 64-byte piece of a cache line
__device__ __forceinline__ void load_node(const double *__restrict__ xyz, int node, int n, double (&x)[3][8])
{
    const double2 a = *reinterpret_cast<const double2 *>(xyz + 4 * static_cast<int64_t>(node));
    x[0][n] = a.x;
    x[1][n] = a.y;
    x[2][n] = xyz[4 * static_cast<int64_t>(node) + 2];
}

__global__ void __launch_bounds__(256) node_major_kernel(int n, const double *__restrict__ coords,
                                                        double *__restrict__ xyz)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double2 *o = reinterpret_cast<double2 *>(xyz + 4 * static_cast<int64_t>(i));
    o[0] = make_double2(coords[i], coords[static_cast<int64_t>(n) + i]);
    o[1] = make_double2(coords[2 * static_cast<int64_t>(n) + i], 0.0);
}

// One thread per element; each row of K_e goes to its place in the
// row-gather order, so the gather reads every CSR row's contributions
// contiguously.  The rows' places are scattered, and a row is one 64-byte
// request only if its stores are issued together: the block turns its element
// matrices through LDS so that four lanes write one row.  152,000 elements with
// their nodes in no order: 41 us with K in registers and a row per thread, 34 us
// now; what is left is the latency of its two rounds of wavefronts.
constexpr int kLapThreads = 64;
constexpr int kLapStage = kLapThreads + 1;  // padded against bank conflicts

__global__ void __launch_bounds__(kLapThreads)
laplace_element_kernel(int n_elements, const int *__restrict__ conn, const double *__restrict__ xyz,
                       const int *__restrict__ gpos, double *__restrict__ kbuf)
{
    __shared__ double s_K[36 * kLapStage];  // upper triangles, [entry][element]
    const int t = threadIdx.x, e0 = blockIdx.x * kLapThreads;
    const int e = min(e0 + t, n_elements - 1);  // the last block's spare threads repeat its last element
    const int4 lo = reinterpret_cast<const int4 *>(conn)[2 * static_cast<int64_t>(e)];
    const int4 hi = reinterpret_cast<const int4 *>(conn)[2 * static_cast<int64_t>(e) + 1];
    const int node[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    double x[3][8];
#pragma unroll
    for (int n = 0; n < 8; ++n) load_node(xyz, node[n], n, x);
    laplace_element_upper(x, [] {}, [&](int i, double v) { s_K[i * kLapStage + t] = v; });
    __syncthreads();
    // lane t stores columns 2 (t & 3) and the next of element row 16 q + t / 4:
    // row ms = (t / 4) & 7 of every second element
    const int ms = (t >> 2) & 7, j = 2 * (t & 3), le0 = t >> 5;
    const int k0 = ms <= j ? lap_upper(ms, j) : lap_upper(j, ms);
    const int k1 = ms <= j + 1 ? lap_upper(ms, j + 1) : lap_upper(j + 1, ms);
    const int n_here = min(kLapThreads, n_elements - e0);
#pragma unroll 8
    for (int le = le0; le < n_here; le += 2) {
        const int pos = gpos[static_cast<int64_t>(e0 + le) * 8 + ms];
        *reinterpret_cast<double2 *>(kbuf + static_cast<int64_t>(pos) * 8 + j) =
            make_double2(s_K[k0 * kLapStage + le], s_K[k1 * kLapStage + le]);
    }
}

// slot offsets permuted into the row-gather order
__global__ void __launch_bounds__(256) permute_offsets_kernel(int64_t n, const int *__restrict__ idx,
                                                             const uint64_t *__restrict__ offs,
                                                             uint64_t *__restrict__ out)
{
    for (int64_t p = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; p < n;
         p += static_cast<int64_t>(gridDim.x) * blockDim.x)
        out[p] = offs[idx[p]];
}

// Eight lanes per CSR row (32 rows per block): lane j adds column j of each
// of the row's element rows, in ascending element order, into the block's
// LDS copy of its CSR segment; a chunk's global loads (eight element rows)
// are issued before its LDS adds.  The block then writes the segment once.
constexpr int kLapGatherRows = 32;

__global__ void __launch_bounds__(8 * kLapGatherRows)
laplace_row_gather_kernel(int n_rows, const int64_t *__restrict__ row_ptr, const int *__restrict__ gptr,
                          const double *__restrict__ kbuf, const uint8_t *__restrict__ offs,
                          double *__restrict__ values, double *__restrict__ rhs)
{
    extern __shared__ unsigned char s_raw[];
    double *s_seg = reinterpret_cast<double *>(s_raw);
    const int t = threadIdx.x, j = t & 7;
    const int r0 = blockIdx.x * kLapGatherRows, r = r0 + (t >> 3);
    const int r_end = min(r0 + kLapGatherRows, n_rows);
    const int64_t base = row_ptr[r0];
    const int seg = static_cast<int>(row_ptr[r_end] - base);
    for (int k = t; k < seg; k += 8 * kLapGatherRows) s_seg[k] = 0.0;
    __syncthreads();
    if (r < n_rows) {
        if (j == 0) rhs[r] = 0.0;  // the RHS element vector is 0 (:542)
        double *row = s_seg + (row_ptr[r] - base);
        const int c_end = gptr[r + 1];
        for (int c0 = gptr[r]; c0 < c_end; c0 += 8) {
            double v[8];
            int o[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                if (c0 + c < c_end) {
                    const int64_t p = static_cast<int64_t>(c0 + c) * 8 + j;
                    v[c] = kbuf[p];
                    o[c] = offs[p];
                }
            }
#pragma unroll
            for (int c = 0; c < 8; ++c)
                if (c0 + c < c_end) row[o[c]] += v[c];
        }
    }
    __syncthreads();
    for (int k = t; k < seg; k += 8 * kLapGatherRows) values[base + k] = s_seg[k];
}

// Small meshes in one launch: eight lanes per CSR row, eight rows per
// wavefront.  Lane j forms the matrix of the row's j-th element (of each eight
// in ascending order) in LDS, then adds column j of all eight in that order, so
// every element matrix is formed by each of its eight rows.  While the mesh
// leaves most of the GPU idle that costs nothing, and the element buffer's
// second launch and round trip are saved.
__global__ void __launch_bounds__(64)
laplace_small_kernel(int n_rows, const int64_t *__restrict__ row_ptr, const int *__restrict__ gptr,
                     const int *__restrict__ erow, const int *__restrict__ conn, const double *__restrict__ xyz,
                     const uint8_t *__restrict__ offs, double *__restrict__ values,
                     double *__restrict__ rhs)
{
    extern __shared__ unsigned char s_raw[];
    __shared__ double s_K[36 * kLapStage];  // upper triangles, [entry][lane]
    double *s_seg = reinterpret_cast<double *>(s_raw);
    const int t = threadIdx.x, j = t & 7, g0 = t & ~7;
    const int r0 = blockIdx.x * 8, r = r0 + (t >> 3), r_end = min(r0 + 8, n_rows);
    const int64_t base = row_ptr[r0];
    const int seg = static_cast<int>(row_ptr[r_end] - base);
    for (int k = t; k < seg; k += 64) s_seg[k] = 0.0;
    const bool in = r < n_rows;
    if (in && j == 0) rhs[r] = 0.0;  // the RHS element vector is 0 (:542)
    double *row = s_seg + (in ? row_ptr[r] - base : 0);
    const int c_end = in ? gptr[r + 1] : 0;
    for (int c0 = in ? gptr[r] : 0; __any(c0 < c_end); c0 += 8) {
        int ms = 0, o[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) o[c] = c0 + c < c_end ? offs[static_cast<int64_t>(c0 + c) * 8 + j] : 0;
        if (c0 + j < c_end) {
            const int er = erow[c0 + j];  // element * 8 + the row's local node
            ms = er & 7;
            double x[3][8];
#pragma unroll
            for (int n = 0; n < 8; ++n) load_node(xyz, conn[static_cast<int64_t>(er & ~7) + n], n, x);
            laplace_element_upper(x, [] {}, [&](int i, double v) { s_K[i * kLapStage + t] = v; });
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int m = __shfl(ms, g0 + c);
            const double v = s_K[(m <= j ? lap_upper(m, j) : lap_upper(j, m)) * kLapStage + g0 + c];
            if (c0 + c < c_end) row[o[c]] += v;
        }
        __syncthreads();
    }
    for (int k = t; k < seg; k += 64) values[base + k] = s_seg[k];
}

// ---------------------------------------------------------------------------
// Fused Laplace assembly of a structured hexahedral grid (nx x ny x nz
// elements, nodes and elements numbered x fastest, local nodes xi1 fastest):
// no element-matrix buffer.  A block owns the CSR rows of a kLapTX x kLapTY
// column of nodes over `seg` element layers and walks up the layers.  Per
// layer, each thread computes one element matrix of the column's element
// footprint (one element wider on the low x and y sides) into LDS; each node
// thread then
//   * finishes the row of its node in the layer's bottom plane: the partial
//     sums from the layer below (kept in its registers) plus the four
//     elements above the plane, and writes it to its CSR segment once;
//   * starts the row of its node in the top plane with the layer's four
//     elements below that plane.
// A row's entries thus add the element matrices that hold them in ascending
// element order from 0, as the two-pass row gather does, so values are
// bit-identical to it.  Blocks share only recomputed footprint elements
// (x, y halo and the layer below a segment), never output.
constexpr int kLapTX = 15, kLapTY = 7;
constexpr int kLapFX = kLapTX + 1, kLapFusedThreads = (kLapTX + 1) * (kLapTY + 1);  // 128

typedef double Entries2 __attribute__((ext_vector_type(2), aligned(8)));  // 16-byte store at an 8-byte address

__global__ void __launch_bounds__(kLapFusedThreads)
laplace_fused_kernel(int nx, int ny, int nz, int seg, const double *__restrict__ coords, int n_nodes,
                     const int64_t *__restrict__ row_ptr, double *__restrict__ values, double *__restrict__ rhs)
{
    // the layer's element matrices (upper triangles, [entry][element]), then the finished rows (27 per node)
    __shared__ double s_buf[36 * kLapFusedThreads];
    double(*sK)[kLapFusedThreads] = reinterpret_cast<double(*)[kLapFusedThreads]>(s_buf);
    const int t = threadIdx.x;
    const int tiles_x = (nx + kLapTX) / kLapTX, tiles_y = (ny + kLapTY) / kLapTY;  // nx + 1 nodes
    int b = static_cast<int>(blockIdx.x);
    const int i0 = (b % tiles_x) * kLapTX;
    b /= tiles_x;
    const int j0 = (b % tiles_y) * kLapTY;
    const int k0 = (b / tiles_y) * seg, k1 = min(nz, k0 + seg);
    const int NX = nx + 1;
    const int64_t NXY = static_cast<int64_t>(nx + 1) * (ny + 1);
    // this thread's footprint element and node column; an element outside the
    // grid is never read, so its thread repeats the nearest one inside
    const int ie = min(max(i0 - 1 + t % kLapFX, 0), nx - 1), je = min(max(j0 - 1 + t / kLapFX, 0), ny - 1);
    const int ni = i0 + t % kLapTX, nj = j0 + t / kLapTX;
    const bool has_node = t < kLapTX * kLapTY && ni <= nx && nj <= ny;
    const int dxlo = ni > 0 ? -1 : 0, cx = (ni < nx ? 2 : 1) - dxlo;
    const int dylo = nj > 0 ? -1 : 0, cy = (nj < ny ? 2 : 1) - dylo;
    // partial row of the column's node in the next plane (slots dz = -1, 0):
    // the thread keeps its column over the layers, so it stays in registers
    double P[18];
#pragma unroll
    for (int q = 0; q < 18; ++q) P[q] = 0.0;
    // Rows of plane k: entry (dx, dy, dz) of a node's stencil is at
    // ((dz - dzlo) cy + dy - dylo) cx + dx - dxlo of its CSR row (columns
    // ascend), and neighbours in x have neighbouring rows, so the block turns
    // its rows through LDS and stores each of its kLapTY runs in x as one
    // contiguous piece, two entries a lane.  A thread storing its own row puts
    // each 8-byte entry into a request of its own, 216 bytes apart.
    constexpr int kRun = kLapTX * 27;
    auto write_rows = [&](int k, const double(&R)[27]) {
        const int dzlo = k > 0 ? -1 : 0, cz = (k < nz ? 2 : 1) - dzlo;
        __syncthreads();  // the element matrices are read
        if (has_node) {
            rhs[ni + NX * nj + NXY * k] = 0.0;  // the RHS element vector is 0 (:542)
            // of the run's nodes only the grid's first and last have cx = 2
            double *row = s_buf + t / kLapTX * kRun + cy * cz * (3 * (ni - i0) - (i0 == 0 && ni > 0 ? 1 : 0));
            if (cx * cy * cz == 27) {
#pragma unroll
                for (int q = 0; q < 27; ++q) row[q] = R[q];
            } else {
#pragma unroll
                for (int dz = -1; dz <= 1; ++dz)
#pragma unroll
                    for (int dy = -1; dy <= 1; ++dy)
#pragma unroll
                        for (int dx = -1; dx <= 1; ++dx) {
                            if (dz < dzlo || dz >= dzlo + cz || dy < dylo || dy >= dylo + cy || dx < dxlo ||
                                dx >= dxlo + cx)
                                continue;
                            row[((dz - dzlo) * cy + dy - dylo) * cx + dx - dxlo] = R[(dz + 1) * 9 + (dy + 1) * 3 + dx + 1];
                        }
            }
        }
        __syncthreads();
        const int last = min(i0 + kLapTX - 1, nx);  // the runs' last node
        const int slots = 3 * (last - i0 + 1) - (i0 == 0 ? 1 : 0) - (last == nx ? 1 : 0);
        for (int q = __builtin_amdgcn_readfirstlane(t >> 6); q < kLapTY && j0 + q <= ny; q += kLapFusedThreads / 64) {
            const int qj = j0 + q, len = cz * (1 + (qj > 0) + (qj < ny)) * slots;
            double *out = values + row_ptr[i0 + NX * qj + NXY * k];
            const double *src = s_buf + q * kRun;
#pragma unroll
            for (int u = 0; u < (kRun + 127) / 128; ++u) {
                const int idx = 128 * u + 2 * (t & 63);
                if (idx + 1 < len) *reinterpret_cast<Entries2 *>(out + idx) = Entries2{src[idx], src[idx + 1]};
                else if (idx < len) out[idx] = src[idx];
            }
        }
    };
    for (int k = max(k0 - 1, 0); k < k1; ++k) {
        double x[3][8];
        const int64_t base = ie + static_cast<int64_t>(NX) * je + NXY * k;
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            const int64_t node = base + (n & 1) + NX * ((n >> 1) & 1) + NXY * (n >> 2);
#pragma unroll
            for (int c = 0; c < 3; ++c) x[c][n] = coords[static_cast<int64_t>(c) * n_nodes + node];
        }
        // the barrier before the stores: the previous layer's rows are stored
        laplace_element_upper(x, [] { __syncthreads(); }, [&](int i, double v) { sK[i][t] = v; });
        __syncthreads();
        // the elements around the column in this layer, ascending:
        // (ni-1, nj-1), (ni, nj-1), (ni-1, nj), (ni, nj); local node a of the
        // column's node is (a1, a2) = (ni - ex, nj - ey) in the plane
        auto add = [&](double *acc, int top) {
#pragma unroll
            for (int a2 = 1; a2 >= 0; --a2)
#pragma unroll
                for (int a1 = 1; a1 >= 0; --a1) {
                    const int ex = ni - a1, ey = nj - a2;
                    if (!has_node || ex < 0 || ex >= nx || ey < 0 || ey >= ny) continue;
                    const int te = ex - i0 + 1 + kLapFX * (ey - j0 + 1);
                    const int ms = a1 + 2 * a2 + 4 * top;  // bottom or top face of the element
#pragma unroll
                    for (int ns = 0; ns < 8; ++ns) {
                        const int b1 = ns & 1, b2 = (ns >> 1) & 1, b3 = ns >> 2;
                        acc[(b3 + 1 - top) * 9 + (b2 - a2 + 1) * 3 + b1 - a1 + 1] +=
                            sK[ms <= ns ? lap_upper(ms, ns) : lap_upper(ns, ms)][te];
                    }
                }
        };
        double R[27];
#pragma unroll
        for (int q = 0; q < 18; ++q) R[q] = P[q];
#pragma unroll
        for (int q = 18; q < 27; ++q) R[q] = 0.0;
#pragma unroll
        for (int q = 0; q < 18; ++q) P[q] = 0.0;
        if (k >= k0) add(R, 0);  // plane k is this block's: its rows are finished
        add(P, 1);
        if (k >= k0) write_rows(k, R);
    }
    if (k1 == nz) {  // the top plane has no elements above it
        double R[27];
#pragma unroll
        for (int q = 0; q < 18; ++q) R[q] = P[q];
#pragma unroll
        for (int q = 18; q < 27; ++q) R[q] = 0.0;
        write_rows(nz, R);
    }
}

// Structured-grid check of a Laplace set: nodes and elements numbered x
// fastest on an nx x ny x nz grid with xi1-fastest local nodes, and the CSR
// rows the 27-point stencils with ascending columns.  Sets s.lap_grid, or
// leaves it zero (the two-pass assembly then serves the mesh).
void laplace_detect_grid(EquationsSet &s, const std::vector<int32_t> &conn)
{
    s.lap_grid[0] = s.lap_grid[1] = s.lap_grid[2] = 0;
    if (s.n_elements < 1 || conn.size() < 8 || conn[0] != 0 || conn[1] != 1) return;
    const int64_t NX = conn[2];
    if (NX < 2 || conn[4] % NX != 0) return;
    const int64_t NY = conn[4] / NX;
    if (NY < 2 || s.n_nodes % (NX * NY) != 0) return;
    const int64_t NZ = s.n_nodes / (NX * NY);
    const int64_t nx = NX - 1, ny = NY - 1, nz = NZ - 1;
    if (nz < 1 || nx * ny * nz != s.n_elements) return;
    for (int64_t e = 0; e < s.n_elements; ++e) {
        const int64_t ie = e % nx, je = (e / nx) % ny, ke = e / (nx * ny);
        const int64_t base = ie + NX * (je + NY * ke);
        for (int n = 0; n < 8; ++n)
            if (conn[e * 8 + n] != base + (n & 1) + NX * ((n >> 1) & 1) + NX * NY * (n >> 2)) return;
    }
    for (int64_t node = 0; node < s.n_nodes; ++node) {
        const int64_t i = node % NX, j = (node / NX) % NY, k = node / (NX * NY);
        int64_t p = s.h_row_ptr[node];
        for (int dz = -1; dz <= 1; ++dz)
            for (int dy = -1; dy <= 1; ++dy)
                for (int dx = -1; dx <= 1; ++dx) {
                    if (i + dx < 0 || i + dx > nx || j + dy < 0 || j + dy > ny || k + dz < 0 || k + dz > nz) continue;
                    if (p >= s.h_row_ptr[node + 1] || s.h_col_idx[p] != node + dx + NX * dy + NX * NY * dz) return;
                    ++p;
                }
        if (p != s.h_row_ptr[node + 1]) return;
    }
    s.lap_grid[0] = static_cast<int>(nx);
    s.lap_grid[1] = static_cast<int>(ny);
    s.lap_grid[2] = static_cast<int>(nz);
}

// Element layers per block of the fused launch: the most of 8, 4 and 2 whose
// blocks give every CU two and a half (each block forms one layer besides, so
// long segments repeat less, but a block walks its layers one after another).
// At 80^3 8 layers take 84 us, 4 94; at 64^3 83 and 54, at 56^3 62 and 48,
// and 2 layers 37.  0: even 2 leave too few blocks, and the two passes are as
// fast (48^3: 32 both; 40^3: 29 against 25).
static int64_t laplace_fused_blocks(const EquationsSet &s, int seg)
{
    const int nx = s.lap_grid[0], ny = s.lap_grid[1], nz = s.lap_grid[2];
    return static_cast<int64_t>((nx + kLapTX) / kLapTX) * ((ny + kLapTY) / kLapTY) * ((nz + seg - 1) / seg);
}

static int laplace_fused_layers(const EquationsSet &s)
{
    for (int seg = 8; seg >= 2; seg /= 2)
        if (2 * laplace_fused_blocks(s, seg) >= 5 * static_cast<int64_t>(runtime().num_cus)) return seg;
    return 0;
}

bool laplace_fused_serves(const EquationsSet &s)
{
    if (s.lap_grid[0] <= 0 || s.lap_fused == 0) return false;
    return s.lap_fused == 2 || laplace_fused_layers(s) > 0;
}

int launch_laplace_fused(EquationsSet &s)
{
    Runtime &rt = runtime();
    const int nx = s.lap_grid[0], ny = s.lap_grid[1], nz = s.lap_grid[2];
    if (nx < 1 || ny < 1 || nz < 1) return set_error(OC_ERR_UNSUPPORTED, "the Laplace set is not a structured grid");
    KernelTimer timer("laplace_fused");
    const int seg = std::max(laplace_fused_layers(s), 2);
    laplace_fused_kernel<<<static_cast<unsigned>(laplace_fused_blocks(s, seg)), kLapFusedThreads, 0, rt.stream>>>(
        nx, ny, nz, seg, s.coords.ptr, s.n_nodes, s.row_ptr.ptr, s.values.ptr, s.rhs.ptr);
    OC_HIP_CHECK(hipGetLastError());
    return OC_NO_ERROR;
}

// Meshes up to this many rows are assembled by laplace_small_kernel: 6.4 us
// against 8.6 for the two launches at 810 rows, 9.8 against 10.9 at 9,702; from
// 16,250 rows on (15.2 against 12.7) its eightfold element work no longer fits
// into idle compute units.
constexpr int kLapSmallRows = 12000;

static int laplace_prepare(EquationsSet &s)
{
    if (s.slot_offsets8.ptr) return OC_NO_ERROR;
    OC_CHECK(s.slot_offsets8.alloc(static_cast<size_t>(s.n_elements) * 64));
    DevBuf<int> bad;
    OC_CHECK(bad.alloc(1));
    Runtime &rt = runtime();
    OC_HIP_CHECK(hipMemsetAsync(bad.ptr, 0, sizeof(int), rt.stream));
    const int64_t nthreads = static_cast<int64_t>(s.n_elements) * 8;
    laplace_slot_offsets_kernel<<<static_cast<unsigned>((nthreads + 255) / 256), 256, 0, rt.stream>>>(
        s.n_elements, s.conn.ptr, s.row_ptr.ptr, s.col_idx.ptr, s.slot_offsets8.ptr, bad.ptr);
    OC_HIP_CHECK(hipGetLastError());
    int h_bad = 0;
    OC_HIP_CHECK(hipMemcpyAsync(&h_bad, bad.ptr, sizeof(int), hipMemcpyDeviceToHost, rt.stream));
    OC_HIP_CHECK(hipStreamSynchronize(rt.stream));
    if (h_bad) {
        s.slot_offsets8.release();
        return set_error(OC_ERR_PATTERN, "%d Laplace element entries missing from the CSR structure or beyond "
                                         "the 8-bit scatter map", h_bad);
    }
    if (static_cast<int64_t>(s.n_elements) * 8 >= INT32_MAX)
        return set_error(OC_ERR_UNSUPPORTED, "%d elements exceed the int32 element-row gather lists", s.n_elements);
    // the CSR segment of a row-gather block must fit the LDS
    int64_t max_seg = 0;
    for (int r0 = 0; r0 < s.n_rows; r0 += kLapGatherRows)
        max_seg = std::max(max_seg, s.h_row_ptr[std::min(r0 + kLapGatherRows, s.n_rows)] - s.h_row_ptr[r0]);
    if (max_seg > 8192)
        return set_error(OC_ERR_UNSUPPORTED, "Laplace CSR rows too long for the row gather (%lld entries in %d rows)",
                         static_cast<long long>(max_seg), kLapGatherRows);
    s.max_row_len = static_cast<int>(max_seg);
    // DOF -> element rows, ascending element order
    std::vector<int32_t> hconn(static_cast<size_t>(s.n_elements) * 8);
    OC_HIP_CHECK(hipMemcpy(hconn.data(), s.conn.ptr, hconn.size() * sizeof(int32_t), hipMemcpyDeviceToHost));
    std::vector<int32_t> ptr(static_cast<size_t>(s.n_rows) + 1, 0), idx(hconn.size());
    for (size_t k = 0; k < hconn.size(); ++k) ptr[hconn[k] + 1]++;
    for (int d = 0; d < s.n_rows; ++d) ptr[d + 1] += ptr[d];
    std::vector<int32_t> fillp(ptr.begin(), ptr.end() - 1);
    for (size_t k = 0; k < hconn.size(); ++k) idx[fillp[hconn[k]]++] = static_cast<int32_t>(k);
    std::vector<int32_t> gpos(idx.size());
    for (size_t p = 0; p < idx.size(); ++p) gpos[idx[p]] = static_cast<int32_t>(p);
    OC_CHECK(s.gather_ptr.upload(ptr.data(), ptr.size()));
    OC_CHECK(s.gather_idx.upload(gpos.data(), gpos.size()));  // element row -> gather position
    DevBuf<int32_t> didx;
    OC_CHECK(didx.upload(idx.data(), idx.size()));
    DevBuf<uint8_t> permuted;
    OC_CHECK(permuted.alloc(s.slot_offsets8.n));
    const int64_t n = static_cast<int64_t>(idx.size());
    permute_offsets_kernel<<<static_cast<unsigned>(std::min<int64_t>((n + 255) / 256, 65535)), 256, 0, rt.stream>>>(
        n, didx.ptr, reinterpret_cast<const uint64_t *>(s.slot_offsets8.ptr), reinterpret_cast<uint64_t *>(permuted.ptr));
    OC_CHECK(s.lap_xyz.alloc(static_cast<size_t>(4) * s.n_nodes));
    node_major_kernel<<<static_cast<unsigned>((s.n_nodes + 255) / 256), 256, 0, rt.stream>>>(s.n_nodes, s.coords.ptr,
                                                                                          s.lap_xyz.ptr);
    OC_HIP_CHECK(hipGetLastError());
    OC_HIP_CHECK(hipStreamSynchronize(rt.stream));
    s.slot_offsets8 = std::move(permuted);
    if (s.n_rows <= kLapSmallRows) s.lap_erow = std::move(didx);
    OC_CHECK(s.kbuf64.alloc(static_cast<size_t>(s.n_elements) * 64));
    return OC_NO_ERROR;
}

int launch_laplace_assemble(EquationsSet &s)
{
    if (laplace_fused_serves(s)) return launch_laplace_fused(s);
    OC_CHECK(laplace_prepare(s));
    Runtime &rt = runtime();
    if (s.lap_erow.ptr) {
        KernelTimer timer("laplace_row_gather");
        laplace_small_kernel<<<static_cast<unsigned>((s.n_rows + 7) / 8), 64,
                               static_cast<size_t>(s.max_row_len) * sizeof(double), rt.stream>>>(
            s.n_rows, s.row_ptr.ptr, s.gather_ptr.ptr, s.lap_erow.ptr, s.conn.ptr, s.lap_xyz.ptr,
            s.slot_offsets8.ptr, s.values.ptr, s.rhs.ptr);
        OC_HIP_CHECK(hipGetLastError());
        return OC_NO_ERROR;
    }
    {
        KernelTimer timer("laplace_element");
        const unsigned blocks = static_cast<unsigned>((s.n_elements + kLapThreads - 1) / kLapThreads);
        laplace_element_kernel<<<blocks, kLapThreads, 0, rt.stream>>>(s.n_elements, s.conn.ptr, s.lap_xyz.ptr,
                                                                     s.gather_idx.ptr, s.kbuf64.ptr);
        OC_HIP_CHECK(hipGetLastError());
    }
    KernelTimer timer("laplace_row_gather");
    const size_t lds = static_cast<size_t>(s.max_row_len) * sizeof(double);
    laplace_row_gather_kernel<<<static_cast<unsigned>((s.n_rows + kLapGatherRows - 1) / kLapGatherRows),
                                8 * kLapGatherRows, lds, rt.stream>>>(s.n_rows, s.row_ptr.ptr, s.gather_ptr.ptr,
                                                                       s.kbuf64.ptr, s.slot_offsets8.ptr, s.values.ptr,
                                                                       s.rhs.ptr);
    OC_HIP_CHECK(hipGetLastError());
    return OC_NO_ERROR;
}

}  // namespace oc
