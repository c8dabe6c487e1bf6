// oc_multigrid.hip -- geometric multigrid V-cycle for the displacement block
// K_uu of the Mooney-Rivlin Jacobian on regular generated meshes (no
// counterpart in the reference, whose PETSc KSP uses the preconditioner the
// user selects; solver_routines.f90:10957-11006).
//
// Hierarchy, per mesh of n^3 elements:
//   level 0  triquadratic nodes (2n+1)^3: the assembled CSR itself (u-u part,
//            columns left of the first pressure column of each row);
//   level 1  trilinear nodes (n+1)^3 on the same elements (numbered like the
//            pressure nodes); operator P0^T (A P0) from the assembled rows, A
//            masked by the free DOFs, as a 27-point stencil;
//   level l+1 (ceil(n_l/2)+1)^3 nodes, linear interpolation in each lattice
//            direction (even fine index -> coarse i/2, odd -> mean of its two
//            coarse neighbours), operator P^T A_l P on the stencils.
// Dirichlet DOFs: interpolation rows of fixed fine DOFs are dropped, a coarse
// DOF coinciding with a fixed fine DOF is fixed (its column dropped), and a
// coarse DOF left with an empty row is fixed too; fixed rows and columns are
// the identity.
// Smoother: damped nodal 3x3 block Jacobi; coarsest level (<= 3 nodes per
// direction): dense inverse per mesh.  Every reduction order is fixed, so the
// V-cycle is a fixed linear operator (usable inside GMRES).
#include <algorithm>
#include <cstdint>
#include <memory>
#include <utility>

#include "oc_fe_device.h"
#include "oc_internal.h"

namespace oc {
namespace {

__device__ __forceinline__ int find_mesh(const int *__restrict__ off, int M, int node)
{
    int lo = 0, hi = M - 1;  // off[lo] <= node < off[lo + 1]
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= node) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ double lin_weight(int delta) { return delta == 0 ? 1.0 : 0.5; }

// bf16 values: the upper 16 bits of an FP32 value, rounded to nearest even
// (NaN kept quiet)
__device__ __forceinline__ uint16_t bf16_round(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return static_cast<uint16_t>((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return static_cast<uint16_t>(u >> 16);
}

// ---- interpolation by blocks -------------------------------------------------------------
// Node i = (ix, iy, iz) of a level's lattice couples, through its own row and
// the interpolation, to the coarse nodes lo .. lo + c - 1 per direction: c = 3
// from i/2 - 1 for an even index, c = 2 from i/2 for an odd one, those outside
// the coarse grid holding zeros.  Its S = cx cy cz blocks stand in x, y, z
// order, entry rc of block s at 9 first + rc S + s; before(i) blocks precede
// index i in a direction.  Level 0 is the triquadratic lattice of 2n + 1 nodes.
__device__ __forceinline__ int product_count(int i) { return (i & 1) ? 2 : 3; }
__device__ __forceinline__ int product_lo(int i) { return (i >> 1) - ((i & 1) ? 0 : 1); }
__host__ __device__ __forceinline__ int64_t product_before(int k)
{
    return static_cast<int64_t>((k >> 1) * 5 + (k & 1) * 3);
}
__device__ __forceinline__ int64_t product_first(int dim, const int (&i)[3])
{
    const int64_t X = product_before(dim);
    const int cy = product_count(i[1]), cz = product_count(i[2]);
    return cz * cy * product_before(i[0]) + cz * X * product_before(i[1]) + X * X * product_before(i[2]);
}
// s / c for c = 2 or 3 and s < 27
__device__ __forceinline__ int div_count(int s, int c) { return c == 3 ? (s * 43) >> 7 : s >> 1; }

// What the V-cycle needs of a fine node, in one 16-byte load: with the lattice
// coordinates found by division (and the mesh by bisection) the correction
// kernel issued most of its instructions on those and took 83 us at 32^3.  The
// MgNode of node q: first block, coarse node at (lo, lo, lo) (as an index, also
// where lo is outside), and bits: k the parity of i_k, 3 + 2k lo_k outside
// (i_k = 0), 4 + 2k lo_k + c_k - 1 outside, 9 + k i_k the last, 12 an odd fine
// dimension, 16.. the coarse dimension N.
__global__ void __launch_bounds__(256)
mg_nodes_kernel(int M, const int *__restrict__ dim_f, const int *__restrict__ off_f, const int *__restrict__ dim_c,
                const int *__restrict__ off_c, const int64_t *__restrict__ first, int nn, MgNode *__restrict__ nodes)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nn) return;
    const int m = find_mesh(off_f, M, q);
    const int T = dim_f[m], N = dim_c[m], local = q - off_f[m];
    const int i[3] = {local % T, (local / T) % T, local / (T * T)};
    MgNode v;
    v.first = first[m] + product_first(T, i);
    v.lo = off_c[m] + product_lo(i[0]) + N * (product_lo(i[1]) + N * product_lo(i[2]));
    v.bits = static_cast<uint32_t>(N) << 16 | (T & 1 ? 1u << 12 : 0u);
    for (int k = 0; k < 3; ++k) {
        if (i[k] & 1) v.bits |= 1u << k;
        if (i[k] == 0) v.bits |= 8u << (2 * k);
        if (product_lo(i[k]) + product_count(i[k]) > N) v.bits |= 16u << (2 * k);
        if (i[k] == T - 1) v.bits |= 512u << k;
    }
    nodes[q] = v;
}

// ---- setup -----------------------------------------------------------------------------
// A P0 of the masked displacement block (fixed rows and columns dropped), in
// FP64, and in FP32 beside it for an FP32 Jacobian's correction kernel.  A
// group of 32 lanes stages its node's nine runs of values in LDS, read once in
// whole runs, and lane s adds the up to 27 neighbours that interpolate from
// its trilinear node, in z, y, x order.  Every later use of the interpolated
// operator reads this quarter of the matrix (15.6 blocks a node against 64).
// The rows' pressure entries go beside it, packed by the same slots, and from
// the same reading of the matrix the nodal blocks' inverses and an FP32
// Jacobian's bf16 copy: passes of their own took 282 and 382 us at 32^3, this
// one went from 758 to 946.
constexpr int kProductNodes = 4;  // per block: 36 KB of FP64 values, four blocks per CU

template <typename VT>
__global__ void __launch_bounds__(32 * kProductNodes)
q1_product_kernel(int M, const int *__restrict__ n_mesh, const int *__restrict__ q_off,
                  const MgNode *__restrict__ nodes, int nq, const int64_t *__restrict__ row_ptr,
                  const int64_t *__restrict__ pstart, const int *__restrict__ col_idx, const VT *__restrict__ vals,
                  const uint8_t *__restrict__ free_mask, double *__restrict__ ap, float *__restrict__ ap_sp,
                  VT *__restrict__ bt, const int64_t *__restrict__ uu_off, uint16_t *__restrict__ uu_bf,
                  double *__restrict__ inv_u, double *__restrict__ diag_u)
{
    __shared__ VT s_run[kProductNodes][9 * 125];
    const int lane = threadIdx.x & 31, grp = threadIdx.x >> 5;
    const int q = xcd_block(blockIdx.x, gridDim.x) * kProductNodes + grp;
    const int64_t nq64 = nq;
    VT *run = s_run[grp];
    int m = 0, n = 0, deg = 0, i[3] = {0, 0, 0}, blo[3] = {0, 0, 0}, len[3] = {0, 0, 0};
    if (q < nq) {
        m = find_mesh(q_off, M, q);
        n = n_mesh[m];
        const int T = 2 * n + 1, local = q - q_off[m];
        i[0] = local % T;
        i[1] = (local / T) % T;
        i[2] = local / (T * T);
        for (int k = 0; k < 3; ++k) {  // the neighbours are this box of the lattice, x fastest
            const int reach = (i[k] & 1) ? 1 : 2;
            blo[k] = max(i[k] - reach, 0);
            len[k] = min(i[k] + reach, 2 * n) - blo[k] + 1;
        }
        deg = len[0] * len[1] * len[2];
        const int64_t sr[3] = {row_ptr[q], row_ptr[nq64 + q], row_ptr[2 * nq64 + q]};
        for (int p = lane; p < deg; p += 32) {
            const int j = col_idx[sr[0] + p];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const bool fc = free_mask[c * nq64 + j];
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    const VT v = vals[sr[r] + c * deg + p];
                    run[(3 * r + c) * deg + p] = fc && free_mask[r * nq64 + q] ? v : static_cast<VT>(0);
                }
            }
        }
    }
    __syncthreads();
    if (q >= nq) return;
    if (sizeof(VT) == sizeof(float)) {  // four neighbours a lane; fixed DOFs' iterate is zero, so the mask is no matter
        const int n4 = (deg + 3) >> 2;
        uint2 *o = reinterpret_cast<uint2 *>(uu_bf + 9 * uu_off[q]);
        if (lane < n4)
#pragma unroll
            for (int rc = 0; rc < 9; ++rc) {
                uint32_t b[4];
#pragma unroll
                for (int n = 0; n < 4; ++n)
                    b[n] = 4 * lane + n < deg ? bf16_round(static_cast<float>(run[rc * deg + 4 * lane + n])) : 0u;
                o[rc * n4 + lane] = make_uint2(b[0] | (b[1] << 16), b[2] | (b[3] << 16));
            }
    }
    if (lane == 31) {  // no slot's lane: the node's own block, fixed DOFs as the identity
        const int own = (i[0] - blo[0]) + len[0] * ((i[1] - blo[1]) + len[1] * (i[2] - blo[2]));
        double D[9];
#pragma unroll
        for (int rc = 0; rc < 9; ++rc) D[rc] = static_cast<double>(run[rc * deg + own]);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            if (!free_mask[c * nq64 + q]) D[4 * c] = 1.0;
            diag_u[c * nq64 + q] = D[4 * c];
        }
        invert_block(D, inv_u + static_cast<int64_t>(q) * 9);
    }
    const int cx = product_count(i[0]), cy = product_count(i[1]), S = cx * cy * product_count(i[2]);
    if (lane >= S) return;
    const int K[3] = {product_lo(i[0]) + lane % cx, product_lo(i[1]) + (lane / cx) % cy,
                      product_lo(i[2]) + lane / (cx * cy)};
    // per direction the first of three neighbours 2K - 1 .. 2K + 1, moved into the
    // box, and their weights, zero outside it (the box is at least three wide)
    int lo[3];
    double w[3][3];
    bool inside = true;
    for (int k = 0; k < 3; ++k) {
        inside = inside && K[k] >= 0 && K[k] <= n;
        lo[k] = min(max(2 * K[k] - 1 - blo[k], 0), len[k] - 3);
        for (int d = 0; d < 3; ++d) {
            const int off = blo[k] + lo[k] + d - 2 * K[k];
            w[k][d] = off == 0 ? 1.0 : (off == 1 || off == -1 ? 0.5 : 0.0);
        }
    }
    double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (inside)
#pragma unroll 1
        for (int yz = 0; yz < 9; ++yz) {
            const int y = yz % 3, z = yz / 3;
            const double wy = y == 0 ? w[1][0] : (y == 1 ? w[1][1] : w[1][2]);
            const double wyz = wy * (z == 0 ? w[2][0] : (z == 1 ? w[2][1] : w[2][2]));
            const VT *v = run + lo[0] + len[0] * (lo[1] + y + len[1] * (lo[2] + z));
#pragma unroll
            for (int rc = 0; rc < 9; ++rc) {
                const VT *u = v + rc * deg;
                acc[rc] += wyz * (w[0][0] * static_cast<double>(u[0]) + w[0][1] * static_cast<double>(u[1]) +
                                  w[0][2] * static_cast<double>(u[2]));
            }
        }
    const int64_t first = nodes[q].first, at = 9 * first + lane;
    // the pressure columns are the trilinear nodes of the grid among the slots,
    // x fastest: slot s of row r at 3 first + r S + s of bt
    int plo[3], plen[3];
    for (int k = 0; k < 3; ++k) {
        plo[k] = max(product_lo(i[k]), 0);
        plen[k] = min(product_lo(i[k]) + product_count(i[k]), n + 1) - plo[k];
    }
    const int pp = (K[0] - plo[0]) + plen[0] * ((K[1] - plo[1]) + plen[1] * (K[2] - plo[2]));
#pragma unroll
    for (int r = 0; r < 3; ++r)
        bt[3 * first + r * S + lane] = inside ? vals[pstart[r * nq64 + q] + pp] : static_cast<VT>(0);
#pragma unroll
    for (int rc = 0; rc < 9; ++rc) {
        ap[at + rc * S] = acc[rc];
        if (sizeof(VT) == sizeof(float)) ap_sp[at + rc * S] = static_cast<float>(acc[rc]);
    }
}

// A P of a stencil level (A's fixed rows dropped), by blocks as above: one
// 32-lane group per node, lane s its slot, adding the up to 8 neighbours of an
// odd and 27 of an even node that interpolate from the slot's coarse node
__global__ void __launch_bounds__(256)
stencil_product_kernel(int M, const int *__restrict__ dim, const int *__restrict__ off, int nn,
                       const int *__restrict__ dim_c, const MgNode *__restrict__ nodes, const double *__restrict__ A,
                       const uint8_t *__restrict__ freed, double *__restrict__ ap)
{
    const int node = static_cast<int>((static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) >> 5);
    const int s = threadIdx.x & 31;
    if (node >= nn) return;
    const int m = find_mesh(off, M, node);
    const int N = dim[m], Nc = dim_c[m], local = node - off[m];
    const int i[3] = {local % N, (local / N) % N, local / (N * N)};
    const int cx = product_count(i[0]), cy = product_count(i[1]), S = cx * cy * product_count(i[2]);
    if (s >= S) return;
    const int K[3] = {product_lo(i[0]) + s % cx, product_lo(i[1]) + (s / cx) % cy, product_lo(i[2]) + s / (cx * cy)};
    int lo[3], hi[3];
    bool inside = true;
    for (int k = 0; k < 3; ++k) {
        inside = inside && K[k] >= 0 && K[k] < Nc;
        lo[k] = max(max(2 * K[k] - 1, i[k] - 1), 0);
        hi[k] = min(min(2 * K[k] + 1, i[k] + 1), N - 1);
    }
    double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (inside)
        for (int z = lo[2]; z <= hi[2]; ++z)
            for (int y = lo[1]; y <= hi[1]; ++y)
                for (int x = lo[0]; x <= hi[0]; ++x) {
                    const double w = lin_weight(x - 2 * K[0]) * lin_weight(y - 2 * K[1]) * lin_weight(z - 2 * K[2]);
                    const int d = (x - i[0] + 1) + 3 * (y - i[1] + 1) + 9 * (z - i[2] + 1);
                    const double *a = A + (static_cast<int64_t>(node) * 27 + d) * 9;
#pragma unroll
                    for (int rc = 0; rc < 9; ++rc) acc[rc] += w * a[rc];
                }
    double *o = ap + 9 * nodes[node].first + s;
#pragma unroll
    for (int rc = 0; rc < 9; ++rc) o[rc * S] = freed[static_cast<int64_t>(node) * 3 + rc / 3] ? acc[rc] : 0.0;
}

// the coarse stencil P^T (A P): block (I, I+d) = sum over the fine nodes 2I + s
// near I that couple to I+d, in z, y, x order; one 32-lane group per node,
// lane d < 27 its block, so a fine node's blocks are read side by side
__global__ void __launch_bounds__(256)
coarse_stencil_kernel(int M, const int *__restrict__ dim_f, const int *__restrict__ off_f,
                      const int *__restrict__ dim_c, const int *__restrict__ off_c, int nn,
                      const MgNode *__restrict__ nodes, const double *__restrict__ ap, double *__restrict__ A)
{
    const int node = static_cast<int>((static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) >> 5);
    const int d = threadIdx.x & 31;
    if (node >= nn || d >= 27) return;
    const int m = find_mesh(off_c, M, node);
    const int T = dim_f[m], N = dim_c[m], local = node - off_c[m];
    const int I[3] = {local % N, (local / N) % N, local / (N * N)}, e[3] = {d % 3 - 1, (d / 3) % 3 - 1, d / 9 - 1};
    double blk[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    int lo[3], hi[3];
    bool inside = true;
    for (int k = 0; k < 3; ++k) {  // fine nodes of the grid near both I and I + e
        inside = inside && I[k] + e[k] >= 0 && I[k] + e[k] < N;
        lo[k] = max(e[k] <= 0 ? -1 : 0, -2 * I[k]);
        hi[k] = min(e[k] >= 0 ? 1 : 0, T - 1 - 2 * I[k]);
    }
    if (inside)
        for (int s2 = lo[2]; s2 <= hi[2]; ++s2)
            for (int s1 = lo[1]; s1 <= hi[1]; ++s1)
                for (int s0 = lo[0]; s0 <= hi[0]; ++s0) {
                    const int i[3] = {2 * I[0] + s0, 2 * I[1] + s1, 2 * I[2] + s2};
                    const double w = lin_weight(s0) * lin_weight(s1) * lin_weight(s2);
                    const int cx = product_count(i[0]), cy = product_count(i[1]), S = cx * cy * product_count(i[2]);
                    const int slot = I[0] + e[0] - product_lo(i[0]) +
                                     cx * (I[1] + e[1] - product_lo(i[1]) + cy * (I[2] + e[2] - product_lo(i[2])));
                    const double *a = ap + 9 * nodes[off_f[m] + i[0] + T * (i[1] + T * i[2])].first + slot;
#pragma unroll
                    for (int rc = 0; rc < 9; ++rc) blk[rc] += w * a[rc * S];
                }
    double *o = A + (static_cast<int64_t>(node) * 27 + d) * 9;
#pragma unroll
    for (int rc = 0; rc < 9; ++rc) o[rc] = blk[rc];
}

// The V-cycle's two halves on a stencil level as one linear map each.  With one
// Jacobi step from zero, x1 = omega Dinv b, the residual restricted and one
// sweep after the correction e,
//   b_c = P^T (b - A x1)                       = R b,
//   x   = x1 + P e + omega Dinv (b - A (x1 + P e)) = U b + V e,
// with R = P^T (I - omega A Dinv) (125 blocks a coarse node), U = omega Dinv (2 I -
// omega A Dinv) (27 a node) and V = P - omega Dinv (A P) (8 to 27 a node): as many
// values as the stencil read twice, in two launches instead of four.  At 16^3 (three
// such levels) 26 us a V-cycle against 54, at 32^3 (four) 66 us against 108.

// V from A P in place, and U; 32 lanes a node, lane by slot and by neighbour.
__global__ void __launch_bounds__(256)
stencil_up_setup_kernel(int M, const int *__restrict__ dim, const int *__restrict__ off, int nn,
                        const MgNode *__restrict__ nodes, const double *__restrict__ A,
                        const uint8_t *__restrict__ freed, const double *__restrict__ Dinv, double omega,
                        double *__restrict__ U, double *__restrict__ V)
{
    const int node = static_cast<int>((static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) >> 5);
    const int d = threadIdx.x & 31;
    if (node >= nn || d >= 27) return;
    const int m = find_mesh(off, M, node);
    const int N = dim[m], local = node - off[m];
    const int i[3] = {local % N, (local / N) % N, local / (N * N)};
    double D[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) D[k] = Dinv[static_cast<int64_t>(node) * 9 + k];
    const int J[3] = {i[0] + d % 3 - 1, i[1] + (d / 3) % 3 - 1, i[2] + d / 9 - 1};
    double u[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (J[0] >= 0 && J[0] < N && J[1] >= 0 && J[1] < N && J[2] >= 0 && J[2] < N) {
        const int64_t j = off[m] + J[0] + static_cast<int64_t>(N) * (J[1] + static_cast<int64_t>(N) * J[2]);
        const double *a = A + (static_cast<int64_t>(node) * 27 + d) * 9, *q = Dinv + j * 9;
        double w[9];  // 2 I - omega A Dinv
        for (int c = 0; c < 3; ++c)
            for (int cp = 0; cp < 3; ++cp)
                w[3 * c + cp] = (d == 13 && c == cp ? 2.0 : 0.0) -
                                omega * (a[3 * c] * q[cp] + a[3 * c + 1] * q[3 + cp] + a[3 * c + 2] * q[6 + cp]);
        for (int c = 0; c < 3; ++c)
            for (int cp = 0; cp < 3; ++cp)
                u[3 * c + cp] = omega * (D[3 * c] * w[cp] + D[3 * c + 1] * w[3 + cp] + D[3 * c + 2] * w[6 + cp]);
    }
#pragma unroll
    for (int rc = 0; rc < 9; ++rc) U[(static_cast<int64_t>(node) * 9 + rc) * 27 + d] = u[rc];
    const int cx = product_count(i[0]), cy = product_count(i[1]), S = cx * cy * product_count(i[2]);
    if (d >= S) return;
    const int k[3] = {d % cx, (d / cx) % cy, d / (cx * cy)};
    double w = 1.0;
    for (int a = 0; a < 3; ++a) w *= (i[a] & 1) ? 0.5 : (k[a] == 1 ? 1.0 : 0.0);
    double *v = V + 9 * nodes[node].first + d;
    double g[9];
#pragma unroll
    for (int rc = 0; rc < 9; ++rc) g[rc] = v[rc * S];
    for (int c = 0; c < 3; ++c) {
        const bool f = freed[static_cast<int64_t>(node) * 3 + c];
        for (int cp = 0; cp < 3; ++cp) {
            const double p = f && c == cp ? w : 0.0;
            v[(3 * c + cp) * S] = p - omega * (D[3 * c] * g[cp] + D[3 * c + 1] * g[3 + cp] + D[3 * c + 2] * g[6 + cp]);
        }
    }
}

// R: a thread a (coarse node, fine neighbour 2K + d - 2), entries rc of a node
// in runs of 125
__global__ void __launch_bounds__(256)
stencil_down_setup_kernel(int M, const int *__restrict__ dim, const int *__restrict__ off,
                          const int *__restrict__ dim_c, const int *__restrict__ off_c, int nn_c,
                          const double *__restrict__ A, const uint8_t *__restrict__ freed,
                          const double *__restrict__ Dinv, const uint8_t *__restrict__ freed_c, double omega,
                          double *__restrict__ R)
{
    const int64_t total = static_cast<int64_t>(nn_c) * 125;
    for (int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < total;
         t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int node = static_cast<int>(t / 125), d = static_cast<int>(t % 125);
        const int m = find_mesh(off_c, M, node);
        const int N = dim[m], Nc = dim_c[m], local = node - off_c[m];
        const int e[3] = {d % 5 - 2, (d / 5) % 5 - 2, d / 25 - 2};
        const int K[3] = {2 * (local % Nc), 2 * ((local / Nc) % Nc), 2 * (local / (Nc * Nc))};
        double r[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        bool inside = true;
        int lo[3], hi[3];
        for (int k = 0; k < 3; ++k) {
            inside = inside && K[k] + e[k] >= 0 && K[k] + e[k] < N;
            lo[k] = max(max(-1, e[k] - 1), -K[k]);
            hi[k] = min(min(1, e[k] + 1), N - 1 - K[k]);
        }
        if (inside) {
            const int64_t N64 = N;
            double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
            for (int z = lo[2]; z <= hi[2]; ++z)
                for (int y = lo[1]; y <= hi[1]; ++y)
                    for (int x = lo[0]; x <= hi[0]; ++x) {
                        const double w = lin_weight(x) * lin_weight(y) * lin_weight(z);
                        const int64_t i = off[m] + K[0] + x + N64 * (K[1] + y + N64 * (K[2] + z));
                        const int b = (e[0] - x + 1) + 3 * (e[1] - y + 1) + 9 * (e[2] - z + 1);
                        for (int c = 0; c < 3; ++c)
                            if (freed[i * 3 + c])
                                for (int cp = 0; cp < 3; ++cp) acc[3 * c + cp] += w * A[(i * 27 + b) * 9 + 3 * c + cp];
                    }
            const int64_t j = off[m] + K[0] + e[0] + N64 * (K[1] + e[1] + N64 * (K[2] + e[2]));
            const double *q = Dinv + j * 9;
            const bool near = e[0] * e[0] <= 1 && e[1] * e[1] <= 1 && e[2] * e[2] <= 1;
            for (int c = 0; c < 3; ++c)
                for (int cp = 0; cp < 3; ++cp) {
                    const double p = near && c == cp && freed[j * 3 + c]
                                         ? lin_weight(e[0]) * lin_weight(e[1]) * lin_weight(e[2])
                                         : 0.0;
                    r[3 * c + cp] = freed_c[static_cast<int64_t>(node) * 3 + c]
                                        ? p - omega * (acc[3 * c] * q[cp] + acc[3 * c + 1] * q[3 + cp] +
                                                       acc[3 * c + 2] * q[6 + cp])
                                        : 0.0;
                }
        }
#pragma unroll
        for (int rc = 0; rc < 9; ++rc) R[(static_cast<int64_t>(node) * 9 + rc) * 125 + d] = r[rc];
    }
}

// Coarse DOFs that coincide with a fixed fine DOF are fixed (a Dirichlet
// face stays Dirichlet on every level).  Level 1 from the triquadratic mask:
// coarse node I coincides with fine lattice node 2I.
__global__ void __launch_bounds__(256) coincident_q2_kernel(int M, const int *__restrict__ n_mesh,
                                                           const int *__restrict__ q_off, int nq_total,
                                                           const int *__restrict__ off1, int nn1,
                                                           const uint8_t *__restrict__ free_mask,
                                                           uint8_t *__restrict__ freed1)
{
    for (int node = blockIdx.x * blockDim.x + threadIdx.x; node < nn1; node += gridDim.x * blockDim.x) {
        const int m = find_mesh(off1, M, node);
        const int n = n_mesh[m], N = n + 1, T = 2 * n + 1, local = node - off1[m];
        const int64_t q = q_off[m] + 2 * (local % N) +
                          static_cast<int64_t>(T) * (2 * ((local / N) % N) + static_cast<int64_t>(T) * 2 * (local / (N * N)));
        for (int c = 0; c < 3; ++c) freed1[static_cast<int64_t>(node) * 3 + c] = free_mask[static_cast<int64_t>(c) * nq_total + q];
    }
}

// level l -> l+1: coarse I coincides with fine 2I; the extra coarse node of
// an odd fine grid (2I beyond the last fine index) takes the flag of the
// boundary node it extends, so every Dirichlet face stays one on the coarse
// grid and the masked interpolation keeps full column rank
__global__ void __launch_bounds__(256) coincident_kernel(int M, const int *__restrict__ dim_f,
                                                        const int *__restrict__ off_f,
                                                        const uint8_t *__restrict__ freed_f,
                                                        const int *__restrict__ dim_c, const int *__restrict__ off_c,
                                                        int nn_c, uint8_t *__restrict__ freed_c)
{
    for (int node = blockIdx.x * blockDim.x + threadIdx.x; node < nn_c; node += gridDim.x * blockDim.x) {
        const int m = find_mesh(off_c, M, node);
        const int Nc = dim_c[m], Nf = dim_f[m], local = node - off_c[m];
        const int i0 = min(2 * (local % Nc), Nf - 1), i1 = min(2 * ((local / Nc) % Nc), Nf - 1),
                  i2 = min(2 * (local / (Nc * Nc)), Nf - 1);
        const int64_t f = off_f[m] + i0 + static_cast<int64_t>(Nf) * (i1 + static_cast<int64_t>(Nf) * i2);
        for (int c = 0; c < 3; ++c) freed_c[static_cast<int64_t>(node) * 3 + c] = freed_f[f * 3 + c];
    }
}

// freed &= (diagonal != 0): a DOF whose Galerkin row is empty is fixed too
__global__ void __launch_bounds__(256) level_freed_kernel(int nn, const double *__restrict__ A,
                                                         uint8_t *__restrict__ freed)
{
    for (int node = blockIdx.x * blockDim.x + threadIdx.x; node < nn; node += gridDim.x * blockDim.x) {
        const double *D = A + (static_cast<int64_t>(node) * 27 + 13) * 9;
        for (int c = 0; c < 3; ++c) {
            const int64_t k = static_cast<int64_t>(node) * 3 + c;
            freed[k] = (freed[k] && D[4 * c] != 0.0) ? 1 : 0;
        }
    }
}

// Fixed rows and columns replaced by the identity; inverse diagonal blocks.
__global__ void __launch_bounds__(256) level_mask_kernel(int M, const int *__restrict__ dim,
                                                        const int *__restrict__ off, int nn, double *__restrict__ A,
                                                        const uint8_t *__restrict__ freed, double *__restrict__ Dinv)
{
    const int64_t total = static_cast<int64_t>(nn) * 27;
    for (int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < total;
         t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int node = static_cast<int>(t / 27), d = static_cast<int>(t % 27);
        const int m = find_mesh(off, M, node);
        const int N = dim[m], local = node - off[m];
        const int J[3] = {local % N + d % 3 - 1, (local / N) % N + (d / 3) % 3 - 1, local / (N * N) + d / 9 - 1};
        double *a = A + t * 9;
        if (J[0] < 0 || J[0] >= N || J[1] < 0 || J[1] >= N || J[2] < 0 || J[2] >= N) {
            for (int k = 0; k < 9; ++k) a[k] = 0.0;
            continue;
        }
        const int64_t j = off[m] + J[0] + static_cast<int64_t>(N) * (J[1] + static_cast<int64_t>(N) * J[2]);
        for (int c = 0; c < 3; ++c)
            for (int cp = 0; cp < 3; ++cp) {
                const bool keep = freed[static_cast<int64_t>(node) * 3 + c] && freed[j * 3 + cp];
                if (!keep) a[3 * c + cp] = (d == 13 && c == cp) ? 1.0 : 0.0;
            }
        if (d != 13) continue;
        const double *D = a;
        const double c00 = D[4] * D[8] - D[5] * D[7], c01 = D[5] * D[6] - D[3] * D[8], c02 = D[3] * D[7] - D[4] * D[6];
        const double det = D[0] * c00 + D[1] * c01 + D[2] * c02;
        double *o = Dinv + static_cast<int64_t>(node) * 9;
        if (fabs(det) < 1e-300) {
            for (int i = 0; i < 9; ++i) o[i] = (i % 4 == 0) ? 1.0 : 0.0;
            continue;
        }
        const double id = 1.0 / det;
        o[0] = c00 * id;
        o[1] = (D[2] * D[7] - D[1] * D[8]) * id;
        o[2] = (D[1] * D[5] - D[2] * D[4]) * id;
        o[3] = c01 * id;
        o[4] = (D[0] * D[8] - D[2] * D[6]) * id;
        o[5] = (D[2] * D[3] - D[0] * D[5]) * id;
        o[6] = c02 * id;
        o[7] = (D[1] * D[6] - D[0] * D[7]) * id;
        o[8] = (D[0] * D[4] - D[1] * D[3]) * id;
    }
}

constexpr int kCoarseMax = 81;  // 27 nodes x 3 components

// dense inverse of each mesh's coarsest level (in-place Gauss-Jordan, one
// block per mesh; the masked operator is symmetric positive definite).  The
// steps follow one another, so a step's latency is all there is to it: the
// matrix stays in registers (thread by column and row modulo 12), a step puts
// the pivot's row and column into the LDS buffer of its parity and takes one
// barrier.  81 DOFs: 105 us; in LDS with three barriers a step 287 us.
constexpr int kInvGroups = 12, kInvRows = (kCoarseMax + kInvGroups - 1) / kInvGroups;

__global__ void __launch_bounds__(1024) coarse_inverse_kernel(int M, const int *__restrict__ dim,
                                                             const int *__restrict__ off,
                                                             const double *__restrict__ A, int stride,
                                                             double *__restrict__ inv)
{
    __shared__ double s_row[2][kCoarseMax], s_col[2][kInvGroups * kInvRows];
    const int m = blockIdx.x;
    if (m >= M) return;
    const int N = dim[m], nodes = N * N * N, nd = 3 * nodes;
    const int j = threadIdx.x % kCoarseMax, g = threadIdx.x / kCoarseMax;
    const bool mine = g < kInvGroups && j < nd;
    double a[kInvRows];
#pragma unroll
    for (int r = 0; r < kInvRows; ++r) {
        const int i = g + kInvGroups * r;
        a[r] = 0.0;
        if (!mine || i >= nd) continue;
        const int nr = i / 3, c = i % 3, nc = j / 3, cp = j % 3;
        const int e0 = nc % N - nr % N, e1 = (nc / N) % N - (nr / N) % N, e2 = nc / (N * N) - nr / (N * N);
        if (e0 >= -1 && e0 <= 1 && e1 >= -1 && e1 <= 1 && e2 >= -1 && e2 <= 1)
            a[r] = A[((static_cast<int64_t>(off[m]) + nr) * 27 + (e0 + 1) + 3 * (e1 + 1) + 9 * (e2 + 1)) * 9 + 3 * c + cp];
    }
    for (int k = 0; k < nd; ++k) {
        double *row = s_row[k & 1], *col = s_col[k & 1];
        if (mine) {
#pragma unroll
            for (int r = 0; r < kInvRows; ++r) {
                if (g + kInvGroups * r == k) row[j] = a[r];
                if (j == k) col[g + kInvGroups * r] = a[r];
            }
        }
        __syncthreads();
        if (mine) {
            const double p = fabs(col[k]) > 1e-300 ? col[k] : 1.0;  // fixed DOFs are identity rows
            const double pr = (j == k ? 1.0 : row[j]) / p;
#pragma unroll
            for (int r = 0; r < kInvRows; ++r) {
                const int i = g + kInvGroups * r;
                a[r] = i == k ? pr : (j == k ? 0.0 : a[r]) - col[i] * pr;
            }
        }
    }
#pragma unroll
    for (int r = 0; r < kInvRows; ++r) {
        const int i = g + kInvGroups * r;
        if (mine && i < nd) inv[static_cast<int64_t>(m) * stride + i * nd + j] = a[r];
    }
}

// The last two levels as one dense matrix per mesh, D = U + V Ainv R on the
// level above the coarsest (at most 5 nodes per direction, 375 DOFs): one
// product replaces three launches of 4 us whose work is next to nothing (load
// steps of 4^3 to 12^3 elements 4 to 8% faster, 16^3 37.4 -> 37.0 ms).
// W = Ainv R first, then D; blockIdx.y is the mesh.
__global__ void __launch_bounds__(256)
dense_w_kernel(const int *__restrict__ dim, const int *__restrict__ dim_c, const int *__restrict__ off_c,
               const double *__restrict__ R, const double *__restrict__ inv, int inv_stride, int w_stride,
               double *__restrict__ W)
{
    const int m = blockIdx.y, N = dim[m], Nc = dim_c[m], nf = 3 * N * N * N, nc = 3 * Nc * Nc * Nc;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < nc * nf; t += gridDim.x * blockDim.x) {
        const int i = t / nf, j = t % nf, node = j / 3, cp = j % 3;
        const int J[3] = {node % N, (node / N) % N, node / (N * N)};
        int lo[3], hi[3];  // coarse nodes with J within two of 2K
        for (int k = 0; k < 3; ++k) {
            lo[k] = max((J[k] - 1) / 2, 0);
            hi[k] = min((J[k] + 2) / 2, Nc - 1);
        }
        double acc = 0.0;
        for (int z = lo[2]; z <= hi[2]; ++z)
            for (int y = lo[1]; y <= hi[1]; ++y)
                for (int x = lo[0]; x <= hi[0]; ++x) {
                    const int K = x + Nc * (y + Nc * z);
                    const int d = (J[0] - 2 * x + 2) + 5 * (J[1] - 2 * y + 2) + 25 * (J[2] - 2 * z + 2);
                    const double *a = inv + static_cast<int64_t>(m) * inv_stride + i * nc + 3 * K;
                    const double *r = R + (static_cast<int64_t>(off_c[m] + K) * 9 + cp) * 125 + d;
                    acc += a[0] * r[0] + a[1] * r[3 * 125] + a[2] * r[6 * 125];
                }
        W[static_cast<int64_t>(m) * w_stride + t] = acc;
    }
}

__global__ void __launch_bounds__(256)
dense_kernel(const int *__restrict__ dim, const int *__restrict__ off, const int *__restrict__ dim_c,
             const MgNode *__restrict__ nodes, const double *__restrict__ U, const double *__restrict__ V,
             const double *__restrict__ W, int w_stride, int stride, double *__restrict__ D)
{
    const int m = blockIdx.y, N = dim[m], Nc = dim_c[m], nf = 3 * N * N * N;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < nf * nf; t += gridDim.x * blockDim.x) {
        const int row = t / nf, j = t % nf, node = row / 3, c = row % 3, nj = j / 3, cp = j % 3;
        const int I[3] = {node % N, (node / N) % N, node / (N * N)};
        const int e[3] = {nj % N - I[0], (nj / N) % N - I[1], nj / (N * N) - I[2]};
        double acc = 0.0;
        if (e[0] >= -1 && e[0] <= 1 && e[1] >= -1 && e[1] <= 1 && e[2] >= -1 && e[2] <= 1)
            acc = U[(static_cast<int64_t>(off[m] + node) * 9 + 3 * c + cp) * 27 + (e[0] + 1) + 3 * (e[1] + 1) + 9 * (e[2] + 1)];
        const int cx = product_count(I[0]), cy = product_count(I[1]), S = cx * cy * product_count(I[2]);
        const double *v = V + 9 * nodes[off[m] + node].first + 3 * c * S;
        const double *w = W + static_cast<int64_t>(m) * w_stride + j;
        for (int s = 0; s < S; ++s) {
            const int yz = div_count(s, cx), sz = div_count(yz, cy);
            const int K[3] = {product_lo(I[0]) + s - cx * yz, product_lo(I[1]) + yz - cy * sz, product_lo(I[2]) + sz};
            if (K[0] < 0 || K[0] >= Nc || K[1] < 0 || K[1] >= Nc || K[2] < 0 || K[2] >= Nc) continue;
            const int64_t k = 3 * (K[0] + Nc * (K[1] + Nc * K[2]));
            acc += v[s] * w[k * nf] + v[S + s] * w[(k + 1) * nf] + v[2 * S + s] * w[(k + 2) * nf];
        }
        D[static_cast<int64_t>(m) * stride + t] = acc;
    }
}

// ---- V-cycle kernels -------------------------------------------------------------------

// The packed bf16 copy of K_uu (EquationsSet::uu_bf): padded neighbour
// counts, then the padded column lists, once per set
__global__ void __launch_bounds__(256) uu_degp_kernel(int nq, const int64_t *__restrict__ row_ptr,
                                                     const int64_t *__restrict__ pstart, int64_t *__restrict__ degp)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nq) return;
    const int64_t deg = (pstart[i] - row_ptr[i]) / 3;
    degp[i] = (deg + 3) & ~static_cast<int64_t>(3);
}

constexpr int kPackLanes = 32;  // lanes per node in the packing kernels

__global__ void __launch_bounds__(256) uu_cols_kernel(int nq, const int64_t *__restrict__ row_ptr,
                                                     const int64_t *__restrict__ pstart, const int *__restrict__ col_idx,
                                                     const int64_t *__restrict__ uu_off, int *__restrict__ uu_col)
{
    const int lane = threadIdx.x % kPackLanes;
    const int i = static_cast<int>((static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / kPackLanes);
    if (i >= nq) return;
    const int64_t s0 = row_ptr[i], off = uu_off[i];
    const int deg = static_cast<int>((pstart[i] - s0) / 3), degp = static_cast<int>(uu_off[i + 1] - off);
    for (int p = lane; p < degp; p += kPackLanes) uu_col[off + p] = p < deg ? col_idx[s0 + p] : i;
}

// values of one FP32 Jacobian into the packed bf16 copy, without a multigrid setup
// (whose q1_product_kernel forms it in passing): the autotuner times the smoother on it
__global__ void __launch_bounds__(256) uu_pack_kernel(int nq, const int64_t *__restrict__ row_ptr,
                                                     const int64_t *__restrict__ pstart, const float *__restrict__ v,
                                                     const int64_t *__restrict__ uu_off, uint16_t *__restrict__ uu_bf)
{
    const int lane = threadIdx.x % kPackLanes;
    const int i = static_cast<int>((static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / kPackLanes);
    if (i >= nq) return;
    const int64_t nq64 = nq, off = uu_off[i];
    const int deg = static_cast<int>((pstart[i] - row_ptr[i]) / 3), degp = static_cast<int>(uu_off[i + 1] - off);
    const int64_t rows[3] = {row_ptr[i], row_ptr[nq64 + i], row_ptr[2 * nq64 + i]};
    // run (r, c) starts at 9 off + (3 r + c) degp, a multiple of four (degp
    // and every offset are), so a lane writes two neighbours as one 4-byte
    // word: the lower address holds the even neighbour
    uint32_t *o = reinterpret_cast<uint32_t *>(uu_bf + 9 * off);
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float *src = v + rows[r] + static_cast<int64_t>(c) * deg;
            uint32_t *dst = o + (3 * r + c) * (degp / 2);
            for (int p = 2 * lane; p < degp; p += 2 * kPackLanes) {
                const uint32_t lo = p < deg ? bf16_round(src[p]) : 0u;
                const uint32_t hi = p + 1 < deg ? bf16_round(src[p + 1]) : 0u;
                dst[p / 2] = lo | (hi << 16);
            }
        }
}

// the iterate as FP32 node quadruples (x, y, z, 0) for the bf16 kernels'
// gathers: one 16-byte load per neighbour, and no accuracy lost against the
// bf16 values' 8-bit significands
__global__ void __launch_bounds__(256) pack_x4_kernel(int nq, const double *__restrict__ x, float4 *__restrict__ x4)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nq) return;
    const int64_t nq64 = nq;
    x4[j] = make_float4(static_cast<float>(x[j]), static_cast<float>(x[nq64 + j]), static_cast<float>(x[2 * nq64 + j]),
                        0.0f);
}

// level 0 residual by nodes from the packed bf16 K_uu: one group of kLanes
// lanes per node; a lane takes four neighbours at a time (kQ quads in
// flight): one 16-byte column load, one 8-byte load per (row, component)
// run and one 16-byte iterate load per neighbour (x4: pack_x4_kernel of x).
// r = b - K_uu x on free rows, 0 on fixed ones; kSweep 1 writes the block
// Jacobi update x + omega Kblock^-1 r instead (as uu_node_residual_kernel),
// and with out4 also its FP32 node quadruples for the next pass.
template <int kLanes, int kSweep, int kQ>
__global__ void __launch_bounds__(256)
uu_node_bf16_kernel(int nq, const int64_t *__restrict__ uu_off, const int *__restrict__ uu_col,
                    const uint16_t *__restrict__ uu_bf, const uint8_t *__restrict__ free_mask,
                    const double *__restrict__ b, const float4 *__restrict__ x4, const double *__restrict__ x,
                    const double *__restrict__ inv_u, double omega, const double *__restrict__ scale,
                    double *__restrict__ out, float *__restrict__ out4)
{
    const int lane = threadIdx.x % kLanes;
    const int64_t xb = xcd_block(blockIdx.x, gridDim.x);
    const int i = static_cast<int>((xb * blockDim.x + threadIdx.x) / kLanes);
    if (i >= nq) return;  // whole groups
    const int64_t nq64 = nq, off = uu_off[i];
    const int n4 = static_cast<int>((uu_off[i + 1] - off) >> 2);
    const int4 *cols = reinterpret_cast<const int4 *>(uu_col + off);
    const uint2 *vals = reinterpret_cast<const uint2 *>(uu_bf + 9 * off);  // run rc: vals[rc n4 + q]
    double a[3] = {0.0, 0.0, 0.0};
    for (int q0 = lane; q0 < n4; q0 += kLanes * kQ) {
        int4 cj[kQ];
        uint2 v[kQ][9];
#pragma unroll
        for (int u = 0; u < kQ; ++u) {
            // lanes past the end repeat the last quad's loads and select zeros
            const bool ok = q0 + u * kLanes < n4;
            const int q = min(q0 + u * kLanes, n4 - 1);
            cj[u] = cols[q];
#pragma unroll
            for (int rc = 0; rc < 9; ++rc) {
                const uint2 w = vals[rc * n4 + q];
                v[u][rc] = make_uint2(ok ? w.x : 0u, ok ? w.y : 0u);
            }
        }
#pragma unroll
        for (int u = 0; u < kQ; ++u) {
            const int j[4] = {cj[u].x, cj[u].y, cj[u].z, cj[u].w};
            double xv[4][3];
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                const float4 q4 = x4[j[n]];
                xv[n][0] = q4.x;
                xv[n][1] = q4.y;
                xv[n][2] = q4.z;
            }
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const uint2 w = v[u][3 * r + c];
                    const float f[4] = {__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u),
                                        __uint_as_float(w.y << 16), __uint_as_float(w.y & 0xffff0000u)};
#pragma unroll
                    for (int n = 0; n < 4; ++n) a[r] = fma(static_cast<double>(f[n]), xv[n][c], a[r]);
                }
        }
    }
    double a0 = a[0], a1 = a[1], a2 = a[2];
#pragma unroll
    for (int o = kLanes / 2; o > 0; o >>= 1) {
        a0 += __shfl_xor(a0, o, kLanes);
        a1 += __shfl_xor(a1, o, kLanes);
        a2 += __shfl_xor(a2, o, kLanes);
    }
    if (kSweep == 0) {
        if (lane < 3) {
            const int64_t row = lane * nq64 + i;
            const double a = lane == 0 ? a0 : (lane == 1 ? a1 : a2);
            out[row] = free_mask[row] ? b[row] - a : 0.0;
        }
    } else if (lane < 3) {
        const double r0 = free_mask[i] ? b[i] - a0 : 0.0;
        const double r1 = free_mask[nq64 + i] ? b[nq64 + i] - a1 : 0.0;
        const double r2 = free_mask[2 * nq64 + i] ? b[2 * nq64 + i] - a2 : 0.0;
        const double *o = inv_u + static_cast<int64_t>(i) * 9 + 3 * lane;
        const int64_t row = lane * nq64 + i;
        const double xn = x[row] + omega * (o[0] * r0 + o[1] * r1 + o[2] * r2);
        out[row] = scale ? scale[row] * xn : xn;
        if (out4) out4[4 * static_cast<int64_t>(i) + lane] = static_cast<float>(xn);
    }
}

// level 0 residual by nodes (EquationsSet::node_rows): one group of kLanes
// lanes per node reads the neighbour list once and the nine value blocks of
// its three rows; r = b - K_uu x on free rows, 0 on fixed ones.  kSweep 0
// writes r to out; kSweep 1 writes the block Jacobi update
// x + omega Kblock^-1 r to out (not x: neighbours still read the old x).
template <typename VT, int kLanes, int kSweep, int kU>
__global__ void __launch_bounds__(256)
uu_node_residual_kernel(int nq, const int64_t *__restrict__ row_ptr, const int64_t *__restrict__ pstart,
                        const int *__restrict__ col_idx, const VT *__restrict__ vals,
                        const uint8_t *__restrict__ free_mask, const double *__restrict__ b,
                        const double *__restrict__ x, const double *__restrict__ inv_u, double omega,
                        const double *__restrict__ scale, double *__restrict__ out)
{
    const int lane = threadIdx.x % kLanes;
    const int64_t xb = xcd_block(blockIdx.x, gridDim.x);
    const int i = static_cast<int>((xb * blockDim.x + threadIdx.x) / kLanes);
    if (i >= nq) return;  // whole groups
    const int64_t nq64 = nq;
    const int64_t sr[3] = {row_ptr[i], row_ptr[nq64 + i], row_ptr[2 * nq64 + i]};
    const int deg = static_cast<int>((pstart[i] - sr[0]) / 3);
    double a[3] = {0.0, 0.0, 0.0};
    node_rows_uu<VT, kLanes, kU>(sr, deg, lane, nq64, col_idx, vals, x, a);
    double a0 = a[0], a1 = a[1], a2 = a[2];
#pragma unroll
    for (int o = kLanes / 2; o > 0; o >>= 1) {
        a0 += __shfl_xor(a0, o, kLanes);
        a1 += __shfl_xor(a1, o, kLanes);
        a2 += __shfl_xor(a2, o, kLanes);
    }
    if (kSweep == 0) {
        if (lane < 3) {
            const int64_t row = lane * nq64 + i;
            const double a = lane == 0 ? a0 : (lane == 1 ? a1 : a2);
            out[row] = free_mask[row] ? b[row] - a : 0.0;
        }
    } else if (lane < 3) {
        const double r0 = free_mask[i] ? b[i] - a0 : 0.0;
        const double r1 = free_mask[nq64 + i] ? b[nq64 + i] - a1 : 0.0;
        const double r2 = free_mask[2 * nq64 + i] ? b[2 * nq64 + i] - a2 : 0.0;
        const double *o = inv_u + static_cast<int64_t>(i) * 9 + 3 * lane;
        const int64_t row = lane * nq64 + i;
        const double xn = x[row] + omega * (o[0] * r0 + o[1] * r1 + o[2] * r2);
        out[row] = scale ? scale[row] * xn : xn;
    }
}

// the same by one wavefront per node (node_rows_flat): FP64 values' default
// where the rows fit its LDS.  At 32^3 276 us against 332 with 16 lanes x 2
// neighbours, at 16^3 30.8 against 38.6.
template <typename VT, int kSweep>
__global__ void __launch_bounds__(256)
uu_flat_kernel(int nq, const int64_t *__restrict__ row_ptr, const int64_t *__restrict__ pstart,
               const int *__restrict__ col_idx, const VT *__restrict__ vals, const uint8_t *__restrict__ free_mask,
               const double *__restrict__ b, const double *__restrict__ x, const double *__restrict__ inv_u,
               double omega, const double *__restrict__ scale, double *__restrict__ out)
{
    __shared__ double s_x[4][kFlatLds];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = xcd_block(blockIdx.x, gridDim.x) * 4 + wave;
    if (i >= nq) return;  // whole wavefronts
    double a[3] = {0.0, 0.0, 0.0};
    node_rows_flat<VT, false>(i, nq, lane, row_ptr, pstart, col_idx, vals, x, s_x[wave], a);
    const double t = wave_total3(a, lane);
    const int c = lane >> 4;
    const int64_t row = c * static_cast<int64_t>(nq) + i;
    const bool mine = (lane & 15) == 0 && c < 3;
    const double r = mine && free_mask[row] ? b[row] - t : 0.0;
    if (kSweep == 0) {
        if (mine) out[row] = r;
        return;
    }
    const double r0 = __shfl(r, 0), r1 = __shfl(r, 16), r2 = __shfl(r, 32);
    if (!mine) return;
    const double *o = inv_u + static_cast<int64_t>(i) * 9 + 3 * c;
    const double xn = x[row] + omega * (o[0] * r0 + o[1] * r1 + o[2] * r2);
    out[row] = scale ? scale[row] * xn : xn;
}

// The V-cycle's start: z_p = scale inv_p .* r_p, t = r_u - B^T (inv_p .* r_p) on
// free rows (0 on fixed ones) and the first smoothing step x = omega Kblock^-1 t
// from zero (and, with x4, its FP32 node quadruples for the bf16 passes).  A
// group of 8 lanes per node, lane by pressure neighbour as in q1_correct_kernel:
// the packed B^T needs no columns and its lines hold nothing else, where the
// CSR rows' ends are 16 entries in lines of 32.  At 32^3 with FP32 values 39 us
// against 57 + 9 for the product from the CSR and the step (and 5 for the
// scaling of z); 16^3 in FP64 9.1 against 10.3 + 4.6 (and 4.7).
template <typename VT>
__global__ void __launch_bounds__(256)
mg_start_kernel(int nq, int nl, const MgNode *__restrict__ nodes, const VT *__restrict__ bt,
                const double *__restrict__ inv_p, const double *__restrict__ r, const double *__restrict__ scale,
                const uint8_t *__restrict__ free_mask, const double *__restrict__ inv_u, double omega,
                double *__restrict__ z, double *__restrict__ t, double *__restrict__ x, float *__restrict__ x4)
{
    constexpr int kLanes = 8, kRounds = 4;  // 27 slots at most
    const int lane = threadIdx.x % kLanes;
    const int64_t xb = xcd_block(blockIdx.x, gridDim.x);
    const int q = static_cast<int>((xb * blockDim.x + threadIdx.x) / kLanes);
    if (q >= nq) return;  // whole groups
    const int64_t nq64 = nq;
    const double *rp = r + 3 * nq64;
    if (q < nl && lane == kLanes - 1) z[3 * nq64 + q] = scale[3 * nq64 + q] * (inv_p[q] * rp[q]);
    const MgNode nd = nodes[q];
    const int N = static_cast<int>(nd.bits >> 16);
    const bool odd[3] = {(nd.bits & 1) != 0, (nd.bits & 2) != 0, (nd.bits & 4) != 0};
    const int cx = odd[0] ? 2 : 3, cy = odd[1] ? 2 : 3, cz = odd[2] ? 2 : 3, S = cx * cy * cz;
    const VT *a = bt + 3 * nd.first;
    double v[4] = {0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < kRounds; ++u) {
        const int s = lane + u * kLanes;
        if (s >= S) break;
        const int yz = div_count(s, cx), sz = div_count(yz, cy), k[3] = {s - cx * yz, yz - cy * sz, sz};
        bool inside = true;
#pragma unroll
        for (int d = 0; d < 3; ++d)
            inside = inside && !(k[d] == 0 && (nd.bits >> (3 + 2 * d) & 1)) && !(k[d] == 2 && (nd.bits >> (4 + 2 * d) & 1));
        const int l = inside ? nd.lo + k[0] + N * (k[1] + N * k[2]) : 0;
        const double zp = inside ? inv_p[l] * rp[l] : 0.0;
#pragma unroll
        for (int c = 0; c < 3; ++c) v[c] += static_cast<double>(a[c * S + s]) * zp;
    }
    // lanes 2c and 2c + 1 of the group are left with the total of v[c]
    const bool h4 = lane & 4, h2 = lane & 2;
    double f[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) f[k] = (h4 ? v[k + 2] : v[k]) + __shfl_xor(h4 ? v[k] : v[k + 2], 4, kLanes);
    double sum = (h2 ? f[1] : f[0]) + __shfl_xor(h2 ? f[0] : f[1], 2, kLanes);
    sum += __shfl_xor(sum, 1, kLanes);
    const int c = lane >> 1;
    const int64_t row = c * nq64 + q;
    const double tc = c < 3 && free_mask[row] ? r[row] - sum : 0.0;
    const double t0 = __shfl(tc, 0, kLanes), t1 = __shfl(tc, 2, kLanes), t2 = __shfl(tc, 4, kLanes);
    if (c >= 3 || (lane & 1)) return;
    const double *o = inv_u + static_cast<int64_t>(q) * 9 + 3 * c;
    const double xn = omega * (o[0] * t0 + o[1] * t1 + o[2] * t2);
    t[row] = tc;
    x[row] = xn;
    if (x4) x4[4 * static_cast<int64_t>(q) + c] = static_cast<float>(xn);
}

// level 0 -> 1 restriction b1 = P0^T r0 (r0 is zero on fixed DOFs)
__global__ void __launch_bounds__(256) restrict_q2_kernel(int M, const int *__restrict__ n_mesh,
                                                         const int *__restrict__ q_off, int nq_total,
                                                         const int *__restrict__ off1, int nn1,
                                                         const uint8_t *__restrict__ freed1,
                                                         const double *__restrict__ r0, double *__restrict__ b1)
{
    // one 32-lane group per coarse node: lane s < 27 takes fine node s of its
    // neighbourhood, a fixed butterfly adds them
    const int node = static_cast<int>((static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) >> 5);
    const int s = threadIdx.x & 31;
    if (node >= nn1) return;  // whole 32-lane groups
    const int m = find_mesh(off1, M, node);
    const int n = n_mesh[m], N = n + 1, T = 2 * n + 1, local = node - off1[m];
    const int I[3] = {local % N, (local / N) % N, local / (N * N)};
    double acc[3] = {0.0, 0.0, 0.0};
    if (s < 27) {
        const int i[3] = {2 * I[0] + s % 3 - 1, 2 * I[1] + (s / 3) % 3 - 1, 2 * I[2] + s / 9 - 1};
        if (i[0] >= 0 && i[0] < T && i[1] >= 0 && i[1] < T && i[2] >= 0 && i[2] < T) {
            const double w = lin_weight(s % 3 - 1) * lin_weight((s / 3) % 3 - 1) * lin_weight(s / 9 - 1);
            const int64_t q = q_off[m] + i[0] + static_cast<int64_t>(T) * (i[1] + static_cast<int64_t>(T) * i[2]);
#pragma unroll
            for (int c = 0; c < 3; ++c) acc[c] = w * r0[static_cast<int64_t>(c) * nq_total + q];
        }
    }
#pragma unroll
    for (int sh = 16; sh > 0; sh >>= 1)
#pragma unroll
        for (int c = 0; c < 3; ++c) acc[c] += __shfl_xor(acc[c], sh, 32);
    if (s != 0) return;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const int64_t k = static_cast<int64_t>(node) * 3 + c;
        b1[k] = freed1[k] ? acc[c] : 0.0;
    }
}

// Coarse correction of level 0 and the smoothing sweep after it, in place:
//   x <- x + P0 e + omega Kblock^-1 (r0 - A P0 e),
// which is the sweep at x + P0 e, as its residual is r0 - A P0 e with r0 the
// residual that was restricted: the sweep reads A P0, a quarter of the matrix,
// and the prolongation needs no pass of its own.  One group of 8 lanes per
// node, lane by trilinear neighbour (8, 12, 18 or 27 of them: 2.5 rounds on
// average); the loads of a round depend on the node's record alone.  At 32^3
// with FP32 values 63 us (205 MB) where the sweep over the bf16 matrix and the
// prolongation took 124 + 14; at 16^3 in FP64 17 us where they took 38 + 7.
template <typename VT>
__global__ void __launch_bounds__(256)
q1_correct_kernel(int nq, const MgNode *__restrict__ nodes, const VT *__restrict__ ap, const double *__restrict__ e,
                  const uint8_t *__restrict__ free_mask, const double *__restrict__ r0,
                  const double *__restrict__ inv_u, double omega, const double *__restrict__ scale,
                  double *__restrict__ x, float *__restrict__ x4)
{
    constexpr int kLanes = 8, kRounds = 4;  // 27 slots at most
    const int lane = threadIdx.x % kLanes;
    const int64_t xb = xcd_block(blockIdx.x, gridDim.x);
    const int q = static_cast<int>((xb * blockDim.x + threadIdx.x) / kLanes);
    if (q >= nq) return;  // whole groups
    const int64_t nq64 = nq;
    const MgNode nd = nodes[q];
    const int N = static_cast<int>(nd.bits >> 16);
    const bool odd[3] = {(nd.bits & 1) != 0, (nd.bits & 2) != 0, (nd.bits & 4) != 0};
    const int cx = odd[0] ? 2 : 3, cy = odd[1] ? 2 : 3, cz = odd[2] ? 2 : 3, S = cx * cy * cz;
    const VT *a = ap + 9 * nd.first;
    double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // A P0 e and P0 e
#pragma unroll
    for (int u = 0; u < kRounds; ++u) {
        const int s = lane + u * kLanes;
        if (s >= S) break;
        const int yz = div_count(s, cx), sz = div_count(yz, cy), k[3] = {s - cx * yz, yz - cy * sz, sz};
        double w = 1.0;
        bool inside = true;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            w *= odd[d] ? 0.5 : (k[d] == 1 ? 1.0 : 0.0);
            inside = inside && !(k[d] == 0 && (nd.bits >> (3 + 2 * d) & 1)) && !(k[d] == 2 && (nd.bits >> (4 + 2 * d) & 1));
        }
        const double *ek = e + 3 * static_cast<int64_t>(inside ? nd.lo + k[0] + N * (k[1] + N * k[2]) : 0);
        double b[9];
#pragma unroll
        for (int rc = 0; rc < 9; ++rc) b[rc] = static_cast<double>(a[rc * S + s]);  // zeros where outside
        const double ev[3] = {inside ? ek[0] : 0.0, inside ? ek[1] : 0.0, inside ? ek[2] : 0.0};
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            v[r] += b[3 * r] * ev[0] + b[3 * r + 1] * ev[1] + b[3 * r + 2] * ev[2];
            v[4 + r] += w * ev[r];
        }
    }
    // lane l of the group is left with the total of v[l]
    const bool h4 = lane & 4, h2 = lane & 2, h1 = lane & 1;
    double f[4], t[2];
#pragma unroll
    for (int k = 0; k < 4; ++k) f[k] = (h4 ? v[k + 4] : v[k]) + __shfl_xor(h4 ? v[k] : v[k + 4], 4, kLanes);
#pragma unroll
    for (int k = 0; k < 2; ++k) t[k] = (h2 ? f[k + 2] : f[k]) + __shfl_xor(h2 ? f[k] : f[k + 2], 2, kLanes);
    const double sum = (h1 ? t[1] : t[0]) + __shfl_xor(h1 ? t[0] : t[1], 1, kLanes);
    const int64_t row = (lane & 3) * nq64 + q;
    const double d = lane < 3 ? r0[row] - sum : 0.0;
    const double d0 = __shfl(d, 0, kLanes), d1 = __shfl(d, 1, kLanes), d2 = __shfl(d, 2, kLanes);
    const double pe = __shfl(sum, 4 | lane, kLanes);
    if (lane >= 3) return;
    const double *o = inv_u + static_cast<int64_t>(q) * 9 + 3 * lane;
    const double xn = x[row] + (free_mask[row] ? pe : 0.0) + omega * (o[0] * d0 + o[1] * d1 + o[2] * d2);
    x[row] = scale ? scale[row] * xn : xn;
    if (x4) x4[4 * static_cast<int64_t>(q) + lane] = static_cast<float>(xn);
}

// b_c = R b: one wavefront per coarse node, lanes over its 125 fine neighbours
__global__ void __launch_bounds__(256)
stencil_down_kernel(int M, const int *__restrict__ dim, const int *__restrict__ off, const int *__restrict__ dim_c,
                    const int *__restrict__ off_c, int nn_c, const double *__restrict__ R,
                    const double *__restrict__ b, double *__restrict__ bc)
{
    const int node = static_cast<int>(blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    if (node >= nn_c) return;  // whole wavefronts
    const int m = find_mesh(off_c, M, node);
    const int N = dim[m], Nc = dim_c[m], local = node - off_c[m];
    const int K[3] = {2 * (local % Nc), 2 * ((local / Nc) % Nc), 2 * (local / (Nc * Nc))};
    const double *r = R + static_cast<int64_t>(node) * (9 * 125);
    double a[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int d = min(lane + 64 * u, 124);
        double v[9];
#pragma unroll
        for (int rc = 0; rc < 9; ++rc) v[rc] = r[rc * 125 + d];
        const int i[3] = {K[0] + d % 5 - 2, K[1] + (d / 5) % 5 - 2, K[2] + d / 25 - 2};
        const bool ok = lane + 64 * u < 125 && i[0] >= 0 && i[0] < N && i[1] >= 0 && i[1] < N && i[2] >= 0 && i[2] < N;
        const double *bj = b + 3 * static_cast<int64_t>(ok ? off[m] + i[0] + N * (i[1] + N * i[2]) : 0);
        const double b0 = ok ? bj[0] : 0.0, b1 = ok ? bj[1] : 0.0, b2 = ok ? bj[2] : 0.0;
#pragma unroll
        for (int c = 0; c < 3; ++c) a[c] += v[3 * c] * b0 + v[3 * c + 1] * b1 + v[3 * c + 2] * b2;
    }
    const double t = wave_total3(a, lane);
    if ((lane & 15) == 0 && lane < 48) bc[static_cast<int64_t>(node) * 3 + (lane >> 4)] = t;
}

// x = U b + V e: one 32-lane group per node, lanes over its 27 neighbours and
// its 8 to 27 coarse ones
__global__ void __launch_bounds__(256)
stencil_up_kernel(int nn, const MgNode *__restrict__ nodes, const double *__restrict__ U,
                  const double *__restrict__ V, const double *__restrict__ b, const double *__restrict__ e,
                  double *__restrict__ x)
{
    const int node = static_cast<int>((static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) >> 5);
    const int lane = threadIdx.x & 31;
    if (node >= nn) return;  // whole 32-lane groups
    const MgNode nd = nodes[node];
    const int N = static_cast<int>(nd.bits >> 16), Nf = 2 * N - 2 + (nd.bits >> 12 & 1);
    const int d = min(lane, 26);
    double u[9];
#pragma unroll
    for (int rc = 0; rc < 9; ++rc) u[rc] = U[(static_cast<int64_t>(node) * 9 + rc) * 27 + d];
    const bool odd[3] = {(nd.bits & 1) != 0, (nd.bits & 2) != 0, (nd.bits & 4) != 0};
    const int cx = odd[0] ? 2 : 3, cy = odd[1] ? 2 : 3, cz = odd[2] ? 2 : 3, S = cx * cy * cz;
    const int s = min(lane, S - 1);
    double v[9];
#pragma unroll
    for (int rc = 0; rc < 9; ++rc) v[rc] = V[9 * nd.first + rc * S + s];
    const int n[3] = {d % 3, (d / 3) % 3, d / 9};
    const int yz = div_count(s, cx), sz = div_count(yz, cy), k[3] = {s - cx * yz, yz - cy * sz, sz};
    bool okb = lane < 27, oke = lane < S;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        okb = okb && !(n[a] == 0 && (nd.bits >> (3 + 2 * a) & 1)) && !(n[a] == 2 && (nd.bits >> (9 + a) & 1));
        oke = oke && !(k[a] == 0 && (nd.bits >> (3 + 2 * a) & 1)) && !(k[a] == 2 && (nd.bits >> (4 + 2 * a) & 1));
    }
    const double *bj = b + 3 * static_cast<int64_t>(okb ? node + n[0] - 1 + Nf * (n[1] - 1 + Nf * (n[2] - 1)) : 0);
    const double *ek = e + 3 * static_cast<int64_t>(oke ? nd.lo + k[0] + N * (k[1] + N * k[2]) : 0);
    const double bv[3] = {okb ? bj[0] : 0.0, okb ? bj[1] : 0.0, okb ? bj[2] : 0.0};
    const double ev[3] = {oke ? ek[0] : 0.0, oke ? ek[1] : 0.0, oke ? ek[2] : 0.0};
    double p[3];
#pragma unroll
    for (int c = 0; c < 3; ++c)
        p[c] = u[3 * c] * bv[0] + u[3 * c + 1] * bv[1] + u[3 * c + 2] * bv[2] + v[3 * c] * ev[0] +
               v[3 * c + 1] * ev[1] + v[3 * c + 2] * ev[2];
#pragma unroll
    for (int sh = 16; sh > 0; sh >>= 1)
#pragma unroll
        for (int c = 0; c < 3; ++c) p[c] += __shfl_xor(p[c], sh, 32);
    if (lane < 3) x[static_cast<int64_t>(node) * 3 + lane] = lane == 0 ? p[0] : (lane == 1 ? p[1] : p[2]);
}

__global__ void __launch_bounds__(256) coarse_apply_kernel(int M, const int *__restrict__ dim,
                                                          const int *__restrict__ off, int nn,
                                                          const double *__restrict__ inv, int stride,
                                                          const double *__restrict__ b, double *__restrict__ x)
{
    // one wavefront per coarse DOF: its row of the dense inverse against b,
    // lanes over the row, a fixed butterfly for the sum
    const int k = static_cast<int>((static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) >> 6);
    const int lane = threadIdx.x & 63;
    if (k >= 3 * nn) return;  // whole wavefronts
    const int node = k / 3;
    const int m = find_mesh(off, M, node);
    const int N = dim[m], nd = 3 * N * N * N;
    const int r = k - 3 * off[m];
    const double *row = inv + static_cast<int64_t>(m) * stride + static_cast<int64_t>(r) * nd;
    const double *bm = b + static_cast<int64_t>(off[m]) * 3;
    double acc = 0.0;
    for (int j = lane; j < nd; j += 64) acc += row[j] * bm[j];
#pragma unroll
    for (int sh = 32; sh > 0; sh >>= 1) acc += __shfl_xor(acc, sh, 64);
    if (lane == 0) x[k] = acc;
}

unsigned group_grid(int nn) { return static_cast<unsigned>((static_cast<int64_t>(nn) * 32 + 255) / 256); }
unsigned grid1(int64_t n) { return static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 16384))); }

}  // namespace

// What the V-cycle of a precision needs, made before its setup is recorded;
// *made tells whether something was missing (a recorded setup then lacks it)
int mg_prepare(EquationsSet &s, int precision, bool *made)
{
    *made = false;
    if (s.node_rows != 1) return set_error(OC_ERR_UNSUPPORTED, "the multigrid preconditioner needs node rows");
    Multigrid &g = *s.mg;
    const size_t blocks = g.levels[0].up.n / 9;
    if (precision != OC_FP32) {
        *made = !g.bt.ptr;
        return g.bt.ptr ? OC_NO_ERROR : g.bt.alloc(blocks * 3);
    }
    *made = !s.uu_bf.ptr || !g.ap_sp.ptr || !g.bt_sp.ptr;
    if (!s.values_sp.ptr) OC_CHECK(s.values_sp.alloc(s.nnz));
    OC_CHECK(prepare_uu_bf16(s));
    if (!g.ap_sp.ptr) OC_CHECK(g.ap_sp.alloc(blocks * 9));
    if (!g.bt_sp.ptr) OC_CHECK(g.bt_sp.alloc(blocks * 3));
    return OC_NO_ERROR;
}

int mg_setup(EquationsSet &s, int precision, double *inv_u, double *diag_u)
{
    Multigrid &g = *s.mg;
    Runtime &rt = runtime();
    const int M = s.n_meshes;
    const int nq = s.n_nodes;
    const unsigned gp = static_cast<unsigned>((nq + kProductNodes - 1) / kProductNodes);
    MgLevel &L0 = g.levels[0], &L1 = g.levels[1];
    if (precision == OC_FP64)
        q1_product_kernel<double><<<gp, 32 * kProductNodes, 0, rt.stream>>>(
            M, g.n.ptr, s.q_off.ptr, L0.nodes.ptr, nq, s.row_ptr.ptr, s.pstart.ptr, s.col_idx.ptr, s.values.ptr,
            s.free_mask.ptr, L0.up.ptr, nullptr, g.bt.ptr, nullptr, nullptr, inv_u, diag_u);
    else
        q1_product_kernel<float><<<gp, 32 * kProductNodes, 0, rt.stream>>>(
            M, g.n.ptr, s.q_off.ptr, L0.nodes.ptr, nq, s.row_ptr.ptr, s.pstart.ptr, s.col_idx.ptr, s.values_sp.ptr,
            s.free_mask.ptr, L0.up.ptr, g.ap_sp.ptr, g.bt_sp.ptr, s.uu_off.ptr, s.uu_bf.ptr, inv_u, diag_u);
    OC_HIP_CHECK(hipGetLastError());
    coarse_stencil_kernel<<<group_grid(L1.nn), 256, 0, rt.stream>>>(M, L0.dim.ptr, L0.off.ptr, L1.dim.ptr, L1.off.ptr,
                                                                   L1.nn, L0.nodes.ptr, L0.up.ptr, L1.A.ptr);
    coincident_q2_kernel<<<grid1(L1.nn), 256, 0, rt.stream>>>(M, g.n.ptr, s.q_off.ptr, s.n_nodes, L1.off.ptr, L1.nn,
                                                              s.free_mask.ptr, L1.freed.ptr);
    level_freed_kernel<<<grid1(L1.nn), 256, 0, rt.stream>>>(L1.nn, L1.A.ptr, L1.freed.ptr);
    level_mask_kernel<<<grid1(static_cast<int64_t>(L1.nn) * 27), 256, 0, rt.stream>>>(
        M, L1.dim.ptr, L1.off.ptr, L1.nn, L1.A.ptr, L1.freed.ptr, L1.Dinv.ptr);
    OC_HIP_CHECK(hipGetLastError());
    const int nl = static_cast<int>(g.levels.size());
    for (int l = 1; l + 1 < nl; ++l) {
        MgLevel &F = g.levels[l], &C = g.levels[l + 1];
        stencil_product_kernel<<<group_grid(F.nn), 256, 0, rt.stream>>>(M, F.dim.ptr, F.off.ptr, F.nn, C.dim.ptr,
                                                                       F.nodes.ptr, F.A.ptr, F.freed.ptr, F.up.ptr);
        coarse_stencil_kernel<<<group_grid(C.nn), 256, 0, rt.stream>>>(M, F.dim.ptr, F.off.ptr, C.dim.ptr, C.off.ptr,
                                                                      C.nn, F.nodes.ptr, F.up.ptr, C.A.ptr);
        coincident_kernel<<<grid1(C.nn), 256, 0, rt.stream>>>(M, F.dim.ptr, F.off.ptr, F.freed.ptr, C.dim.ptr,
                                                             C.off.ptr, C.nn, C.freed.ptr);
        level_freed_kernel<<<grid1(C.nn), 256, 0, rt.stream>>>(C.nn, C.A.ptr, C.freed.ptr);
        level_mask_kernel<<<grid1(static_cast<int64_t>(C.nn) * 27), 256, 0, rt.stream>>>(
            M, C.dim.ptr, C.off.ptr, C.nn, C.A.ptr, C.freed.ptr, C.Dinv.ptr);
        stencil_up_setup_kernel<<<group_grid(F.nn), 256, 0, rt.stream>>>(M, F.dim.ptr, F.off.ptr, F.nn, F.nodes.ptr,
                                                                        F.A.ptr, F.freed.ptr, F.Dinv.ptr, g.omega,
                                                                        F.own.ptr, F.up.ptr);
        stencil_down_setup_kernel<<<grid1(static_cast<int64_t>(C.nn) * 125), 256, 0, rt.stream>>>(
            M, F.dim.ptr, F.off.ptr, C.dim.ptr, C.off.ptr, C.nn, F.A.ptr, F.freed.ptr, F.Dinv.ptr, C.freed.ptr,
            g.omega, F.down.ptr);
        OC_HIP_CHECK(hipGetLastError());
    }
    MgLevel &Lc = g.levels[nl - 1];
    coarse_inverse_kernel<<<static_cast<unsigned>(M), 1024, 0, rt.stream>>>(M, Lc.dim.ptr, Lc.off.ptr, Lc.A.ptr,
                                                                         g.coarse_stride, g.coarse_inv.ptr);
    if (g.dense.ptr) {
        MgLevel &F = g.levels[nl - 2];
        dense_w_kernel<<<dim3(64, M), 256, 0, rt.stream>>>(F.dim.ptr, Lc.dim.ptr, Lc.off.ptr, F.down.ptr, g.coarse_inv.ptr,
                                                           g.coarse_stride, g.dense_w_stride, g.dense_w.ptr);
        dense_kernel<<<dim3(256, M), 256, 0, rt.stream>>>(F.dim.ptr, F.off.ptr, Lc.dim.ptr, F.nodes.ptr, F.own.ptr,
                                                          F.up.ptr, g.dense_w.ptr, g.dense_w_stride, g.dense_stride,
                                                          g.dense.ptr);
    }
    OC_HIP_CHECK(hipGetLastError());
    return OC_NO_ERROR;
}


// Launch shapes of the level-0 node kernels: lanes per node (below) x
// neighbours per lane in flight (1, 2, 2, 4, 1; the cases of launch_uu_node);
// the autotuner may pick one (LaunchShapes::smoother).
constexpr int kNodeVariants = 5;
constexpr int kNodeVariantLanes[kNodeVariants] = {32, 32, 16, 16, 64};

template <typename VT, int kSweep>
static int launch_uu_node(int variant, int nq, const EquationsSet &s, const VT *vals, const double *b,
                          const double *x, const double *inv_u, double omega, const double *scale, double *out)
{
    Runtime &rt = runtime();
    // one wavefront per node for FP64 values where the rows fit
    if (variant < 0 || variant >= kNodeVariants) variant = sizeof(VT) == sizeof(double) ? 4 : 0;
    if (variant == 4 && !s.flat_rows()) variant = 0;
    const unsigned grid =
        static_cast<unsigned>((static_cast<int64_t>(nq) * kNodeVariantLanes[variant] + 255) / 256);
#define OC_UU_NODE(L, U)                                                                                       \
    uu_node_residual_kernel<VT, L, kSweep, U><<<grid, 256, 0, rt.stream>>>(nq, s.row_ptr.ptr, s.pstart.ptr,   \
                                                                         s.col_idx.ptr, vals, s.free_mask.ptr, \
                                                                         b, x, inv_u, omega, scale, out)
    switch (variant) {
    case 1: OC_UU_NODE(32, 2); break;
    case 2: OC_UU_NODE(16, 2); break;
    case 3: OC_UU_NODE(16, 4); break;
    case 4:
        uu_flat_kernel<VT, kSweep><<<grid, 256, 0, rt.stream>>>(nq, s.row_ptr.ptr, s.pstart.ptr, s.col_idx.ptr, vals,
                                                               s.free_mask.ptr, b, x, inv_u, omega, scale, out);
        break;
    default: OC_UU_NODE(32, 1); break;
    }
#undef OC_UU_NODE
    OC_HIP_CHECK(hipGetLastError());
    return OC_NO_ERROR;
}

// The packed bf16 level-0 kernels' shapes: lanes per node x quads of
// neighbours per lane in flight (variants as kNodeVariants).
constexpr int kBf16VariantLanes[kNodeVariants] = {16, 8, 32, 8, 16};

template <int kSweep>
// x4: the FP32 node quadruples of x when the caller has them (nullptr: packed
// here, into the first of the set's two quadruple buffers); out4: where a
// sweep also writes its result's quadruples (nullptr: not written)
static int launch_uu_bf16(int variant, const EquationsSet &s, const double *b, const double *x, const double *inv_u,
                          double omega, const double *scale, double *out, const float *x4_in = nullptr,
                          float *out4 = nullptr)
{
    Runtime &rt = runtime();
    if (variant < 0 || variant >= kNodeVariants) variant = 0;
    const int nq = s.n_nodes;
    const unsigned grid = static_cast<unsigned>((static_cast<int64_t>(nq) * kBf16VariantLanes[variant] + 255) / 256);
    const float4 *x4 = reinterpret_cast<const float4 *>(x4_in);
    if (!x4) {
        pack_x4(nq, x, reinterpret_cast<float4 *>(s.uu_x4.ptr));
        x4 = reinterpret_cast<const float4 *>(s.uu_x4.ptr);
    }
#define OC_UU_BF16(L, Q)                                                                                          \
    uu_node_bf16_kernel<L, kSweep, Q><<<grid, 256, 0, rt.stream>>>(nq, s.uu_off.ptr, s.uu_col.ptr, s.uu_bf.ptr, \
                                                                 s.free_mask.ptr, b, x4, x, inv_u, omega, scale, \
                                                                 out, out4)
    switch (variant) {
    case 1: OC_UU_BF16(8, 1); break;
    case 2: OC_UU_BF16(32, 1); break;
    case 3: OC_UU_BF16(8, 2); break;
    case 4: OC_UU_BF16(16, 2); break;
    default: OC_UU_BF16(16, 1); break;
    }
#undef OC_UU_BF16
    OC_HIP_CHECK(hipGetLastError());
    return OC_NO_ERROR;
}

void pack_x4(int nq, const double *x, float4 *x4)
{
    pack_x4_kernel<<<static_cast<unsigned>((nq + 255) / 256), 256, 0, runtime().stream>>>(nq, x, x4);
}

int launch_uu_pack(EquationsSet &s)
{
    uu_pack_kernel<<<static_cast<unsigned>((static_cast<int64_t>(s.n_nodes) * kPackLanes + 255) / 256), 256, 0,
                     runtime().stream>>>(s.n_nodes, s.row_ptr.ptr, s.pstart.ptr, s.values_sp.ptr, s.uu_off.ptr,
                                         s.uu_bf.ptr);
    OC_HIP_CHECK(hipGetLastError());
    return OC_NO_ERROR;
}

int prepare_uu_bf16(EquationsSet &s)
{
    if (s.uu_bf.ptr) return OC_NO_ERROR;
    if (s.node_rows != 1 || !s.pstart.ptr) return set_error(OC_ERR_UNSUPPORTED, "the packed bf16 block needs node rows");
    Runtime &rt = runtime();
    const int nq = s.n_nodes;
    DevBuf<int64_t> degp;
    OC_CHECK(degp.alloc(nq));
    uu_degp_kernel<<<static_cast<unsigned>((nq + 255) / 256), 256, 0, rt.stream>>>(nq, s.row_ptr.ptr, s.pstart.ptr,
                                                                                   degp.ptr);
    OC_HIP_CHECK(hipGetLastError());
    std::vector<int64_t> off(static_cast<size_t>(nq) + 1, 0);
    OC_HIP_CHECK(hipMemcpyAsync(off.data() + 1, degp.ptr, sizeof(int64_t) * nq, hipMemcpyDeviceToHost, rt.stream));
    OC_HIP_CHECK(hipStreamSynchronize(rt.stream));
    for (int i = 0; i < nq; ++i) off[i + 1] += off[i];
    const int64_t total = off[nq];
    OC_CHECK(s.uu_off.upload(off.data(), off.size()));
    OC_CHECK(s.uu_col.alloc(static_cast<size_t>(total)));
    OC_CHECK(s.uu_bf.alloc(static_cast<size_t>(total) * 9));
    OC_CHECK(s.uu_x4.alloc(static_cast<size_t>(nq) * 8));  // two quadruple buffers
    uu_cols_kernel<<<static_cast<unsigned>((static_cast<int64_t>(nq) * kPackLanes + 255) / 256), 256, 0, rt.stream>>>(
        nq, s.row_ptr.ptr, s.pstart.ptr, s.col_idx.ptr, s.uu_off.ptr, s.uu_col.ptr);
    OC_HIP_CHECK(hipGetLastError());
    OC_HIP_CHECK(hipStreamSynchronize(rt.stream));
    return OC_NO_ERROR;
}

int launch_smoother_residual(EquationsSet &s, int precision, int variant, const double *b, const double *x,
                             double *r)
{
    if (s.node_rows != 1) return set_error(OC_ERR_UNSUPPORTED, "the node-wise smoother needs node rows");
    // every array the kernel reads must exist: the free-DOF mask only does once
    // boundary conditions are set or a solve has prepared the set
    const void *vals = precision == OC_FP32 ? (s.uu_bf.ptr ? static_cast<const void *>(s.uu_bf.ptr)
                                                           : static_cast<const void *>(s.values_sp.ptr))
                                            : static_cast<const void *>(s.values.ptr);
    if (!s.free_mask.ptr || !s.pstart.ptr || !vals || !b || !x || !r)
        return set_error(OC_ERR_INVALID_ARGUMENT, "smoother residual: free-DOF mask, pressure starts or values missing");
    if (precision == OC_FP32 && s.uu_bf.ptr) return launch_uu_bf16<0>(variant, s, b, x, nullptr, 0.0, nullptr, r);
    if (precision == OC_FP32) return launch_uu_node<float, 0>(variant, s.n_nodes, s, s.values_sp.ptr, b, x, nullptr, 0.0,
                                                                     nullptr, r);
    return launch_uu_node<double, 0>(variant, s.n_nodes, s, s.values.ptr, b, x, nullptr, 0.0, nullptr, r);
}

// z = scale .* (P^-1 r): z_p = inv_p .* r_p and the displacement part, component-
// major, the V-cycle applied to r_u - B^T z_p
int mg_apply(EquationsSet &s, int precision, const double *r, const double *inv_p, const double *scale, double *z)
{
    Multigrid &g = *s.mg;
    Runtime &rt = runtime();
    const int M = s.n_meshes, nq = s.n_nodes, nl = static_cast<int>(g.levels.size());
    const double *inv_u = s.precond.ptr;  // nodal block inverses of the set's block preconditioner
    const bool bf = precision == OC_FP32;  // an FP32 Jacobian's packed bf16 values (mg_prepare)
    const int variant = s.tuned[precision].smoother;  // -1: a wavefront per node for FP64 values, 16 lanes x one quad for bf16
    // with the packed bf16 values the kernels that produce the iterate also
    // write its FP32 node quadruples, into the two halves of uu_x4 in turn
    // (a sweep gathers one half and writes the other); q4 is the current one
    float *q4 = bf ? s.uu_x4.ptr : nullptr, *q4_other = bf ? s.uu_x4.ptr + 4 * static_cast<int64_t>(nq) : nullptr;
    // level 0 pre-smoothing from x = 0.  A sweep is one kernel writing the
    // other of z and x0; the first Jacobi step picks the buffer that leaves
    // the last post-smoothing sweep in z.  The first post-smoothing sweep
    // comes with the coarse correction, in place.
    const int post = g.post;
    double *t = g.t0.ptr, *cur = z, *other = g.x0.ptr;
    if ((std::max(g.pre - 1, 0) + std::max(post - 1, 0)) & 1) std::swap(cur, other);
    auto sweep0 = [&](const double *sc) -> int {
        if (bf)
            OC_CHECK(launch_uu_bf16<1>(variant, s, t, cur, inv_u, g.omega, sc, other, q4, q4_other));
        else
            OC_CHECK((launch_uu_node<double, 1>(variant, nq, s, s.values.ptr, t, cur, inv_u, g.omega, sc, other)));
        std::swap(cur, other);
        std::swap(q4, q4_other);
        return OC_NO_ERROR;
    };
    MgLevel &L0 = g.levels[0], &L1 = g.levels[1];
    const unsigned gc = static_cast<unsigned>((static_cast<int64_t>(nq) * 8 + 255) / 256);
    if (bf)
        mg_start_kernel<float><<<gc, 256, 0, rt.stream>>>(nq, s.n_nodes_l, L0.nodes.ptr, g.bt_sp.ptr, inv_p, r, scale,
                                                          s.free_mask.ptr, inv_u, g.omega, z, t, cur, q4);
    else
        mg_start_kernel<double><<<gc, 256, 0, rt.stream>>>(nq, s.n_nodes_l, L0.nodes.ptr, g.bt.ptr, inv_p, r, scale,
                                                           s.free_mask.ptr, inv_u, g.omega, z, t, cur, nullptr);
    OC_HIP_CHECK(hipGetLastError());
    for (int k = 1; k < g.pre; ++k) OC_CHECK(sweep0(nullptr));
    if (bf)
        OC_CHECK(launch_uu_bf16<0>(variant, s, t, cur, nullptr, 0.0, nullptr, g.r0.ptr, q4));
    else
        OC_CHECK((launch_uu_node<double, 0>(variant, nq, s, s.values.ptr, t, cur, nullptr, 0.0, nullptr, g.r0.ptr)));
    restrict_q2_kernel<<<group_grid(L1.nn), 256, 0, rt.stream>>>(M, g.n.ptr, s.q_off.ptr, nq, L1.off.ptr, L1.nn,
                                                            L1.freed.ptr, g.r0.ptr, L1.b.ptr);
    OC_HIP_CHECK(hipGetLastError());
    // down the stencil levels, to the last or with the dense matrix the last but one
    const int bottom = nl - (g.dense.ptr ? 2 : 1);
    for (int l = 1; l < bottom; ++l) {
        MgLevel &F = g.levels[l], &C = g.levels[l + 1];
        stencil_down_kernel<<<static_cast<unsigned>((C.nn + 3) / 4), 256, 0, rt.stream>>>(
            M, F.dim.ptr, F.off.ptr, C.dim.ptr, C.off.ptr, C.nn, F.down.ptr, F.b.ptr, C.b.ptr);
        OC_HIP_CHECK(hipGetLastError());
    }
    MgLevel &Lc = g.levels[bottom];
    coarse_apply_kernel<<<static_cast<unsigned>((3 * static_cast<int64_t>(Lc.nn) * 64 + 255) / 256), 256, 0, rt.stream>>>(
        M, Lc.dim.ptr, Lc.off.ptr, Lc.nn, g.dense.ptr ? g.dense.ptr : g.coarse_inv.ptr,
        g.dense.ptr ? g.dense_stride : g.coarse_stride, Lc.b.ptr, Lc.x.ptr);
    OC_HIP_CHECK(hipGetLastError());
    // up
    for (int l = bottom - 1; l >= 1; --l) {
        MgLevel &F = g.levels[l], &C = g.levels[l + 1];
        stencil_up_kernel<<<group_grid(F.nn), 256, 0, rt.stream>>>(F.nn, F.nodes.ptr, F.own.ptr, F.up.ptr, F.b.ptr,
                                                                  C.x.ptr, F.x.ptr);
        OC_HIP_CHECK(hipGetLastError());
    }
    const double omega1 = post > 0 ? g.omega : 0.0;  // without post-smoothing only x + P0 e
    const double *sc = post > 1 ? nullptr : scale;   // the last step scales z
    if (bf)
        q1_correct_kernel<float><<<gc, 256, 0, rt.stream>>>(nq, L0.nodes.ptr, g.ap_sp.ptr, L1.x.ptr, s.free_mask.ptr,
                                                            g.r0.ptr, inv_u, omega1, sc, cur, q4);
    else
        q1_correct_kernel<double><<<gc, 256, 0, rt.stream>>>(nq, L0.nodes.ptr, L0.up.ptr, L1.x.ptr, s.free_mask.ptr,
                                                             g.r0.ptr, inv_u, omega1, sc, cur, nullptr);
    OC_HIP_CHECK(hipGetLastError());
    for (int k = 1; k < post; ++k) OC_CHECK(sweep0(k + 1 == post ? scale : nullptr));
    return OC_NO_ERROR;
}

}  // namespace oc

using namespace oc;

extern "C" int oc_multigrid_structure_set(oc_equations_set h, const int *n_per_mesh)
{
    OC_CHECK(require_runtime());
    if (!h) return set_error(OC_ERR_INVALID_HANDLE, "equations set handle is NULL");
    EquationsSet &s = h->s;
    if (s.cls != OC_EQUATIONS_SET_MOONEY_RIVLIN || !n_per_mesh)
        return set_error(OC_ERR_INVALID_ARGUMENT, "multigrid structure: a Mooney-Rivlin set and n per mesh");
    const int M = s.n_meshes;
    // the connectivity must be that of regular generated n^3 meshes
    std::vector<int32_t> cq(static_cast<size_t>(s.n_elements) * 27), cl(static_cast<size_t>(s.n_elements) * 8);
    OC_HIP_CHECK(hipMemcpy(cq.data(), s.conn.ptr, cq.size() * sizeof(int32_t), hipMemcpyDeviceToHost));
    OC_HIP_CHECK(hipMemcpy(cl.data(), s.conn_l.ptr, cl.size() * sizeof(int32_t), hipMemcpyDeviceToHost));
    for (int m = 0; m < M; ++m) {
        const int64_t n = n_per_mesh[m];
        const int64_t T = 2 * n + 1, N = n + 1;
        if (n < 1 || n * n * n != s.h_e_off[m + 1] - s.h_e_off[m] || T * T * T != s.h_q_off[m + 1] - s.h_q_off[m] ||
            N * N * N != s.h_l_off[m + 1] - s.h_l_off[m])
            return set_error(OC_ERR_INVALID_ARGUMENT, "mesh %d is not a regular mesh of %lld^3 elements", m,
                             static_cast<long long>(n));
        for (int64_t e = 0; e < n * n * n; ++e) {
            const int64_t ex = e % n, ey = (e / n) % n, ez = e / (n * n);
            const int64_t ge = s.h_e_off[m] + e;
            for (int a = 0; a < 27; ++a) {
                const int64_t q = s.h_q_off[m] + (2 * ex + a % 3) + T * ((2 * ey + (a / 3) % 3) + T * (2 * ez + a / 9));
                if (cq[ge * 27 + a] != q)
                    return set_error(OC_ERR_INVALID_ARGUMENT, "mesh %d element %lld: not the regular node numbering",
                                     m, static_cast<long long>(e));
            }
            for (int k = 0; k < 8; ++k) {
                const int64_t p = s.h_l_off[m] + (ex + (k & 1)) + N * ((ey + ((k >> 1) & 1)) + N * (ez + (k >> 2)));
                if (cl[ge * 8 + k] != p)
                    return set_error(OC_ERR_INVALID_ARGUMENT, "mesh %d element %lld: not the regular pressure numbering",
                                     m, static_cast<long long>(e));
            }
        }
    }
    auto g = new (std::nothrow) Multigrid();
    if (!g) return set_error(OC_ERR_ALLOCATION, "out of host memory");
    std::unique_ptr<Multigrid> guard(g);
    g->h_n.assign(n_per_mesh, n_per_mesh + M);
    OC_CHECK(g->n.upload(g->h_n.data(), M));
    // levels: [0] the triquadratic lattice (tables and A P0 only), [1] trilinear
    // (n+1)^3, then coarsening until every dim <= 3
    g->levels.resize(2);
    std::vector<int32_t> dims(M);
    const auto tables = [&](MgLevel &L) -> int {
        L.h_dim = dims;
        L.h_off.assign(M + 1, 0);
        for (int m = 0; m < M; ++m) L.h_off[m + 1] = L.h_off[m] + dims[m] * dims[m] * dims[m];
        L.nn = L.h_off[M];
        OC_CHECK(L.dim.upload(L.h_dim.data(), M));
        return L.off.upload(L.h_off.data(), M + 1);
    };
    for (int m = 0; m < M; ++m) dims[m] = 2 * g->h_n[m] + 1;
    OC_CHECK(tables(g->levels[0]));
    for (int m = 0; m < M; ++m) dims[m] = g->h_n[m] + 1;
    while (true) {
        MgLevel &L = g->levels.back();
        OC_CHECK(tables(L));
        OC_CHECK(L.A.alloc(static_cast<size_t>(L.nn) * 27 * 9));
        OC_CHECK(L.Dinv.alloc(static_cast<size_t>(L.nn) * 9));
        OC_CHECK(L.freed.alloc(static_cast<size_t>(L.nn) * 3));
        OC_CHECK(L.x.alloc(static_cast<size_t>(L.nn) * 3));
        OC_CHECK(L.b.alloc(static_cast<size_t>(L.nn) * 3));
        if (*std::max_element(dims.begin(), dims.end()) <= 3) break;
        for (int m = 0; m < M; ++m) dims[m] = (dims[m] - 1 + 1) / 2 + 1;  // n -> ceil(n/2)
        g->levels.emplace_back();
    }
    for (size_t l = 0; l + 1 < g->levels.size(); ++l) {
        MgLevel &F = g->levels[l], &C = g->levels[l + 1];
        std::vector<int64_t> first(static_cast<size_t>(M) + 1, 0);
        for (int m = 0; m < M; ++m) {
            const int64_t X = product_before(F.h_dim[m]);
            first[m + 1] = first[m] + X * X * X;
        }
        DevBuf<int64_t> first_d;
        OC_CHECK(first_d.upload(first.data(), first.size()));
        OC_CHECK(F.up.alloc(static_cast<size_t>(first[M]) * 9));
        OC_CHECK(F.nodes.alloc(F.nn));
        mg_nodes_kernel<<<static_cast<unsigned>((F.nn + 255) / 256), 256, 0, runtime().stream>>>(
            M, F.dim.ptr, F.off.ptr, C.dim.ptr, C.off.ptr, first_d.ptr, F.nn, F.nodes.ptr);
        OC_HIP_CHECK(hipGetLastError());
        OC_HIP_CHECK(hipStreamSynchronize(runtime().stream));  // first_d is read
        if (l == 0) continue;
        OC_CHECK(F.own.alloc(static_cast<size_t>(F.nn) * 27 * 9));
        OC_CHECK(F.down.alloc(static_cast<size_t>(C.nn) * 125 * 9));
    }
    int maxnd = 0;
    for (int m = 0; m < M; ++m) maxnd = std::max(maxnd, 3 * dims[m] * dims[m] * dims[m]);
    if (maxnd > 81) return set_error(OC_ERR_UNSUPPORTED, "coarsest multigrid level too large");
    g->coarse_stride = maxnd * maxnd;
    OC_CHECK(g->coarse_inv.alloc(static_cast<size_t>(M) * g->coarse_stride));
    // the dense matrix of the last two levels: 1.1 MB a mesh and product, so for a
    // few meshes only; of many, the stencils of those levels move fewer bytes
    constexpr int kDenseMeshes = 16;
    if (g->levels.size() >= 3 && M <= kDenseMeshes) {
        const std::vector<int32_t> &d = g->levels[g->levels.size() - 2].h_dim;
        const int n = *std::max_element(d.begin(), d.end()), nd = 3 * n * n * n;
        g->dense_stride = nd * nd;
        g->dense_w_stride = maxnd * nd;
        OC_CHECK(g->dense.alloc(static_cast<size_t>(M) * g->dense_stride));
        OC_CHECK(g->dense_w.alloc(static_cast<size_t>(M) * g->dense_w_stride));
    }
    OC_CHECK(g->r0.alloc(static_cast<size_t>(3) * s.n_nodes));
    OC_CHECK(g->t0.alloc(static_cast<size_t>(3) * s.n_nodes));
    OC_CHECK(g->x0.alloc(static_cast<size_t>(3) * s.n_nodes));
    delete s.mg;
    s.mg = guard.release();
    if (s.step_graph) {  // recorded without the multigrid setup
        (void)hipGraphExecDestroy(s.step_graph);
        s.step_graph = nullptr;
    }
    return OC_NO_ERROR;
}

extern "C" int oc_multigrid_options_set(oc_equations_set h, int pre_sweeps, int post_sweeps, double omega)
{
    OC_CHECK(require_runtime());
    if (!h) return set_error(OC_ERR_INVALID_HANDLE, "equations set handle is NULL");
    if (!h->s.mg) return set_error(OC_ERR_INVALID_ARGUMENT, "no multigrid structure (oc_multigrid_structure_set)");
    if (pre_sweeps < 1 || post_sweeps < 0 || !(omega > 0.0 && omega < 2.0))
        return set_error(OC_ERR_INVALID_ARGUMENT, "multigrid options: pre >= 1, post >= 0, 0 < omega < 2");
    h->s.mg->pre = pre_sweeps;
    h->s.mg->post = post_sweeps;
    h->s.mg->omega = omega;
    if (h->s.step_graph) {  // its multigrid setup holds the former omega
        (void)hipGraphExecDestroy(h->s.step_graph);
        h->s.step_graph = nullptr;
    }
    return OC_NO_ERROR;
}
