// demag.hip -- zero-padded demag convolution on gfx950.
//
// B = mu0 Ms0T0Mul * IFFT( K^ . FFT(m .* msat0T0) ), the algorithm of
// MaxwellPlan.UpdateB (src/hotspin-core/modules/maxwell_convolution.go:103-131)
// with the reference's cuFFT 3-D D2Z/Z2D replaced by five pruned passes of
// the library's own LDS-staged FFT (fft.hpp), or by three kernels where the
// columns fit in LDS (demag_fused.hpp: open meshes of up to 32 planes).  Mesh
// N=(N0,N1,N2) internal, transform lengths P >= the logic size (x2 on open
// axes, zeropad.go:12-22; set_lengths), M = P2/2, H2 = M+1.  The five passes:
//   F1  rows, R2C along axis 2 (M-point complex FFT + split), only the N0*N1
//       non-zero rows are read: m (3N)         -> X1 (3, N0, N1, H2)
//   F2  columns along axis 1, input rows j < N1:  X1 -> X2 (3, N0, P1, H2)
//   F3K columns along axis 0 for all 3 components, the symmetric kernel
//       product (tensSYMMVecMul, src/libhotspin/mul.cu:31-90) and the inverse
//       along axis 0, keeping rows i < N0:          X2 -> X2 (in place)
//   I2  inverse along axis 1, keeping j < N1:       X2 -> X1
//   I1  C2R along axis 2, keeping k < N2:           X1 -> B (3N)
// The kernel K^ is Kernel_Arne (kernel_magnetostatic.go:25-241) integrated
// on the GPU in FP64 (one lane per destination cell and source direction, a
// block for the cells next to the source; same operation order as the Go
// code, no FMA contraction), transformed in
// FP64 by the same passes, its real first octant kept and scaled by
// 1/(P0 P1 P2) (maxwell_convolution.go:135-223,350-388).
#include <math.h>
#include <stdio.h>

#include <array>
#include <string.h>

#include <map>
#include <memory>
#include <mutex>
#include <vector>

#include "hostcopy.hpp"
#include "hs_common.hpp"

#define HS_PI_D 3.141592653589793

#include "demag_kernels.hpp"
#include "demag_tune.hpp"
#include "demag_fused.hpp"
#include "fft_any.hpp"

// Kernels by length.  Written by the static constructors of the files that
// compile them and only read afterwards: a look-up of another length finds an
// empty entry and adds none, so threads may look up side by side.
namespace {
template <typename V>
std::map<int, V>& registry() {
    static std::map<int, V> reg;
    return reg;
}
template <typename V>
const V& find_in_registry(int L) {
    static const V none{};
    const auto it = registry<V>().find(L);
    return it == registry<V>().end() ? none : it->second;
}
}  // namespace

hsdm::Variants& hsdm::add_variants(int L) { return registry<hsdm::Variants>()[L]; }
const hsdm::Variants& hsdm::variants(int L) { return find_in_registry<hsdm::Variants>(L); }

namespace fused {
template <typename T>
Rows<T>& add_rows_of(int M) { return registry<Rows<T>>()[M]; }
template <typename T>
Mids<T>& add_mids_of(int Q) { return registry<Mids<T>>()[Q]; }
template <typename T>
const Rows<T>& rows_of(int M) { return find_in_registry<Rows<T>>(M); }
template <typename T>
const Mids<T>& mids_of(int Q) { return find_in_registry<Mids<T>>(Q); }
template Rows<float>& add_rows_of<float>(int);
template Rows<double>& add_rows_of<double>(int);
template Mids<float>& add_mids_of<float>(int);
template Mids<double>& add_mids_of<double>(int);
}  // namespace fused

extern "C" int hs_demag_registered(void) {
    return (int)(registry<hsdm::Variants>().size() + registry<fused::Rows<float>>().size() +
                 registry<fused::Rows<double>>().size() + registry<fused::Mids<float>>().size() +
                 registry<fused::Mids<double>>().size());
}

// ------------------------------------------------------------------ Kernel_Arne (FP64)
// The field of the charged faces of the source cell (direction s), averaged
// over the destination cell (xw,yw,zw) of the computed octant; images of a
// periodic axis are visited in the reference's loop order (z outer, then y,
// then x), kernel_magnetostatic.go:74-183.
__device__ __forceinline__ double delta_d(int d) {
    d = d < 0 ? -d : d;
    if (d > 0) d -= 1;
    return (double)d;
}
__device__ __forceinline__ int first_image(int w, int size, int r1) {
    // smallest v >= r1 with v = w (mod size)
    int q = (r1 - w);
    int k = (q >= 0) ? (q + size - 1) / size : -((-q) / size);
    return w + k * size;
}
// Integration points of one image at cell displacement (x, y, z): source
// points (nv, nw) on each charged face, destination points (nx, ny, nz).
struct ArnePts {
    int nv, nw, nx, ny, nz;
    __device__ __forceinline__ long count() const { return (long)nv * nw * nx * ny * nz; }
};
__device__ __forceinline__ ArnePts arne_points(const double cs[3], int v, int w, int x, int y, int z,
                                               double accuracy) {
#pragma clang fp contract(off)
    double L = cs[0];
    if (cs[1] < L) L = cs[1];
    if (cs[2] < L) L = cs[2];
    double dx = delta_d(x) * cs[0], dy = delta_d(y) * cs[1], dz = delta_d(z) * cs[2];
    double d = sqrt(dx * dx + dy * dy + dz * dz);
    if (d == 0) d = L;
    double maxSize = d / accuracy;
    ArnePts n;
    n.nv = 2 * (int)(fmax(cs[v] / maxSize, 1.0) + 0.5);
    n.nw = 2 * (int)(fmax(cs[w] / maxSize, 1.0) + 0.5);
    n.nx = (int)(fmax(cs[0] / maxSize, 1.0) + 0.5);
    n.ny = (int)(fmax(cs[1] / maxSize, 1.0) + 0.5);
    n.nz = (int)(fmax(cs[2] / maxSize, 1.0) + 0.5);
    return n;
}
// Both faces' charge at source point (i, j) seen at destination point (aa, bb, gg).
__device__ __forceinline__ void arne_point(const double cs[3], int u, int v, int w, const double R[3],
                                           const ArnePts& n, double charge, int i, int j, int aa, int bb, int gg,
                                           double B[3]) {
#pragma clang fp contract(off)
    double pole[3];
    pole[v] = -(cs[v] / 2.) + cs[v] / (double)(2 * n.nv) + (double)i * (cs[v] / (double)n.nv);
    pole[w] = -(cs[w] / 2.) + cs[w] / (double)(2 * n.nw) + (double)j * (cs[w] / (double)n.nw);
    const double rx = R[0] - cs[0] / 2 + cs[0] / (double)(2 * n.nx) + (cs[0] / (double)n.nx) * (double)aa;
    const double ry = R[1] - cs[1] / 2 + cs[1] / (double)(2 * n.ny) + (cs[1] / (double)n.ny) * (double)bb;
    const double rz = R[2] - cs[2] / 2 + cs[2] / (double)(2 * n.nz) + (cs[2] / (double)n.nz) * (double)gg;
    pole[u] = cs[u] / 2.;
    double q0 = rx - pole[0], q1 = ry - pole[1], q2 = rz - pole[2];
    double r = sqrt(q0 * q0 + q1 * q1 + q2 * q2);
    double qr = charge / (4 * HS_PI_D * r * r * r);
    const double bx = q0 * qr, by = q1 * qr, bz = q2 * qr;
    pole[u] = -(cs[u] / 2.);
    q0 = rx - pole[0];
    q1 = ry - pole[1];
    q2 = rz - pole[2];
    r = sqrt(q0 * q0 + q1 * q1 + q2 * q2);
    qr = -charge / (4 * HS_PI_D * r * r * r);
    B[0] = bx + q0 * qr;
    B[1] = by + q1 * qr;
    B[2] = bz + q2 * qr;
}
struct ArneP {
    int s0, s1, s2, r10, r11, r12, r20, r21, r22;
    double c0, c1, c2, accuracy;
};
// An image with more points than this is left to k_kernel_arne_near.
constexpr long kArneLight = 64;
// FullTensorIdx (common/index.go:44-47): XX=0 YY=1 ZZ=2 YZ=3 XZ=4 XY=5
__device__ __forceinline__ int tensor_idx(int a, int b) {
    const int idx[3][3] = {{0, 5, 4}, {5, 1, 3}, {4, 3, 2}};
    return idx[a][b];
}

// Lane (s, cell): its images one after the other while all have few points; a
// lane that meets one of many puts itself on the list `near` (nnear entries)
// and leaves its value to k_kernel_arne_near.
__global__ void __launch_bounds__(64) k_kernel_arne(double* __restrict__ oct, ArneP p, unsigned* __restrict__ near,
                                                    unsigned* __restrict__ nnear) {
#pragma clang fp contract(off)
    const int h0 = p.s0 / 2 + 1, h1 = p.s1 / 2 + 1, h2 = p.s2 / 2 + 1;
    const long noct = (long)h0 * h1 * h2;
    long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= 3 * noct) return;
    const int s = (int)(g / noct);
    long I = g % noct;
    const int zw = (int)(I % h2);
    const int yw = (int)((I / h2) % h1);
    const int xw = (int)(I / ((long)h1 * h2));
    const double cs[3] = {p.c0, p.c1, p.c2};
    const int u = s, v = (s + 1) % 3, w = (s + 2) % 3;
    double acc[3] = {0, 0, 0};
    bool many = false;
    for (int z = first_image(zw, p.s2, p.r12); z <= p.r22; z += p.s2)
        for (int y = first_image(yw, p.s1, p.r11); y <= p.r21; y += p.s1)
            for (int x = first_image(xw, p.s0, p.r10); x <= p.r20; x += p.s0) {
                const ArnePts n = arne_points(cs, v, w, x, y, z, p.accuracy);
                if (n.count() > kArneLight || many) {
                    many = true;
                    continue;
                }
                const double R[3] = {(double)x * p.c0, (double)y * p.c1, (double)z * p.c2};
                const double charge = cs[v] * cs[w] * (1 / (double)n.count());
                double B[3] = {0, 0, 0};
                for (int i = 0; i < n.nv; i++)
                    for (int j = 0; j < n.nw; j++)
                        for (int aa = 0; aa < n.nx; aa++)
                            for (int bb = 0; bb < n.ny; bb++)
                                for (int gg = 0; gg < n.nz; gg++) {
                                    double o[3];
                                    arne_point(cs, u, v, w, R, n, charge, i, j, aa, bb, gg, o);
                                    B[0] += o[0];
                                    B[1] += o[1];
                                    B[2] += o[2];
                                }
                for (int dd = s; dd < 3; dd++) acc[dd] += B[dd];
            }
    if (!many)
        for (int dd = s; dd < 3; dd++) oct[tensor_idx(s, dd) * noct + I] = acc[dd];
    if (many) near[atomicAdd(nnear, 1u)] = (unsigned)g;
}

// Block per list entry, all its images in order.  The cells next to the
// source take up to 10^6 points (24 x 24 x 12 x 12 x 6 for a 4 x 4 x 2 nm
// cell), whose square roots and divisions in one lane set the time of the
// whole plan (159 ms of 174 ms at 256x256x8).  Seven waves evaluate the
// points of one chunk while three lanes of the first wave, one per field
// component, add up the chunk before it in the order of the loops, so the
// sums round as in one lane; what is left is the chain of additions (2.8 ms).
constexpr int kNearThreads = 512, kNearChunk = kNearThreads - 64;
__global__ void __launch_bounds__(kNearThreads) k_kernel_arne_near(double* __restrict__ oct, ArneP p,
                                                                   const unsigned* __restrict__ near,
                                                                   const unsigned* __restrict__ nnear) {
#pragma clang fp contract(off)
    __shared__ double val[2][3][kNearChunk];
    const int h0 = p.s0 / 2 + 1, h1 = p.s1 / 2 + 1, h2 = p.s2 / 2 + 1;
    const long noct = (long)h0 * h1 * h2;
    const double cs[3] = {p.c0, p.c1, p.c2};
    const unsigned cnt = *nnear;
    const int tid = threadIdx.x;
    for (unsigned k = blockIdx.x; k < cnt; k += gridDim.x) {
        const long g = near[k];
        const int s = (int)(g / noct);
        const long I = g % noct;
        const int zw = (int)(I % h2);
        const int yw = (int)((I / h2) % h1);
        const int xw = (int)(I / ((long)h1 * h2));
        const int u = s, v = (s + 1) % 3, w = (s + 2) % 3;
        double acc = 0;  // lane dd < 3: component dd
        for (int z = first_image(zw, p.s2, p.r12); z <= p.r22; z += p.s2)
            for (int y = first_image(yw, p.s1, p.r11); y <= p.r21; y += p.s1)
                for (int x = first_image(xw, p.s0, p.r10); x <= p.r20; x += p.s0) {
                    const ArnePts n = arne_points(cs, v, w, x, y, z, p.accuracy);
                    const long cn = n.count();
                    const double R[3] = {(double)x * p.c0, (double)y * p.c1, (double)z * p.c2};
                    const double charge = cs[v] * cs[w] * (1 / (double)cn);
                    double B = 0;
                    // chunk c is evaluated in turn c and added in turn c + 1
                    const long nch = (cn + kNearChunk - 1) / kNearChunk;
                    for (long c = 0; c <= nch; c++) {
                        if (tid >= 64) {
                            const long t = c * kNearChunk + tid - 64;
                            if (c < nch && t < cn) {
                                long q = t;
                                const int gg = (int)(q % n.nz);
                                q /= n.nz;
                                const int bb = (int)(q % n.ny);
                                q /= n.ny;
                                const int aa = (int)(q % n.nx);
                                q /= n.nx;
                                double o[3];
                                arne_point(cs, u, v, w, R, n, charge, (int)(q / n.nw), (int)(q % n.nw), aa, bb, gg,
                                           o);
                                for (int dd = 0; dd < 3; dd++) val[c & 1][dd][tid - 64] = o[dd];
                            }
                        } else if (tid < 3 && c > 0) {
                            const double* o = val[(c - 1) & 1][tid];
                            const int m = (int)(cn - (c - 1) * kNearChunk < kNearChunk ? cn - (c - 1) * kNearChunk
                                                                                       : kNearChunk);
                            int q = 0;
                            for (; q + 16 <= m; q += 16) {  // sixteen reads in flight, then the chain
                                double r[16];
#pragma unroll
                                for (int e = 0; e < 16; e++) r[e] = o[q + e];
#pragma unroll
                                for (int e = 0; e < 16; e++) B += r[e];
                            }
                            for (; q < m; q++) B += o[q];
                        }
                        __syncthreads();
                    }
                    acc += B;
                }
        if (tid < 3 && tid >= s) oct[tensor_idx(s, tid) * noct + I] = acc;
    }
}

// Newell demag tensor (A. J. Newell, W. Williams, D. J. Dunlop, J. Geophys.
// Res. 98 (1993) 9551; no counterpart in the reference): N_xx of two
// uniformly magnetised cuboids is the 27-point second difference of f over
// the cell sizes, N_xy that of g, over 4 pi V; the other components permute
// the axes.  At |R| >= rfar the differences lose digits in FP64, and the
// dipole tensor averaged over both cells to O(h^4/R^4) is used instead:
// N = -V/(4 pi) [T(R)/2 + sum_a (T(R + h_a e_a) + T(R - h_a e_a))/12].
// The kernel value is -N (the sign of Kernel_Arne's field kernel).
__device__ double nw_f(double x, double y, double z) {
    x = fabs(x);
    y = fabs(y);
    z = fabs(z);
    const double x2 = x * x, y2 = y * y, z2 = z * z, R = sqrt(x2 + y2 + z2);
    double r = (2 * x2 - y2 - z2) * R / 6;
    if (y > 0 && x2 + z2 > 0) r += 0.5 * y * (z2 - x2) * asinh(y / sqrt(x2 + z2));
    if (z > 0 && x2 + y2 > 0) r += 0.5 * z * (y2 - x2) * asinh(z / sqrt(x2 + y2));
    if (x > 0 && y > 0 && z > 0) r -= x * y * z * atan(y * z / (x * R));
    return r;
}
__device__ double nw_g(double x, double y, double z) {
    double sg = 1;
    if (x < 0) {
        sg = -sg;
        x = -x;
    }
    if (y < 0) {
        sg = -sg;
        y = -y;
    }
    z = fabs(z);
    const double x2 = x * x, y2 = y * y, z2 = z * z, R = sqrt(x2 + y2 + z2);
    double r = -x * y * R / 3;
    if (z > 0 && x2 + y2 > 0) r += x * y * z * asinh(z / sqrt(x2 + y2));
    if (x > 0 && y2 + z2 > 0) r += y / 6 * (3 * z2 - y2) * asinh(x / sqrt(y2 + z2));
    if (y > 0 && x2 + z2 > 0) r += x / 6 * (3 * z2 - x2) * asinh(y / sqrt(x2 + z2));
    if (z > 0) r -= z2 * z / 6 * atan(x * y / (z * R));
    if (y > 0) r -= z * y2 / 2 * atan(x * z / (y * R));
    if (x > 0) r -= z * x2 / 2 * atan(y * z / (x * R));
    return sg * r;
}
// sum over i, j, k in {-1, 0, 1} of w_i w_j w_k F(X + i a, Y + j b, Z + k c), w_0 = 2, w_1 = -1
template <bool G>
__device__ double nw_stencil(double X, double Y, double Z, double a, double b, double c) {
    double s = 0;
    for (int i = -1; i <= 1; i++)
        for (int j = -1; j <= 1; j++)
            for (int k = -1; k <= 1; k++) {
                const double w = (i ? -1.0 : 2.0) * (j ? -1.0 : 2.0) * (k ? -1.0 : 2.0);
                s += w * (G ? nw_g(X + i * a, Y + j * b, Z + k * c) : nw_f(X + i * a, Y + j * b, Z + k * c));
            }
    return s;
}
__device__ void nw_dipole(const double R[3], double t[6]) {
    const double r2 = R[0] * R[0] + R[1] * R[1] + R[2] * R[2], r5 = r2 * r2 * sqrt(r2);
    t[0] = (3 * R[0] * R[0] - r2) / r5;
    t[1] = (3 * R[1] * R[1] - r2) / r5;
    t[2] = (3 * R[2] * R[2] - r2) / r5;
    t[3] = 3 * R[1] * R[2] / r5;
    t[4] = 3 * R[0] * R[2] / r5;
    t[5] = 3 * R[0] * R[1] / r5;
}
// One lane per octant cell: -N summed over the cell's images (the image
// ranges of k_kernel_arne), components XX, YY, ZZ, YZ, XZ, XY.
__global__ void __launch_bounds__(64) k_kernel_newell(double* __restrict__ oct, int s0, int s1, int s2, double c0,
                                                      double c1, double c2, int r10, int r11, int r12, int r20,
                                                      int r21, int r22, double rfar) {
#pragma clang fp contract(off)
    const int h0 = s0 / 2 + 1, h1 = s1 / 2 + 1, h2 = s2 / 2 + 1;
    const long noct = (long)h0 * h1 * h2;
    const long I = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (I >= noct) return;
    const int zw = (int)(I % h2);
    const int yw = (int)((I / h2) % h1);
    const int xw = (int)(I / ((long)h1 * h2));
    const double V = c0 * c1 * c2, k = 1.0 / (4 * HS_PI_D * V);
    double acc[6] = {0, 0, 0, 0, 0, 0};
    for (int z = first_image(zw, s2, r12); z <= r22; z += s2)
        for (int y = first_image(yw, s1, r11); y <= r21; y += s1)
            for (int x = first_image(xw, s0, r10); x <= r20; x += s0) {
                const double R[3] = {x * c0, y * c1, z * c2};
                const double r = sqrt(R[0] * R[0] + R[1] * R[1] + R[2] * R[2]);
                double N[6];
                if (r >= rfar) {
                    const double h[3] = {c0, c1, c2};
                    double t[6], sum[6];
                    nw_dipole(R, t);
                    for (int c = 0; c < 6; c++) sum[c] = 0.5 * t[c];
                    for (int a = 0; a < 3; a++)
                        for (int sgn = -1; sgn <= 1; sgn += 2) {
                            double Q[3] = {R[0], R[1], R[2]};
                            Q[a] += sgn * h[a];
                            nw_dipole(Q, t);
                            for (int c = 0; c < 6; c++) sum[c] += t[c] / 12;
                        }
                    for (int c = 0; c < 6; c++) N[c] = -V / (4 * HS_PI_D) * sum[c];
                } else {
                    N[0] = k * nw_stencil<false>(R[0], R[1], R[2], c0, c1, c2);
                    N[1] = k * nw_stencil<false>(R[1], R[0], R[2], c1, c0, c2);
                    N[2] = k * nw_stencil<false>(R[2], R[1], R[0], c2, c1, c0);
                    N[3] = k * nw_stencil<true>(R[1], R[2], R[0], c1, c2, c0);
                    N[4] = k * nw_stencil<true>(R[0], R[2], R[1], c0, c2, c1);
                    N[5] = k * nw_stencil<true>(R[0], R[1], R[2], c0, c1, c2);
                }
                for (int c = 0; c < 6; c++) acc[c] -= N[c];
            }
    for (int c = 0; c < 6; c++) oct[c * noct + I] = acc[c];
}

// Fill the full real (P0,P1,P2) kernel of component c from its octant with
// the mirror signs of kernel_magnetostatic.go:190-234 (octant h0 x h1 x h2;
// distances beyond it, which no pair of cells has, are zero).
__global__ void k_kernel_fill(double* __restrict__ full, const double* __restrict__ oct, int s0, int s1, int s2,
                              int h0, int h1, int h2) {
    const long noct = (long)h0 * h1 * h2;
    const long n = (long)s0 * s1 * s2;
    long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    int c = blockIdx.y;
    if (g >= n) return;
    int z = (int)(g % s2);
    int y = (int)((g / s2) % s1);
    int x = (int)(g / ((long)s1 * s2));
    bool fx = x > s0 / 2, fy = y > s1 / 2, fz = z > s2 / 2;
    int xm = fx ? s0 - x : x, ym = fy ? s1 - y : y, zm = fz ? s2 - z : z;
    double sg = 1.0;
    if (c == 5) sg = (fx != fy) ? -1.0 : 1.0;        // XY odd in x and y
    else if (c == 4) sg = (fx != fz) ? -1.0 : 1.0;   // XZ odd in x and z
    else if (c == 3) sg = (fy != fz) ? -1.0 : 1.0;   // YZ odd in y and z
    full[c * n + g] = xm < h0 && ym < h1 && zm < h2 ? sg * oct[c * noct + ((long)xm * h1 + ym) * h2 + zm] : 0.0;
}

// max |oct| of each component into bits[6] (zeroed beforehand).  Copying the octant
// to the host for its maxima took 1.6 of the 10.4 ms of a plan at 256x256x8.
__global__ void __launch_bounds__(256) k_octant_max(const double* __restrict__ oct, long noct,
                                                    unsigned long long* __restrict__ bits) {
    __shared__ double wm[4];
    const int c = blockIdx.y;
    double m = 0;
    for (long g = (long)blockIdx.x * blockDim.x + threadIdx.x; g < noct; g += (long)gridDim.x * blockDim.x)
        m = fmax(m, fabs(oct[c * noct + g]));
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x >> 6); w++) m = fmax(m, wm[w]);
        atomicMax(&bits[c], (unsigned long long)__double_as_longlong(m));
    }
}

// Keep the real part of the first octant of the transformed kernel, scaled by
// 1/(P0 P1 P2); record max|imag| and max|real| (extract(), maxwell_convolution.go:350-388).
// kern64 rows at pitch H2, kern32 rows at pitch KP; the maxima go through a
// block reduction into kExtractLanes (imag, real) pairs of partial maxima.
constexpr int kExtractLanes = 32;
__global__ void __launch_bounds__(256) k_kernel_extract(const cpx<double>* __restrict__ X, double* __restrict__ kern64,
                                 float* __restrict__ kern32, int P0, int P1, int H2, int H2p, int K0, int K1, int KP,
                                 double norm, unsigned long long* __restrict__ maxbits) {
    __shared__ double wm[2][4];
    long nk = (long)K0 * K1 * H2;
    long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    int c = blockIdx.y;
    double mi = 0, mr = 0;
    if (g < nk) {
        int k = (int)(g % H2);
        int j = (int)((g / H2) % K1);
        int i = (int)(g / ((long)K1 * H2));
        cpx<double> v = X[(((long)c * P0 + i) * P1 + j) * H2p + k];
        double r = v.x * norm;
        kern64[c * nk + g] = r;
        if (kern32) kern32[(long)c * K0 * K1 * KP + ((long)i * K1 + j) * KP + k] = (float)r;
        mi = fabs(v.y);
        mr = fabs(v.x);
    }
    for (int o = 32; o > 0; o >>= 1) {
        mi = fmax(mi, __shfl_xor(mi, o, 64));
        mr = fmax(mr, __shfl_xor(mr, o, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        wm[0][threadIdx.x >> 6] = mi;
        wm[1][threadIdx.x >> 6] = mr;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x >> 6); w++) {
            mi = fmax(mi, wm[0][w]);
            mr = fmax(mr, wm[1][w]);
        }
        const int l = (int)((blockIdx.x + blockIdx.y) % kExtractLanes);
        atomicMax(&maxbits[2 * l], (unsigned long long)__double_as_longlong(mi));
        atomicMax(&maxbits[2 * l + 1], (unsigned long long)__double_as_longlong(mr));
    }
}

// The fused kernel's table K~(d; j', k), planes d < N0, from the octant of the
// transformed tensor: the inverse transform along axis 0, real and even in d
// for XX, YY, ZZ, YZ, i kappa and odd for XZ, XY (tw0: w_P0^t); XX is kept
// negated, as the fused kernel uses it.
// kt[((tc N0 + d) KR + pos) 6 + component]: without folding tc = k and
// pos = k1 B + k2 holds row j' = k1 + A k2; folded by R, tc = k (R/2 + 1) + s
// and pos the row j' = R (k1 + A k2) + s.
constexpr int kTabD = 8;  // planes a thread forms at a time
template <typename T>
__global__ void __launch_bounds__(256) k_kernel_table(const double* __restrict__ kern, T* __restrict__ kt, int N0,
                                                      int P0, int P1, int H2, int K0, int K1, int R, int A, int B,
                                                      int KR, const cpx<double>* __restrict__ tw0) {
    const int TC = fused::table_cols(R);
    const long n = (long)H2 * TC * KR;
    const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int c = blockIdx.y;
    if (g >= n) return;
    const int k = (int)(g % H2);  // consecutive lanes read consecutive k
    const int s = (int)((g / H2) % TC), pos = (int)(g / ((long)H2 * TC));
    const int j = R * (pos / B + A * (pos % B)) + s;
    const bool mir = 2 * j > P1;
    const double sg = mir && (c == 3 || c == 5) ? -1.0 : 1.0;  // YZ and XY are odd along axis 1
    const double* q = kern + ((long)c * K0 * K1 + (mir ? P1 - j : j)) * H2 + k;
    T* o = kt + (((long)k * TC + s) * N0 * KR + pos) * 6 + c;
    for (int d0 = 0; d0 < N0; d0 += kTabD) {
        double acc[kTabD];
        for (int u = 0; u < kTabD; u++) acc[u] = 0.0;
        for (int i = 0; i < K0; i++) {
            const double v = sg * q[(long)i * K1 * H2] * ((i == 0 || 2 * i == P0) ? 1.0 : 2.0);
#pragma unroll
            for (int u = 0; u < kTabD; u++) {
                const cpx<double> w = tw0[(int)((long)i * (d0 + u) % P0)];
                acc[u] += v * (c < 4 ? w.x : -w.y);
            }
        }
        for (int u = 0; u < kTabD; u++)
            if (d0 + u < N0) o[(long)(d0 + u) * KR * 6] = T(c == 0 ? -acc[u] : acc[u]);
    }
}

// ------------------------------------------------------------------ dispatch tables
template <typename T>
using r2c_fn = void (*)(const void*, const void*, long, cpx<T>*, long, int, int, const cpx<T>*, const cpx<T>*,
                        hipStream_t, long);

namespace {

// FP64 kernel of a compiled length: the two-level register transforms of
// fft2.hpp where they are the faster, the Stockham kernels of
// demag_kernels.hpp elsewhere.  Times of one pass, Stockham / two-level:
// - rows (33 MB): R2C 14.8 / 9.9 us at M = 64, 19.1 / 11.4 at 256, 16.2 / 13.3
//   at 512; C2R 12.7 / 8.0, 17.0 / 8.8, 15.7 / 9.4; M = 1024 15.0 / 25.5.
//   Eight rows a block (16 where eight give less than a wave), four from 384
//   points on (C2R; R2C at 384 with eight 24.7 against 13.5).  R2C at 512 keeps
//   eight: of the three lengths from 384 on it alone gains in small and large
//   launches.  A field with eight / four: 512x512x16 734 / 753 us and 512x64x34
//   187 / 194; 384x512x16 558 / 567 but 384x64x34 142 / 134, where the tile's 192
//   threads are too few; 640x512x16 962 / 940 and 640x64x34 272 / 257, where its LDS
//   leaves a CU one block.
// - columns (107 MB out and in): 55 / 54 us at 32 points, 65 / 57 at 128,
//   102 / 66 at 320, but 86 / 96 at 512 and within 5 % at 768 and 1024.
// - axis 0 with the product (1.8 MB a plane): one lane a pencil up to 8
//   points (12.0 / 5.7 us at 8), two up to 40 (39 / 16 at 32), four up to 128
//   (86 / 32 at 64, 163 / 100 at 128): 565 / 190 us at 512x512x16, where the
//   Stockham kernel took half the time of the field.
template <int M>
constexpr int rows2_w64(bool c2r) {
    if (M >= 384) return c2r || M != 512 ? 4 : 8;
    return 8 * split2(M).B >= 64 ? 8 : 16;
}
template <typename T, int M>
constexpr bool rows_two_level() { return sizeof(T) == 8 && M >= 16 && M <= 640 && two_level_ok(M); }
template <typename T, int L>
constexpr bool cols_two_level() { return sizeof(T) == 8 && L >= 32 && L <= 384 && two_level_ok(L); }

template <typename T, typename TI, int M>
void launch_r2c(const void* x, const void* msk, long mrows, cpx<T>* out, long nrows, int n2, int H2p,
                const cpx<T>* twM, const cpx<T>* twP, hipStream_t st) {
    if constexpr (rows_two_level<T, M>()) {
        constexpr int W = rows2_w64<M>(false);
        hipLaunchKernelGGL((k_r2c_rows2<T, M, W>), dim3((unsigned)((nrows + W - 1) / W)), dim3(W * split2(M).B), 0, st,
                           (const T*)x, (const T*)msk, mrows, out, nrows, n2, H2p, twM, twP, Live{nullptr, 1});
    } else {
        constexpr int W = row_w<M>();
        unsigned g = (unsigned)((nrows + W - 1) / W);
        hipLaunchKernelGGL((k_r2c_rows<T, TI, M>), dim3(g), dim3(row_nt<M>()), 0, st, (const TI*)x, (const TI*)msk,
                           mrows, out, nrows, n2, H2p, twM, twP, Live{nullptr, 1});
    }
}
template <typename T, typename TO, int M>
void launch_c2r(const cpx<T>* in, void* x, long nrows, int n2, int H2p, const cpx<T>* twM, const cpx<T>* twP,
                hipStream_t st) {
    if constexpr (rows_two_level<T, M>()) {
        constexpr int W = rows2_w64<M>(true);
        hipLaunchKernelGGL((k_c2r_rows2<T, M, W>), dim3((unsigned)((nrows + W - 1) / W)), dim3(W * split2(M).B), 0, st,
                           in, (T*)x, nrows, n2, H2p, twM, twP, Live{nullptr, 1});
    } else {
        constexpr int W = row_w<M>();
        unsigned g = (unsigned)((nrows + W - 1) / W);
        hipLaunchKernelGGL((k_c2r_rows<T, TO, M>), dim3(g), dim3(row_nt<M>()), 0, st, in, (TO*)x, nrows, n2, H2p, twM,
                           twP, Live{nullptr, 1});
    }
}
template <typename T, int L, int S>
void launch_cols(const cpx<T>* in, cpx<T>* out, Geo gi, Geo go, int npencil, int nin, int nkeep, int ncol,
                 const cpx<T>* tw, hipStream_t st) {
    if constexpr (cols_two_level<T, L>()) {
        constexpr int W = 8;  // 128 bytes
        dim3 g((unsigned)((ncol + W - 1) / W), (unsigned)npencil);
        hipLaunchKernelGGL((k_cols2<T, L, S, W>), g, dim3(W * split2(L).B), 0, st, in, out, gi, go, nin, nkeep, ncol,
                           tw, Live{nullptr, 1});
    } else {
        constexpr int W = col_w<T, L>();
        dim3 g((unsigned)((ncol + W - 1) / W), (unsigned)npencil);
        hipLaunchKernelGGL((k_cols<T, L, S>), g, dim3(col_nt<T, L>()), 0, st, in, out, gi, go, nin, nkeep, ncol, tw,
                           Live{nullptr, 1});
    }
}
template <typename T, typename TK, int L>
void launch_zconv(cpx<T>* X, const TK* kern, int N0, int P1, int H2, int H2p, int K1, T srcMul, const cpx<T>* tw,
                  hipStream_t st) {
    auto grid = [&](int W) { return dim3((unsigned)((H2 + W - 1) / W), (unsigned)(P1 / 2 + 1)); };
    const Live all{nullptr, 1};
    if constexpr (sizeof(T) == 8 && L > 1 && L <= 8) {
        hipLaunchKernelGGL((k_zconv2<T, TK, L, 16>), grid(16), dim3(96), 0, st, X, kern, N0, P1, H2, H2p, K1, H2,
                           srcMul, tw, all);
    } else if constexpr (sizeof(T) == 8 && L > 8 && L <= 40 && L % 2 == 0) {
        hipLaunchKernelGGL((k_zconv2m<T, TK, L, 16, 2>), grid(16), dim3(192), 0, st, X, kern, N0, P1, H2, H2p, K1, H2,
                           srcMul, tw, all);
    } else if constexpr (sizeof(T) == 8 && L > 40 && L <= 128 && L % 4 == 0) {
        hipLaunchKernelGGL((k_zconv2m<T, TK, L, 8, 4>), grid(8), dim3(192), 0, st, X, kern, N0, P1, H2, H2p, K1, H2,
                           srcMul, tw, all);
    } else {
        hipLaunchKernelGGL((k_zconv<T, TK, L>), grid(z_w<T, L>()), dim3(z_nt<T, L>()), 0, st, X, kern, N0, P1, H2,
                           H2p, K1, H2, srcMul, tw, all);
    }
}

template <typename T, typename TI>
using r2c_t = void (*)(const void*, const void*, long, cpx<T>*, long, int, int, const cpx<T>*, const cpx<T>*,
                       hipStream_t);
template <typename T, typename TO>
using c2r_t = void (*)(const cpx<T>*, void*, long, int, int, const cpx<T>*, const cpx<T>*, hipStream_t);
template <typename T>
using cols_t = void (*)(const cpx<T>*, cpx<T>*, Geo, Geo, int, int, int, int, const cpx<T>*, hipStream_t);
template <typename T, typename TK>
using zconv_t = void (*)(cpx<T>*, const TK*, int, int, int, int, int, T, const cpx<T>*, hipStream_t);

constexpr long kMaxLds = 163840;
template <typename T, int M>
constexpr bool rows_fit() { return (long)(M + 1) * row_w<M>() * (long)sizeof(cpx<T>) <= kMaxLds; }
template <typename T, int L>
constexpr bool cols_fit() { return (long)L * col_w<T, L>() * (long)sizeof(cpx<T>) <= kMaxLds; }
template <typename T, int L>
constexpr bool z_fit() { return L <= 256 && (long)L * 6 * z_w<T, L>() * (long)sizeof(cpx<T>) <= kMaxLds; }

template <typename T, typename TI>
r2c_t<T, TI> pick_r2c(int M) {
#define X(n) \
    if constexpr (rows_fit<T, n>()) if (M == n) return &launch_r2c<T, TI, n>;
    HS_FFT_SIZES(X)
#undef X
    return nullptr;
}
template <typename T, typename TO>
c2r_t<T, TO> pick_c2r(int M) {
#define X(n) \
    if constexpr (rows_fit<T, n>()) if (M == n) return &launch_c2r<T, TO, n>;
    HS_FFT_SIZES(X)
#undef X
    return nullptr;
}
template <typename T, int S>
cols_t<T> pick_cols(int L) {
#define X(n) \
    if constexpr (cols_fit<T, n>()) if (L == n) return &launch_cols<T, n, S>;
    HS_FFT_SIZES(X)
#undef X
    return nullptr;
}
template <typename T, typename TK>
zconv_t<T, TK> pick_zconv(int L) {
#define X(n) \
    if constexpr (z_fit<T, n>()) if (L == n) return &launch_zconv<T, TK, n>;
    HS_FFT_SIZES(X)
#undef X
    return nullptr;
}

}  // namespace

// ------------------------------------------------------------------ plan
struct hs_demag {
    // P: the lengths of the transforms, K: octant of the transformed kernel
    int N[3], P[3], K[3], pbc[3];
    // the reference's logic size (2 N on open axes) and its octant, which
    // hs_demag_sizes and hs_demag_kernel_f64 report; an open axis whose 2 N has
    // no compiled family is transformed at a longer P (set_lengths)
    int logic[3], logicK[3];
    bool noalloc = false;     // hs_demag_field_f64_noalloc takes the mesh: its spectra at the logic size fit
    double* kernL = nullptr;  // kernel octants at the logic size where P differs, else kern64
    // the FP64 fields at the logic size (its kern64 is kernL), where the spectra at P
    // do not fit the static array of hs_demag_field_f64_noalloc
    hs_demag* f64 = nullptr;
    double cell[3];
    int M, H2, H2p;  // H2p: spectrum row pitch (complex), a multiple of 16 = 128 bytes in FP32
    int KP;          // FP32 kernel row pitch (floats), a multiple of 32 = 128 bytes
    long ncell;
    double* kern64 = nullptr;
    float* kern32 = nullptr;  // the five FP32 passes' copy (fold32 = 0)
    cpx<float>*X1f = nullptr, *X2f = nullptr;
    cpx<double>*X1d = nullptr, *X2d = nullptr;
    cpx<float>*twMf = nullptr, *twP2f = nullptr, *tw1f = nullptr, *tw0f = nullptr;
    cpx<double>*twMd = nullptr, *twP2d = nullptr, *tw1d = nullptr, *tw0d = nullptr;
    unsigned char* tw = nullptr;  // the tables above
    double max_imag_ratio = 0;
    // FP32 pass variants chosen by timing at plan creation
    hsdm::RowV row32{};   // forward (R2C) row pass
    hsdm::RowV rowi32{};  // inverse (C2R) row pass, timed on its own
    hsdm::ColV col32{};
    hsdm::ZV z32{};
    bool tuned = false;
    int cap = 1;  // solves the X1/X2 buffers hold
    // passes without a compiled length family run the run-time-length kernels
    // of fft_any.hpp: rows (R2C/C2R, FFT of gR.L = P2/2, or P2 when odd),
    // columns (P1), axis 0 (P0); FP32 and FP64 decided separately
    bool genR = false, gen1 = false, gen0 = false, genRd = false, gen1d = false, gen0d = false;
    GenFFT gR{}, g1{}, g0{};
    // three-kernel convolution (demag_fused.hpp): the fold of axis 1, 0 = not
    // taken, FP32 and FP64 decided separately; kt64 may be filled on first use
    int fold32 = 0, fold64 = 0;
    fused::Form<float> form32;   // their kernels
    fused::Form<double> form64;
    float* kt32 = nullptr;
    double* kt64 = nullptr;
    cpx<float>* Xzf = nullptr;   // (cap, 3, P0, P1, H2p): the axis-0 spectrum of a run-time-length F3K
    cpx<double>* Xzd = nullptr;  // the same for the FP64 field
};

namespace {
template <typename T>
struct Pipe {
    r2c_t<T, T> r2c;
    c2r_t<T, T> c2r;
    cols_t<T> fwd1, inv1;
    zconv_t<T, T> zc;
};

// Lengths with a compiled family: FP32 with registered tile variants, FP64
// with a Stockham instantiation.
bool rows32(int P2) {
    return P2 % 2 == 0 && fft_supported(P2 / 2) && pick_r2c<float, float>(P2 / 2) &&
           !hsdm::variants(P2 / 2).rows.empty();
}
bool rows64(int P2) {
    return P2 % 2 == 0 && fft_supported(P2 / 2) && pick_r2c<double, double>(P2 / 2) &&
           pick_c2r<double, double>(P2 / 2);
}
bool cols32(int P1) { return pick_cols<float, -1>(P1) && !hsdm::variants(P1).cols.empty(); }
bool cols64(int P1) { return pick_cols<double, -1>(P1) != nullptr; }
bool z32_ok(int P0) { return pick_zconv<float, float>(P0) && !hsdm::variants(P0).z.empty(); }
bool z64_ok(int P0) { return pick_zconv<double, double>(P0) != nullptr; }

// The lengths of the transforms and what follows from them: which passes take
// the run-time-length kernels.  False when a generic length exceeds their LDS
// limit (the FP64 kernel set-up transforms every axis).
bool set_lengths(hs_demag* d, const int P[3]) {
    for (int c = 0; c < 3; c++) d->P[c] = P[c];
    const int P0 = P[0], P1 = P[1], P2 = P[2];
    d->M = P2 / 2;
    d->H2 = d->M + 1;
    d->H2p = (d->H2 + 15) / 16 * 16;
    d->KP = (d->H2 + 31) / 32 * 32;
    d->K[0] = P0 / 2 + 1;
    d->K[1] = P1 / 2 + 1;
    d->K[2] = d->H2;
    d->genR = !rows32(P2);
    d->gen1 = !cols32(P1);
    d->gen0 = !z32_ok(P0);
    d->genRd = !rows64(P2);
    d->gen1d = !cols64(P1);
    d->gen0d = !z64_ok(P0);
    d->gR = gen_fft_plan(P2 % 2 == 0 ? d->M : P2);
    d->g1 = gen_fft_plan(P1);
    d->g0 = gen_fft_plan(P0);
    const int lim = gen_max_len<double>();
    return d->gR.L <= lim && P1 <= lim && P0 <= lim;
}
size_t up256(size_t b) { return (b + 255) / 256 * 256; }
// The roots exp(-2 pi i t / L) of the plan's lengths, FP64 and (f32) FP32, in one
// allocation and one copy; false without memory.
bool make_twiddles(hs_demag* d, bool f32) {
    const int L[4] = {d->M, d->P[2], d->P[1], d->P[0]};
    cpx<double>** pd[4] = {&d->twMd, &d->twP2d, &d->tw1d, &d->tw0d};
    cpx<float>** pf[4] = {&d->twMf, &d->twP2f, &d->tw1f, &d->tw0f};
    size_t at[5] = {0};  // an FP64 table, then its FP32 copy
    for (int k = 0; k < 4; k++)
        at[k + 1] = at[k] + up256(sizeof(cpx<double>) * (L[k] + 1)) + (f32 ? up256(sizeof(cpx<float>) * (L[k] + 1)) : 0);
    if (hipMalloc(&d->tw, at[4]) != hipSuccess) {
        d->tw = nullptr;
        return false;
    }
    std::vector<unsigned char> host(at[4]);
    for (int k = 0; k < 4; k++) {
        const size_t f = at[k] + up256(sizeof(cpx<double>) * (L[k] + 1));
        cpx<double>* hd = reinterpret_cast<cpx<double>*>(&host[at[k]]);
        cpx<float>* hf = f32 ? reinterpret_cast<cpx<float>*>(&host[f]) : nullptr;
        for (int t = 0; t < L[k]; t++) {
            const long double a = -2.0L * 3.14159265358979323846264338327950288L * (long double)t / (long double)L[k];
            const long double c = cosl(a), s = sinl(a);
            hd[t] = {(double)c, (double)s};
            if (hf) hf[t] = {(float)c, (float)s};
        }
        *pd[k] = reinterpret_cast<cpx<double>*>(d->tw + at[k]);
        if (f32) *pf[k] = reinterpret_cast<cpx<float>*>(d->tw + f);
    }
    return hipMemcpy(d->tw, host.data(), at[4], hipMemcpyHostToDevice) == hipSuccess;
}
// Axis c of length L runs compiled kernels in FP32 and FP64.
bool axis_compiled(int c, int L) {
    if (c == 0) return z32_ok(L) && z64_ok(L);
    return c == 1 ? cols32(L) && cols64(L) : rows32(L) && rows64(L);
}
// The shortest compiled length >= P of axis c, P itself if there is none.
// An open axis is zero-padded, so any length from 2 N - 1 on gives the same
// convolution.  2 N itself where it is compiled; otherwise the next of 2^k,
// 3 2^k and 5 2^k costs at most 1.33 times the points and runs the compiled
// kernels instead of the run-time-length ones (FP32 field, run-time lengths
// against padded: 100x75x7 78 -> 20 us, 33^3 171 -> 25, 100^3 383 -> 222,
// 300x300x33 2086 -> 334, 300x300x17 2502 -> 138; no mesh was slower).
int compiled_length(int c, int P) {
    int best = 0;
#define X(n) \
    for (int L : {n, 2 * n}) \
        if (L >= P && axis_compiled(c, L) && (!best || L < best)) best = L;
    HS_FFT_SIZES(X)
#undef X
    return best ? best : P;
}
// Relative time of the five passes of N at lengths P: points of each pass (rows
// and axis 1 there and back, axis 0 with the product in one) times 2, and for a
// run-time length 2 more for each stage of up to 8 points or R for a stage of a
// prime R, which sums directly.
double passes_cost(const int N[3], const int P[3]) {
    auto len = [&](int c) {
        if (axis_compiled(c, P[c])) return 2;
        const GenFFT g = gen_fft_plan(c == 2 && P[2] % 2 == 0 ? P[2] / 2 : P[c]);
        int t = 2;
        for (int s = 0; s < g.nst; s++) t += g.r[s] <= 8 ? 2 : g.r[s];
        return t;
    };
    const double H2 = P[2] / 2 + 1;
    return 2.0 * N[0] * N[1] * (P[2] / 2) * len(2) + 2.0 * N[0] * P[1] * H2 * len(1) +
           P[0] * P[1] * H2 * (2 * len(0) + 4);
}
// Lengths of the transforms: open axes at their next compiled length.  Where one
// has none (more than 128 planes, more than 1024 rows, 2048 cells along x) its
// run-time pass pays for the padding of the others, so only the axes are padded
// with which passes_cost is least: 100x64x140 291 us a field at 2 N, 331 padded;
// 49x49x130 301 / 383; but 16x37x140 511 / 63.  (Run-time lengths of
// periodic axes do not count: at 60 such meshes padding the others was 9 %
// slower at worst, in FP64, and up to 40 times faster.)
void padded_lengths(const int N[3], const int logic[3], int P[3]) {
    int full[3];
    bool all = true;
    for (int c = 0; c < 3; c++) {
        const bool open = logic[c] > N[c];
        full[c] = open ? compiled_length(c, logic[c]) : logic[c];
        all = all && (!open || axis_compiled(c, full[c]));
    }
    std::copy(all ? full : logic, (all ? full : logic) + 3, P);
    if (all) return;
    double least = passes_cost(N, logic);
    for (int s = 1; s < 8; s++) {
        int Q[3];
        for (int c = 0; c < 3; c++) Q[c] = s >> c & 1 ? full[c] : logic[c];
        const double t = passes_cost(N, Q);
        if (t < least) {
            least = t;
            std::copy(Q, Q + 3, P);
        }
    }
}

// Fold R of axis 1 with which the fused kernels take the mesh (mid_fold), 0 if
// they do not: open axes 0 and 1 (or one plane), an even padded x length,
// registered lengths.
template <typename T>
int fused_fold(const hs_demag* d) {
    const int P1 = d->P[1], N0 = d->N[0];
    if (d->P[2] % 2 || P1 < 2 * d->N[1] || !(N0 == 1 || d->P[0] >= 2 * N0)) return 0;
    return fused::mid_fold(N0, P1, sizeof(cpx<T>), std::equal(d->P, d->P + 3, d->logic), [&](int R) {
        const fused::Mids<T>& m = fused::mids_of<T>(P1 / R);
        return fused::rows_of<T>(d->M).fwd[fused::fold_index(R)] && m.A && m.pick(N0, R > 1) &&
               fused::mid_fits(N0, P1 / R, m.A, m.B, sizeof(cpx<T>));
    });
}
// the kernels of fold R, resolved at creation: a field call looks nothing up
template <typename T>
fused::Form<T> fused_form(const hs_demag* d, int R) {
    if (!R) return {};
    const fused::Rows<T>& r = fused::rows_of<T>(d->M);
    const fused::Mids<T>& m = fused::mids_of<T>(d->P[1] / R);
    const int f = fused::fold_index(R);
    const bool few = R == 1 && d->N[0] > 8 && fused::mid_nt(d->N[0], d->P[1], 1, fused::kFewIB) <= fused::kMidMax;
    return {r.fwd[f], r.inv[f], m.pick(d->N[0], R > 1), few ? m.few : nullptr, m.A, m.B};
}
// values of the fused spectrum (per solve) and of its kernel table
long fused_spectrum(const hs_demag* d, int R) { return 3L * d->N[0] * (R > 1 ? d->P[1] : d->N[1]) * d->H2p; }
int fused_rows(const hs_demag* d, int R) { return fused::table_rows_of(d->P[1] / R, R > 1); }
long fused_table(const hs_demag* d, int R) {
    return 6L * d->N[0] * fused_rows(d, R) * fused::table_cols(R) * d->H2;
}
// Fills the table of fold R from the FP64 octant.
template <typename T>
void fill_table(const hs_demag* d, T* kt, int R, const fused::Form<T>& m, hipStream_t st) {
    const int KR = fused_rows(d, R);
    hipLaunchKernelGGL(k_kernel_table<T>, dim3(hs::grid1d((long)d->H2 * fused::table_cols(R) * KR), 6),
                       dim3(hs::kBlock), 0, st, d->kern64, kt, d->N[0], d->P[0], d->P[1], d->H2, d->K[0], d->K[1], R,
                       m.A, m.B, KR, d->tw0d);
}

// The fused convolution of nsolve solves (X: nsolve x fused_spectrum values).
template <typename T>
int run_fused(hs_demag* d, const T* m, const T* msk, double srcMul, T* B, hipStream_t st, cpx<T>* X, const T* kt,
              int R, const fused::Form<T>& fm, const cpx<T>* twM, const cpx<T>* twP2, const cpx<T>* tw1, int nsolve,
              const int* live) {
    const int N0 = d->N[0], N1 = d->N[1], Q = d->P[1] / R;
    const fused::RowP g{3 * N0 * N1, N1, Q, 3 * N0, nsolve, d->N[2], (long)N0 * N1};
    const Live lrows{live, g.rows};
    hs::prof_begin(HS_PROF_F1, st);
    fm.fwd(m, msk, X, g, T(0.5 * srcMul), twM, twP2, tw1, st, lrows);
    hs::prof_end(HS_PROF_F1, st);
    hs::prof_begin(HS_PROF_F3K, st);
    const int ncol = d->H2 * R;
    const fused::Mid<T> a{X,    kt,     N0, N1, ncol, fused::mid_cb(N0, Q, fm.A, fm.B, ncol, nsolve, sizeof(cpx<T>)),
                          nsolve, R, tw1, live};
    const long waves = (long)ncol * nsolve * (fused::mid_nt(N0, Q, 1) / 64);
    (fm.few && a.CB == 1 && waves < fused::kFewWaves ? fm.few : fm.mid)(a, st);
    hs::prof_end(HS_PROF_F3K, st);
    hs::prof_begin(HS_PROF_I1, st);
    fm.inv(X, B, g, twM, twP2, tw1, st, lrows);
    hs::prof_end(HS_PROF_I1, st);
    HS_LAUNCH_CHECK("hs_demag_field");
    return hs_last_error();
}

// FFT table of the row transform: P2/2 points (even P2) or P2 (odd)
template <typename T>
const cpx<T>* row_table(const hs_demag* d, const cpx<T>* twM, const cpx<T>* twP2) {
    return (d->P[2] % 2 == 0) ? twM : twP2;
}

// live: per-solve flags of a batch (null = all solves); blocks of solves
// with flag 0 exit without touching memory.
int run_field32(hs_demag* d, const float* m, const float* msk, double srcMul, float* B, hipStream_t st,
                int nsolve = 1, const int* live = nullptr) {
    const int N0 = d->N[0], N1 = d->N[1], N2 = d->N[2], P1 = d->P[1];
    const int H2 = d->H2, H2p = d->H2p;
    cpx<float>*X1 = d->X1f, *X2 = d->X2f;
    if (nsolve > d->cap) {
        hs::set_error(HS_EINVAL, "hs_demag_field: batch larger than reserved");
        return HS_EINVAL;
    }
    if (d->fold32)
        return run_fused<float>(d, m, msk, srcMul, B, st, X1, d->kt32, d->fold32, d->form32, d->twMf, d->twP2f, d->tw1f,
                                nsolve, live);
    const long nrows = 3L * N0 * N1 * nsolve;
    Geo g1 = {(long)N1 * H2p, 0, H2p, 1};
    Geo g2 = {(long)P1 * H2p, 0, H2p, 1};
    const int P0 = d->P[0], P2 = d->P[2];
    const cpx<float>* twR = row_table<float>(d, d->twMf, d->twP2f);
    hs::prof_begin(HS_PROF_F1, st);
    const Live lrows{live, 3L * N0 * N1}, lpen{live, 3L * N0}, lsol{live, 1};
    if (d->genR)
        gen::r2c<float>(m, msk, (long)N0 * N1, X1, nrows, N2, P2, H2p, d->gR, twR, d->twP2f, st, lrows);
    else
        d->row32.r2c(m, msk, (long)N0 * N1, X1, nrows, N2, H2p, d->twMf, d->twP2f, st, lrows);
    hs::prof_end(HS_PROF_F1, st);
    hs::prof_begin(HS_PROF_F2, st);
    if (d->gen1)
        gen::cols<float, -1>(X1, X2, g1, g2, 3 * N0 * nsolve, N1, P1, H2, d->g1, d->tw1f, st, lpen);
    else
        d->col32.fwd(X1, X2, g1, g2, 3 * N0 * nsolve, N1, P1, H2, d->tw1f, st, lpen);
    hs::prof_end(HS_PROF_F2, st);
    hs::prof_begin(HS_PROF_F3K, st);
    if (d->gen0)
        gen::zconv<float, float>(X2, d->Xzf, d->kern32, N0, P0, P1, H2, H2p, d->K[1], d->KP, (float)srcMul, d->g0,
                                 d->tw0f, st, nsolve, lsol);
    else
        d->z32.fn(X2, d->kern32, N0, P1, H2, H2p, d->K[1], d->KP, (float)srcMul, d->tw0f, st, nsolve, lsol);
    hs::prof_end(HS_PROF_F3K, st);
    hs::prof_begin(HS_PROF_I2, st);
    if (d->gen1)
        gen::cols<float, +1>(X2, X1, g2, g1, 3 * N0 * nsolve, P1, N1, H2, d->g1, d->tw1f, st, lpen);
    else
        d->col32.inv(X2, X1, g2, g1, 3 * N0 * nsolve, P1, N1, H2, d->tw1f, st, lpen);
    hs::prof_end(HS_PROF_I2, st);
    hs::prof_begin(HS_PROF_I1, st);
    if (d->genR)
        gen::c2r<float>(X1, B, nrows, N2, P2, H2p, d->gR, twR, d->twP2f, st, lrows);
    else
        d->rowi32.c2r(X1, B, nrows, N2, H2p, d->twMf, d->twP2f, st, lrows);
    hs::prof_end(HS_PROF_I1, st);
    HS_LAUNCH_CHECK("hs_demag_field");
    return hs_last_error();
}

// Time each registered FP32 variant of every pass on the plan's own buffers
// and keep the fastest (the tile autotuner).
// The choice is cached per mesh shape for the life of the process, so every
// plan of one shape runs the same variants: the variants differ in operation
// order, and solves of one shape must give identical results whichever plan
// (batch, slot batch, single solve) steps them.
struct TuneKey {
    int N[3], P[3];
    bool operator<(const TuneKey& o) const {
        for (int i = 0; i < 3; i++) {
            if (N[i] != o.N[i]) return N[i] < o.N[i];
            if (P[i] != o.P[i]) return P[i] < o.P[i];
        }
        return false;
    }
};
std::mutex g_tune_mu;
std::map<TuneKey, std::array<int, 4>>& tune_cache() {
    static std::map<TuneKey, std::array<int, 4>> c;
    return c;
}

// Tuned choices persisted across processes: HS_TUNE_FILE names a text file
// of lines "N0 N1 N2 P0 P1 P2 nr nc nz r c z ri" (mesh, padded size, the
// numbers of registered row/column/axis-0 variants, the picks).  A plan whose
// shape has a line with the same variant counts takes that choice without
// timing; a newly tuned shape is appended.  The variants of a pass differ
// in operation order (FP32 rounding), so processes that share the file give
// the same bits for the same inputs.
bool tune_file_read(const hs_demag* d, const std::array<int, 3>& counts, std::array<int, 4>& pick) {
    const char* path = getenv("HS_TUNE_FILE");
    if (!path || !*path) return false;
    FILE* f = fopen(path, "r");
    if (!f) return false;
    int v[13];
    bool found = false;
    while (!found && fscanf(f, "%d %d %d %d %d %d %d %d %d %d %d %d %d", &v[0], &v[1], &v[2], &v[3], &v[4], &v[5],
                            &v[6], &v[7], &v[8], &v[9], &v[10], &v[11], &v[12]) == 13) {
        found = v[0] == d->N[0] && v[1] == d->N[1] && v[2] == d->N[2] && v[3] == d->P[0] && v[4] == d->P[1] &&
                v[5] == d->P[2] && v[6] == counts[0] && v[7] == counts[1] && v[8] == counts[2] && v[9] >= 0 &&
                v[9] < counts[0] && v[10] >= 0 && v[10] < counts[1] && v[11] >= 0 && v[11] < counts[2] &&
                v[12] >= 0 && v[12] < counts[0];
        if (found) pick = {v[9], v[10], v[11], v[12]};
    }
    fclose(f);
    return found;
}
void tune_file_append(const hs_demag* d, const std::array<int, 3>& counts, const std::array<int, 4>& pick) {
    const char* path = getenv("HS_TUNE_FILE");
    if (!path || !*path) return;
    if (FILE* f = fopen(path, "a")) {
        fprintf(f, "%d %d %d %d %d %d %d %d %d %d %d %d %d\n", d->N[0], d->N[1], d->N[2], d->P[0], d->P[1], d->P[2],
                counts[0], counts[1], counts[2], pick[0], pick[1], pick[2], pick[3]);
        fclose(f);
    }
}

void apply_force(hs_demag* d, const hsdm::Variants& vr, const hsdm::Variants& vc, const hsdm::Variants& vz) {
    // HS_DEMAG_FORCE="r,c,z": variant indices to use instead of the timed
    // choice (-1 keeps it), for tests that cover every registered variant
    if (const char* f = getenv("HS_DEMAG_FORCE")) {
        int ir = -1, ic = -1, iz = -1;
        if (sscanf(f, "%d,%d,%d", &ir, &ic, &iz) == 3) {
            if (ir >= 0 && ir < (int)vr.rows.size()) d->row32 = d->rowi32 = vr.rows[ir];
            if (ic >= 0 && ic < (int)vc.cols.size()) d->col32 = vc.cols[ic];
            if (iz >= 0 && iz < (int)vz.z.size()) d->z32 = vz.z[iz];
        }
    }
}

void tune32(hs_demag* d, hipStream_t st) {
    const hsdm::Variants& vr = hsdm::variants(d->M);
    const hsdm::Variants& vc = hsdm::variants(d->P[1]);
    const hsdm::Variants& vz = hsdm::variants(d->P[0]);
    d->row32 = d->rowi32 = (d->genR || vr.rows.empty()) ? hsdm::RowV{} : vr.rows[0];
    d->col32 = (d->gen1 || vc.cols.empty()) ? hsdm::ColV{} : vc.cols[0];
    d->z32 = (d->gen0 || vz.z.empty()) ? hsdm::ZV{} : vz.z[0];
    if (d->fold32) return;  // none of these passes runs
    // a plan with a run-time-length pass keeps the first variant of its compiled
    // passes
    if (!d->row32.r2c || !d->col32.fwd || !d->z32.fn) return;
    // A plan at longer lengths than its logic size is not timed (0.3 s, which
    // meshes of any size would pay each for themselves).  It takes two-level rows
    // and columns, eight to a block (sixteen where eight make less than a wave), and
    // four lanes a pencil on axis 0 (one lane below 16 points); where a length has
    // none, the last variant, radix stages.  One field in us with these columns,
    // sixteen to a block, and the radix stages: 50x50x49 36.3, 36.9, 38.8;
    // 100x100x36 60.5, 58.6, 64.2; 190x190x33 121, 124, 141; 300x300x33 299, 333,
    // 327 (490 with the first variant of each pass).  Axis 0 with the others it has:
    // 100x100x36 63 against 68 to 125, periodic 100x100x16 41 against 39 to 53.
    if (d->kernL) {
        using hsdm::Kind;
        auto pick = [](const auto& list, Kind kind, int W) {
            const auto* v = hsdm::find_variant(list, kind, W);
            return v ? *v : list.back();
        };
        d->row32 = d->rowi32 = pick(vr.rows, Kind::two_level, 8);
        d->col32 = pick(vc.cols, Kind::two_level, 8);
        d->z32 = d->P[0] < 16 ? pick(vz.z, Kind::lane_nt, 32) : pick(vz.z, Kind::lanes4, 8);
        apply_force(d, vr, vc, vz);
        return;
    }
    const TuneKey key{{d->N[0], d->N[1], d->N[2]}, {d->P[0], d->P[1], d->P[2]}};
    const std::array<int, 3> counts{(int)vr.rows.size(), (int)vc.cols.size(), (int)vz.z.size()};
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        auto it = tune_cache().find(key);
        std::array<int, 4> filed;
        if (it == tune_cache().end() && tune_file_read(d, counts, filed)) it = tune_cache().emplace(key, filed).first;
        if (it != tune_cache().end()) {
            d->row32 = vr.rows[it->second[0]];
            d->rowi32 = vr.rows[it->second[3]];
            d->col32 = vc.cols[it->second[1]];
            d->z32 = vz.z[it->second[2]];
            apply_force(d, vr, vc, vz);
            d->tuned = true;
            return;
        }
    }
    const int N0 = d->N[0], N1 = d->N[1], N2 = d->N[2], P1 = d->P[1];
    const int H2 = d->H2, H2p = d->H2p;
    // Time the passes on a batch of nt solves of this mesh, about 4 M cells
    // (one solve of a large mesh; up to 256 of a small one): batches,
    // ensembles and slot batches of small meshes run the passes over many
    // solves at once, and a tile that is fastest for one small solve
    // (latency-bound grid) is often not the fastest for a full device.  The
    // batch depends on the mesh only, so the choice stays per shape.
    const int nt = (int)std::min<long>(256, std::max<long>(1, ((1L << 22) + d->ncell - 1) / d->ncell));
    const long nrows = 3L * N0 * N1 * nt;
    float *m = nullptr, *B = nullptr;
    cpx<float>*X1t = nullptr, *X2t = nullptr;
    hipMalloc(&m, sizeof(float) * 3 * d->ncell * nt);
    hipMalloc(&B, sizeof(float) * 3 * d->ncell * nt);
    if (nt > d->cap) {
        hipMalloc(&X1t, sizeof(cpx<float>) * 3L * N0 * N1 * H2p * nt);
        hipMalloc(&X2t, sizeof(cpx<float>) * 3L * N0 * P1 * H2p * nt);
    }
    if (!m || !B || (nt > d->cap && (!X1t || !X2t))) {
        hipFree(m);
        hipFree(B);
        hipFree(X1t);
        hipFree(X2t);
        return;  // keeps the first variant of each pass
    }
    // the plan's own spectrum buffers are swapped back in after the timing
    cpx<float>*X1own = d->X1f, *X2own = d->X2f;
    const int capown = d->cap;
    if (nt > d->cap) {
        d->X1f = X1t;
        d->X2f = X2t;
        d->cap = nt;
    }
    hipMemsetAsync(m, 0, sizeof(float) * 3 * d->ncell * nt, st);
    hipEvent_t e0, e1;
    hipEventCreate(&e0);
    hipEventCreate(&e1);
    // best of `rounds` rounds of 3 launches after a warm-up launch
    auto timeit = [&](auto&& launch, int rounds = 2) {
        launch();
        float best_ms = 1e30f;
        for (int round = 0; round < rounds; round++) {
            hipEventRecord(e0, st);
            for (int r = 0; r < 3; r++) launch();
            hipEventRecord(e1, st);
            hipEventSynchronize(e1);
            float ms = 1e30f;
            hipEventElapsedTime(&ms, e0, e1);
            best_ms = std::min(best_ms, ms);
        }
        return best_ms;
    };
    Geo g1 = {(long)N1 * H2p, 0, H2p, 1};
    Geo g2 = {(long)P1 * H2p, 0, H2p, 1};
    std::array<int, 4> pick{0, 0, 0, 0};  // r2c rows, columns, axis 0, c2r rows
    float best = 1e30f, besti = 1e30f;
    for (size_t i = 0; i < vr.rows.size(); i++) {
        auto& v = vr.rows[i];
        const Live all{nullptr, 1};
        float t = timeit([&] { v.r2c(m, nullptr, (long)N0 * N1, d->X1f, nrows, N2, H2p, d->twMf, d->twP2f, st, all); });
        float ti = timeit([&] { v.c2r(d->X1f, B, nrows, N2, H2p, d->twMf, d->twP2f, st, all); });
        if (t < best) { best = t; d->row32 = v; pick[0] = (int)i; }
        if (ti < besti) { besti = ti; d->rowi32 = v; pick[3] = (int)i; }
    }
    best = 1e30f;
    for (size_t i = 0; i < vc.cols.size(); i++) {
        auto& v = vc.cols[i];
        const Live all{nullptr, 1};
        float t = timeit([&] { v.fwd(d->X1f, d->X2f, g1, g2, 3 * N0 * nt, N1, P1, H2, d->tw1f, st, all); }) +
                  timeit([&] { v.inv(d->X2f, d->X1f, g2, g1, 3 * N0 * nt, P1, N1, H2, d->tw1f, st, all); });
        if (t < best) { best = t; d->col32 = v; pick[1] = (int)i; }
    }
    best = 1e30f;
    for (size_t i = 0; i < vz.z.size(); i++) {
        auto& v = vz.z[i];
        float t = timeit([&] { v.fn(d->X2f, d->kern32, N0, P1, H2, H2p, d->K[1], d->KP, 1.0f, d->tw0f, st, nt, Live{nullptr, 1}); });
        if (t < best) { best = t; d->z32 = v; pick[2] = (int)i; }
    }
    // One sweep of refinement inside the whole five-pass convolution: each
    // pass's variants again, the other passes fixed, so a pass is timed with
    // the caches and neighbours it has in a step (isolated timings can rank
    // close variants the other way).  Best of three rounds, and a variant
    // replaces the current one only when it is more than 1 % faster (closer
    // than that they are equivalent, and timing noise would decide).
    {
        auto pipe = [&] { run_field32(d, m, nullptr, 1.0, B, st, nt); };
        float cur = timeit(pipe, 3);
        auto sweep = [&](auto& slot, auto& list, int which) {
            for (size_t i = 0; i < list.size(); i++) {
                if ((int)i == pick[which]) continue;
                auto keep = slot;
                slot = list[i];
                const float t = timeit(pipe, 3);
                if (t < 0.99f * cur) {
                    cur = t;
                    pick[which] = (int)i;
                } else {
                    slot = keep;
                }
            }
        };
        sweep(d->row32, vr.rows, 0);
        sweep(d->col32, vc.cols, 1);
        sweep(d->z32, vz.z, 2);
        sweep(d->rowi32, vr.rows, 3);
    }
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        tune_cache()[key] = pick;
        tune_file_append(d, counts, pick);
    }
    apply_force(d, vr, vc, vz);
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    hipStreamSynchronize(st);
    d->X1f = X1own;
    d->X2f = X2own;
    d->cap = capown;
    hipFree(X1t);
    hipFree(X2t);
    hipFree(m);
    hipFree(B);
    d->tuned = true;
}

template <typename T>
int run_field(hs_demag* d, const T* m, const T* msk, double srcMul, T* B, hipStream_t st, cpx<T>* X1, cpx<T>* X2,
              cpx<T>* Xz, const T* kern, const cpx<T>* twM, const cpx<T>* twP2, const cpx<T>* tw1,
              const cpx<T>* tw0) {
    const int N0 = d->N[0], N1 = d->N[1], N2 = d->N[2], P1 = d->P[1], P0 = d->P[0], P2 = d->P[2];
    const int H2 = d->H2, H2p = d->H2p, M = d->M;
    if constexpr (sizeof(T) == 8)
        if (d->fold64)
            return run_fused<T>(d, m, msk, srcMul, B, st, X1, d->kt64, d->fold64, d->form64, twM, twP2, tw1, 1, nullptr);
    auto r2c = d->genRd ? nullptr : pick_r2c<T, T>(M);
    auto c2r = d->genRd ? nullptr : pick_c2r<T, T>(M);
    auto f1 = d->gen1d ? nullptr : pick_cols<T, -1>(P1);
    auto i1 = d->gen1d ? nullptr : pick_cols<T, +1>(P1);
    auto zc = d->gen0d ? nullptr : pick_zconv<T, T>(P0);
    if ((!d->genRd && (!r2c || !c2r)) || (!d->gen1d && (!f1 || !i1)) || (!d->gen0d && !zc) || (d->gen0d && !Xz)) {
        hs::set_error(HS_ESIZE, "demag: unsupported FFT length");
        return HS_ESIZE;
    }
    const long nrows = 3L * N0 * N1;
    const Live all{nullptr, 1};
    const cpx<T>* twR = row_table<T>(d, twM, twP2);
    // F1: m .* mask, rows of N2 -> X1 (3, N0, N1, H2p); the mask repeats every N0*N1 rows
    hs::prof_begin(HS_PROF_F1, st);
    if (d->genRd)
        gen::r2c<T>(m, msk, (long)N0 * N1, X1, nrows, N2, P2, H2p, d->gR, twR, twP2, st, all);
    else
        r2c(m, msk, (long)N0 * N1, X1, nrows, N2, H2p, twM, twP2, st);
    hs::prof_end(HS_PROF_F1, st);
    // F2: pencils a = (c, i), rows j < N1 of X1 -> P1 rows of X2
    Geo g1 = {(long)N1 * H2p, 0, H2p, 1};
    Geo g2 = {(long)P1 * H2p, 0, H2p, 1};
    hs::prof_begin(HS_PROF_F2, st);
    if (d->gen1d)
        gen::cols<T, -1>(X1, X2, g1, g2, 3 * N0, N1, P1, H2, d->g1, tw1, st, all);
    else
        f1(X1, X2, g1, g2, 3 * N0, N1, P1, H2, tw1, st);
    hs::prof_end(HS_PROF_F2, st);
    // F3K: axis 0, kernel product, inverse axis 0
    hs::prof_begin(HS_PROF_F3K, st);
    if (d->gen0d)
        gen::zconv<T, T>(X2, Xz, kern, N0, P0, P1, H2, H2p, d->K[1], H2, (T)srcMul, d->g0, tw0, st, 1, all);
    else
        zc(X2, kern, N0, P1, H2, H2p, d->K[1], (T)srcMul, tw0, st);
    hs::prof_end(HS_PROF_F3K, st);
    // I2: P1 rows of X2 -> rows j < N1 of X1
    hs::prof_begin(HS_PROF_I2, st);
    if (d->gen1d)
        gen::cols<T, +1>(X2, X1, g2, g1, 3 * N0, P1, N1, H2, d->g1, tw1, st, all);
    else
        i1(X2, X1, g2, g1, 3 * N0, P1, N1, H2, tw1, st);
    hs::prof_end(HS_PROF_I2, st);
    // I1: C2R rows -> B
    hs::prof_begin(HS_PROF_I1, st);
    if (d->genRd)
        gen::c2r<T>(X1, B, nrows, N2, P2, H2p, d->gR, twR, twP2, st, all);
    else
        c2r(X1, B, nrows, N2, H2p, twM, twP2, st);
    hs::prof_end(HS_PROF_I1, st);
    HS_LAUNCH_CHECK("hs_demag_field");
    return hs_last_error();
}
}  // namespace

namespace {
// static scratch of hs_demag_field_f64_noalloc (below)
constexpr size_t kScratchBytes = size_t(64) << 20;
// FP64 spectra of one solve of the plan's mesh: X1, then X2 and (run-time
// axis-0 length only) Xz, each from a 256-byte boundary; fused: X alone
size_t x_bytes(const hs_demag* d, int rows) { return sizeof(cpx<double>) * 3ull * rows * d->P[1] * d->H2p; }
size_t noalloc_bytes(const hs_demag* d, int fold) {
    if (fold) return sizeof(cpx<double>) * (size_t)fused_spectrum(d, fold);
    const size_t x1 = sizeof(cpx<double>) * 3ull * d->N[0] * d->N[1] * d->H2p;
    return up256(x1) + up256(x_bytes(d, d->N[0])) + (d->gen0d ? x_bytes(d, d->P[0]) : 0);
}
}  // namespace

namespace {
struct KernelBufs {
    const double* oct;            // real-space octant at the logic size
    double* full;                 // 6 P0 P1 P2
    cpx<double>* X;               // 6 P0 P1 H2p
    unsigned long long* maxbits;
};
// FP64 transform of the 6 real components at the plan's lengths, R2C rows, then
// axes 1 and 0 in place (lengths without a compiled family take the
// run-time-length passes), and its octant into k64 and k32 (or null).
void kernel_transform(const hs_demag* d, const KernelBufs& b, double* k64, float* k32, hipStream_t st) {
    const int P0 = d->P[0], P1 = d->P[1], P2 = d->P[2], H2 = d->H2, H2p = d->H2p;
    const long P = (long)P0 * P1 * P2, nk = (long)d->K[0] * d->K[1] * d->K[2];
    const Live all{nullptr, 1};
    hipMemsetAsync(b.maxbits, 0, 2 * kExtractLanes * sizeof(unsigned long long), st);
    hipLaunchKernelGGL(k_kernel_fill, dim3(hs::grid1d(P), 6), dim3(hs::kBlock), 0, st, b.full, b.oct, P0, P1, P2,
                       d->logicK[0], d->logicK[1], d->logicK[2]);
    if (d->genRd)
        gen::r2c<double>(b.full, nullptr, 1, b.X, 6L * P0 * P1, P2, P2, H2p, d->gR,
                         row_table<double>(d, d->twMd, d->twP2d), d->twP2d, st, all);
    else
        pick_r2c<double, double>(d->M)(b.full, nullptr, 1, b.X, 6L * P0 * P1, P2, H2p, d->twMd, d->twP2d, st);
    Geo ga1 = {(long)P1 * H2p, 0, H2p, 1};
    if (d->gen1d)
        gen::cols<double, -1>(b.X, b.X, ga1, ga1, 6 * P0, P1, P1, H2, d->g1, d->tw1d, st, all);
    else
        pick_cols<double, -1>(P1)(b.X, b.X, ga1, ga1, 6 * P0, P1, P1, H2, d->tw1d, st);
    Geo ga0 = {(long)P0 * P1 * H2p, (long)H2p, (long)P1 * H2p, P1};
    if (auto f0 = pick_cols<double, -1>(P0))
        f0(b.X, b.X, ga0, ga0, 6 * P1, P0, P0, H2, d->tw0d, st);
    else
        gen::cols<double, -1>(b.X, b.X, ga0, ga0, 6 * P1, P0, P0, H2, d->g0, d->tw0d, st, all);
    hipLaunchKernelGGL(k_kernel_extract, dim3(hs::grid1d(nk), 6), dim3(hs::kBlock), 0, st, b.X, k64, k32, P0, P1, H2,
                       H2p, d->K[0], d->K[1], d->KP, 1.0 / (double)P, b.maxbits);
}
}  // namespace

// kernel: 0 = Kernel_Arne at `accuracy`, 1 = Newell; pad: transform open axes
// without a compiled family at the next compiled length
static hs_demag* demag_create(const int N[3], const double cell[3], const int pbc[3], int accuracy, int kernel,
                              CUstream stream, bool pad = true) {
    if (!N || !cell || N[0] < 1 || N[1] < 1 || N[2] < 1) {
        hs::set_error(HS_EINVAL, "hs_demag_create: bad mesh");
        return nullptr;
    }
    hipStream_t st = hs::S(stream);
    hs_demag* d = new hs_demag();
    d->cap = 1;
    for (int c = 0; c < 3; c++) {
        d->N[c] = N[c];
        d->pbc[c] = pbc ? pbc[c] : 0;
        d->cell[c] = cell[c];
        d->logic[c] = (N[c] > 1 && d->pbc[c] == 0) ? 2 * N[c] : N[c];
        d->logicK[c] = d->logic[c] / 2 + 1;
    }
    d->ncell = (long)N[0] * N[1] * N[2];
    if (!set_lengths(d, d->logic)) {
        hs::set_error(HS_ESIZE, "hs_demag_create: a padded length (or half the padded x length) exceeds 4095");
        delete d;
        return nullptr;
    }
    d->noalloc = noalloc_bytes(d, 0) <= kScratchBytes;
    if (pad) {
        int P[3];
        padded_lengths(N, d->logic, P);
        set_lengths(d, P);
    }
    const int P0 = d->P[0], P1 = d->P[1], P2 = d->P[2], H2 = d->H2, H2p = d->H2p, M = d->M;
    const bool padded = P0 != d->logic[0] || P1 != d->logic[1] || P2 != d->logic[2];
    const long nk = (long)d->K[0] * d->K[1] * d->K[2];
    bool tables = make_twiddles(d, true);
    // the plan at the logic size: for hs_demag_kernel_f64, and for the FP64 fields where
    // the padded ones would take them from hs_demag_field_f64_noalloc
    std::unique_ptr<hs_demag, decltype(&hs_demag_destroy)> low(padded ? new hs_demag() : nullptr, hs_demag_destroy);
    if (padded) {
        std::copy(d->N, d->N + 3, low->N);
        std::copy(d->logic, d->logic + 3, low->logic);
        std::copy(d->logicK, d->logicK + 3, low->logicK);
        set_lengths(low.get(), d->logic);
        tables = make_twiddles(low.get(), false) && tables;
    }
    const bool low64 = padded && d->noalloc && noalloc_bytes(d, fused_fold<double>(d)) > kScratchBytes;
    hipMalloc(&d->kern64, sizeof(double) * 6 * nk);
    // HS_DEMAG_FORCE asks for particular five-pass variants
    d->fold32 = getenv("HS_DEMAG_FORCE") ? 0 : fused_fold<float>(d);
    d->fold64 = low64 ? 0 : fused_fold<double>(d);
    d->form32 = fused_form<float>(d, d->fold32);
    d->form64 = fused_form<double>(d, d->fold64);
    const long nk32 = (long)d->K[0] * d->K[1] * d->KP;
    if (!d->fold32) hipMalloc(&d->kern32, sizeof(float) * 6 * nk32);
    if (d->kern32) hipMemsetAsync(d->kern32, 0, sizeof(float) * 6 * nk32, st);
    hipMalloc(&d->X1f, sizeof(cpx<float>) * fused_spectrum(d, d->fold32));
    if (!d->fold32) hipMalloc(&d->X2f, sizeof(cpx<float>) * 3L * N[0] * P1 * H2p);
    if (!d->fold32 && d->gen0) hipMalloc(&d->Xzf, sizeof(cpx<float>) * 3L * P0 * P1 * H2p);
    if (d->fold32) hipMalloc(&d->kt32, sizeof(float) * fused_table(d, d->fold32));
    // the FP64 table now where hs_demag_field_f64_noalloc takes the mesh (it cannot allocate), else on first use
    const bool tab64 = d->fold64 && d->noalloc;
    if (tab64) hipMalloc(&d->kt64, sizeof(double) * fused_table(d, d->fold64));
    // ---- Kernel_Arne on the device (FP64), at the logic size
    const int *Lg = d->logic, *LK = d->logicK;
    int r1[3], r2[3];
    for (int c = 0; c < 3; c++) {
        if (d->pbc[c] == 0) {
            r1[c] = -(Lg[c] - 1) / 2;
            r2[c] = (Lg[c] - 1) / 2;
        } else {
            r1[c] = -(Lg[c] * d->pbc[c] - 1);
            r2[c] = (Lg[c] * d->pbc[c] - 1);
        }
    }
    if (Lg[2] == 1 && d->pbc[2] == 0) r2[2] = 0;
    const long noct = (long)LK[0] * LK[1] * LK[2];
    const long P = (long)P0 * P1 * P2;  // no length of `logic` is longer
    // the temporaries in one allocation: each further one of some MB takes up to 0.2 ms to free
    const size_t boct = up256(sizeof(double) * 6 * noct), bfull = up256(sizeof(double) * 6 * P),
                 bX = up256(sizeof(cpx<double>) * 6L * P0 * P1 * H2p);
    unsigned char* tmp = nullptr;
    hipMalloc(&tmp, boct + bfull + bX + 2 * kExtractLanes * sizeof(unsigned long long));
    double* const oct = reinterpret_cast<double*>(tmp);
    double* const full = reinterpret_cast<double*>(tmp + boct);
    cpx<double>* const X = reinterpret_cast<cpx<double>*>(tmp + boct + bfull);
    unsigned long long* const maxbits = reinterpret_cast<unsigned long long*>(tmp + boct + bfull + bX);
    if (padded) hipMalloc(&d->kernL, sizeof(double) * 6 * noct);
    if (!tables || !tmp || !d->kern64 || !d->X1f || (padded && !d->kernL) ||
        (!d->fold32 && (!d->kern32 || !d->X2f || (d->gen0 && !d->Xzf))) || (d->fold32 && !d->kt32) || (tab64 && !d->kt64)) {
        hipFree(tmp);
        hs_demag_destroy(d);
        (void)hipGetLastError();
        if (padded) return demag_create(N, cell, pbc, accuracy, kernel, stream, false);
        hs::set_error(HS_ENOMEM, "hs_demag_create: out of device memory");
        return nullptr;
    }
    hipMemsetAsync(oct, 0, sizeof(double) * 6 * noct, st);
    if (kernel == 1) {
        // far-field switch of the Newell tensor: the FP64 second differences
        // and the cell-averaged dipole have equal error (a few 1e-6 relative)
        // near 35 hmax^0.6 hmin^0.4
        const double hmax = std::max(cell[0], std::max(cell[1], cell[2]));
        const double hmin = std::min(cell[0], std::min(cell[1], cell[2]));
        const double rfar = 35.0 * pow(hmax, 0.6) * pow(hmin, 0.4);
        hipLaunchKernelGGL(k_kernel_newell, dim3(hs::div_up(noct, 64)), dim3(64), 0, st, oct, Lg[0], Lg[1], Lg[2],
                           cell[0], cell[1], cell[2], r1[0], r1[1], r1[2], r2[0], r2[1], r2[2], rfar);
    } else {
        const ArneP ap{Lg[0], Lg[1], Lg[2],   r1[0],   r1[1],   r1[2], r2[0],
                       r2[1], r2[2], cell[0], cell[1], cell[2], (double)(accuracy > 0 ? accuracy : 6)};
        // the list of near cells (at most 3 noct entries) in the memory of `full`, which is filled after it is read
        unsigned* near = reinterpret_cast<unsigned*>(full) + 2;
        hipMemsetAsync(full, 0, sizeof(double), st);
        hipLaunchKernelGGL(k_kernel_arne, dim3(hs::div_up(3 * noct, 64)), dim3(64), 0, st, oct, ap, near, near - 2);
        hipLaunchKernelGGL(k_kernel_arne_near, dim3(1024), dim3(kNearThreads), 0, st, oct, ap, near, near - 2);
    }
    // IsZero (maxwell_convolution.go:227-232): components below 1e-12 of the
    // global max are dropped.
    hipMemsetAsync(maxbits, 0, 6 * sizeof(unsigned long long), st);
    hipLaunchKernelGGL(k_octant_max, dim3(std::min(256, hs::div_up(noct, 256)), 6), dim3(256), 0, st, oct, noct,
                       maxbits);
    double gmax = 0, cmax[6];
    hipMemcpyAsync(cmax, maxbits, sizeof(cmax), hipMemcpyDeviceToHost, st);
    hipStreamSynchronize(st);
    for (int c = 0; c < 6; c++) gmax = fmax(gmax, cmax[c]);
    const KernelBufs kb{oct, full, X, maxbits};
    kernel_transform(d, kb, d->kern64, d->kern32, st);
    if (padded) {
        kernel_transform(low.get(), kb, d->kernL, nullptr, st);
        hipStreamSynchronize(st);
        if (low64) {
            low->kern64 = d->kernL;
            d->f64 = low.release();
        }
    }
    for (int c = 0; c < 6; c++) {
        if (gmax > 0 && cmax[c] / gmax < 1e-12) {
            hipMemsetAsync(d->kern64 + c * nk, 0, sizeof(double) * nk, st);
            if (d->kern32) hipMemsetAsync(d->kern32 + c * nk32, 0, sizeof(float) * nk32, st);
            if (padded) hipMemsetAsync(d->kernL + c * noct, 0, sizeof(double) * noct, st);
        }
    }
    if (d->fold32) fill_table<float>(d, d->kt32, d->fold32, d->form32, st);
    if (tab64) fill_table<double>(d, d->kt64, d->fold64, d->form64, st);
    unsigned long long mb[2 * kExtractLanes];
    hipMemcpyAsync(mb, maxbits, sizeof(mb), hipMemcpyDeviceToHost, st);
    hipStreamSynchronize(st);
    double mi = 0, mr = 0;
    for (int l = 0; l < kExtractLanes; l++) {
        double a, b;
        memcpy(&a, &mb[2 * l], 8);
        memcpy(&b, &mb[2 * l + 1], 8);
        mi = fmax(mi, a);
        mr = fmax(mr, b);
    }
    d->max_imag_ratio = mr > 0 ? mi / mr : 0;
    hipFree(tmp);
    tune32(d, st);
    HS_LAUNCH_CHECK("hs_demag_create");
    if (hs_last_error()) {
        hs_demag_destroy(d);
        return nullptr;
    }
    return d;
}

extern "C" hs_demag* hs_demag_create(const int N[3], const double cell[3], const int pbc[3], int accuracy,
                                     CUstream stream) {
    return demag_create(N, cell, pbc, accuracy, 0, stream);
}

extern "C" hs_demag* hs_demag_create_newell(const int N[3], const double cell[3], const int pbc[3], CUstream stream) {
    return demag_create(N, cell, pbc, 0, 1, stream);
}

extern "C" void hs_demag_destroy(hs_demag* d) {
    if (!d) return;
    if (d->f64) {
        d->f64->kern64 = nullptr;  // d's kernL
        hs_demag_destroy(d->f64);
    }
    void* ps[] = {d->kernL, d->kt32, d->kt64, d->kern64, d->kern32, d->X1f, d->X2f,
                  d->X1d,   d->X2d,  d->Xzf,  d->Xzd,    d->tw};
    for (void* p : ps)
        if (p) hipFree(p);
    delete d;
}

extern "C" int hs_demag_sizes(const hs_demag* d, int P[3], int K[3]) {
    if (!d) return HS_EINVAL;
    for (int c = 0; c < 3; c++) {
        if (P) P[c] = d->logic[c];
        if (K) K[c] = d->logicK[c];
    }
    return 0;
}

extern "C" int hs_demag_kernel_f64(const hs_demag* d, double* host_out) {
    if (!d || !host_out) return HS_EINVAL;
    long nk = (long)d->logicK[0] * d->logicK[1] * d->logicK[2];
    const double* k = d->kernL ? d->kernL : d->kern64;
    const std::shared_ptr<HostStage> stage = HostStage::get();
    // a plan is read once: with no solver alive, fresh buffers cost more than they give
    // up to 29 MB (64^3, 13 MB, 2.5 ms against the runtime's 0.75; 256x256x8, 29 MB, 0.9
    // or, where their pages are pinned anew, 2.8 against 1.6; 256x256x16, 53 MB, 1.9
    // against 5.2)
    const hipError_t e = stage ? stage->out(host_out, k, sizeof(double) * 6 * nk, nullptr, size_t(48) << 20)
                               : hipMemcpy(host_out, k, sizeof(double) * 6 * nk, hipMemcpyDeviceToHost);
    return e == hipSuccess ? 0 : (int)e;
}

extern "C" double hs_demag_max_imag_ratio(const hs_demag* d) { return d ? d->max_imag_ratio : -1; }

extern "C" int hs_demag_variant_count(const hs_demag* d, int* out3) {
    if (!d || !out3) return HS_EINVAL;
    out3[0] = d->genR ? 0 : (int)hsdm::variants(d->M).rows.size();
    out3[1] = d->gen1 ? 0 : (int)hsdm::variants(d->P[1]).cols.size();
    out3[2] = d->gen0 ? 0 : (int)hsdm::variants(d->P[0]).z.size();
    return 0;
}

extern "C" int hs_demag_form(const hs_demag* d, int out2[2]) {
    if (!d || !out2) return HS_EINVAL;
    out2[0] = d->fold32;
    out2[1] = d->fold64;
    return 0;
}

extern "C" int hs_demag_tiles(const hs_demag* d, int* out6) {
    if (!d || !out6) return HS_EINVAL;
    out6[0] = d->row32.W;
    out6[1] = d->row32.NT;
    out6[2] = d->col32.W;
    out6[3] = d->col32.NT;
    out6[4] = d->z32.W;
    out6[5] = d->z32.NT;
    return 0;
}

extern "C" int hs_demag_field_f32(hs_demag* d, const float* m, const float* msk, double msat0T0Mul, float* B,
                                  CUstream stream) {
    if (!d || !m || !B) {
        hs::set_error(HS_EINVAL, "hs_demag_field_f32");
        return HS_EINVAL;
    }
    return run_field32(d, m, msk, HS_MU0 * msat0T0Mul, B, hs::S(stream));
}

extern "C" int hs_demag_field_f64(hs_demag* d, const double* m, const double* msk, double msat0T0Mul, double* B,
                                  CUstream stream) {
    if (!d || !m || !B) {
        hs::set_error(HS_EINVAL, "hs_demag_field_f64");
        return HS_EINVAL;
    }
    if (d->f64) d = d->f64;
    if (!d->X1d) {
        hipMalloc(&d->X1d, sizeof(cpx<double>) * fused_spectrum(d, d->fold64));
        if (!d->fold64) hipMalloc(&d->X2d, sizeof(cpx<double>) * 3L * d->N[0] * d->P[1] * d->H2p);
        if (!d->fold64 && d->gen0d) hipMalloc(&d->Xzd, sizeof(cpx<double>) * 3L * d->P[0] * d->P[1] * d->H2p);
        const bool tab = d->fold64 && !d->kt64;
        if (tab) hipMalloc(&d->kt64, sizeof(double) * fused_table(d, d->fold64));
        if (!d->X1d || (!d->fold64 && (!d->X2d || (d->gen0d && !d->Xzd))) || (d->fold64 && !d->kt64)) {
            void* ps[] = {d->X1d, d->X2d, d->Xzd};
            for (void* p : ps)
                if (p) hipFree(p);
            d->X1d = d->X2d = d->Xzd = nullptr;
            if (tab && d->kt64) {
                hipFree(d->kt64);
                d->kt64 = nullptr;
            }
            hs::set_error(HS_ENOMEM, "hs_demag_field_f64: out of device memory");
            return HS_ENOMEM;
        }
        if (tab) {  // ready for calls on any stream
            fill_table<double>(d, d->kt64, d->fold64, d->form64, hs::S(stream));
            hipStreamSynchronize(hs::S(stream));
        }
    }
    return run_field<double>(d, m, msk, HS_MU0 * msat0T0Mul, B, hs::S(stream), d->X1d, d->X2d, d->Xzd, d->kern64,
                             d->twMd, d->twP2d, d->tw1d, d->tw0d);
}

// ---- FP64 field without allocation: spectra in a static device array
// `scratch` holds X1 (3, N0, N1, H2p) and, from the next 256-byte boundary,
// X2 (3, N0, P1, H2p) in FP64 complex.  Every call on one GPU uses that GPU's
// copy of the array, so calls that overlap on one GPU (two streams, two host
// threads) race.  No pass reads a spectrum element that the same call has
// not written first, so the contents left by an earlier call do not matter.
namespace {
constexpr int kMaxDevices = 64;
}  // namespace
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {
std::mutex g_scratch_mu;
void* g_scratch[kMaxDevices] = {};

// Device address of the current device's `scratch` (the array's name is a
// host-side stand-in that kernels must never receive).  Looked up once per
// device with that device current.
void* scratch_address() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return nullptr;
        g_scratch[dev] = p;
    }
    return g_scratch[dev];
}

}  // namespace

extern "C" int hs_demag_field_f64_noalloc(hs_demag* d, const double* m, const double* msk, double msat0T0Mul,
                                          double* B, CUstream stream) {
    if (!d || !m || !B) {
        hs::set_error(HS_EINVAL, "hs_demag_field_f64_noalloc");
        return HS_EINVAL;
    }
    if (!d->noalloc) {
        hs::set_error(HS_ESIZE, "hs_demag_field_f64_noalloc: the mesh's FP64 spectra exceed the 64 MiB static "
                                "scratch; use hs_demag_field_f64");
        return HS_ESIZE;
    }
    if (d->f64) d = d->f64;
    unsigned char* base = static_cast<unsigned char*>(scratch_address());
    if (!base) {
        hs::set_error(HS_EINVAL, "hs_demag_field_f64_noalloc: no device address for the static scratch");
        return HS_EINVAL;
    }
    const size_t x1 = up256(sizeof(cpx<double>) * 3ull * d->N[0] * d->N[1] * d->H2p);
    cpx<double>* X1 = reinterpret_cast<cpx<double>*>(base);
    cpx<double>* X2 = reinterpret_cast<cpx<double>*>(base + x1);
    cpx<double>* Xz = d->gen0d ? reinterpret_cast<cpx<double>*>(base + x1 + up256(x_bytes(d, d->N[0]))) : nullptr;
    return run_field<double>(d, m, msk, HS_MU0 * msat0T0Mul, B, hs::S(stream), X1, X2, Xz, d->kern64, d->twMd,
                             d->twP2d, d->tw1d, d->tw0d);
}

// Internal entry for the solver: FP32 field of a batch of nsolve solves
// (layout [solve][3][cells]) with an FP32 mask; live = per-solve flags or null.
int hs_demag_field_f32_internal(hs_demag* d, const float* m, const float* msk, double msat0T0Mul, float* B,
                                hipStream_t st, int nsolve, const int* live) {
    return run_field32(d, m, msk, HS_MU0 * msat0T0Mul, B, st, nsolve, live);
}

// Grow the FP32 spectrum buffers to hold `nsolve` solves of this mesh.
extern "C" int hs_demag_reserve(hs_demag* d, int nsolve) {
    if (!d || nsolve < 1) return HS_EINVAL;
    if (nsolve <= d->cap) return 0;
    cpx<float>*X1 = nullptr, *X2 = nullptr, *Xz = nullptr;
    hipMalloc(&X1, sizeof(cpx<float>) * fused_spectrum(d, d->fold32) * nsolve);
    if (!d->fold32) hipMalloc(&X2, sizeof(cpx<float>) * 3L * d->N[0] * d->P[1] * d->H2p * nsolve);
    if (!d->fold32 && d->gen0) hipMalloc(&Xz, sizeof(cpx<float>) * 3L * d->P[0] * d->P[1] * d->H2p * nsolve);
    if (!X1 || (!d->fold32 && (!X2 || (d->gen0 && !Xz)))) {
        hipFree(X1);
        hipFree(X2);
        hipFree(Xz);
        hs::set_error(HS_ENOMEM, "hs_demag_reserve: out of device memory");
        return HS_ENOMEM;
    }
    hipFree(d->X1f);
    hipFree(d->X2f);
    hipFree(d->Xzf);
    d->X1f = X1;
    d->X2f = X2;
    d->Xzf = Xz;
    d->cap = nsolve;
    return 0;
}
long hs_demag_ncell(const hs_demag* d) { return d->ncell; }
// device bytes of the plan: kernel octant (FP64; FP32 for the five passes) and
// tables, FP32 spectra of `cap` solves, FP64 spectra when allocated, twiddle tables
long hs_demag_footprint(const hs_demag* d) {
    const long nk = (long)d->K[0] * d->K[1] * d->K[2];
    long b = 6 * nk * (long)sizeof(double);
    if (d->kern32) b += 6L * d->K[0] * d->K[1] * d->KP * (long)sizeof(float);
    if (d->X1f)
        b += (long)sizeof(cpx<float>) *
             (fused_spectrum(d, d->fold32) + (d->X2f ? 3L * d->N[0] * d->P[1] * d->H2p : 0)) * d->cap;
    if (d->f64)
        b += hs_demag_footprint(d->f64);  // with its kern64, d's kernL
    else if (d->kernL)
        b += 6L * d->logicK[0] * d->logicK[1] * d->logicK[2] * (long)sizeof(double);
    if (d->kt32) b += fused_table(d, d->fold32) * (long)sizeof(float);
    if (d->kt64) b += fused_table(d, d->fold64) * (long)sizeof(double);
    if (d->X1d)
        b += (long)sizeof(cpx<double>) * (fused_spectrum(d, d->fold64) + (d->X2d ? 3L * d->N[0] * d->P[1] * d->H2p : 0));
    if (d->Xzf) b += (long)sizeof(cpx<float>) * 3L * d->P[0] * d->P[1] * d->H2p * d->cap;
    if (d->Xzd) b += (long)sizeof(cpx<double>) * 3L * d->P[0] * d->P[1] * d->H2p;
    b += (long)(sizeof(cpx<float>) + sizeof(cpx<double>)) * (d->M + d->P[2] + d->P[1] + d->P[0]);
    return b;
}
