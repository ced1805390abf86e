// mac_inputs.hip -- gfx950 kernels producing the MAC projection's inputs:
//   cell_to_edge  Source/cell_to_edge.f90:14-68        (beta0 on radial edges)
//   make_macrhs   Source/make_macrhs.f90:24-342        (the projection's macrhs)
//   make_s0mac    Source/fill_3d_data.f90:942-1075     (spherical beta0 on faces,
//                 s0mac_interp_type 1, with put_1d_array_on_cart_3d_sphr
//                 :269-533 for the cell values)
// Each is one streaming pass over the per-box arrays (Fortran order with the
// caller's ghost widths), with the reference's expression order.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mac_launch.h"

namespace mac {

static constexpr int ITPB = 256;

__device__ __forceinline__ long box_index(const BoxDev &B, int ng, int fd, int dim, int i, int j, int k)
{
    const long ex = B.hi[0] - B.lo[0] + 1 + 2 * ng + (fd == 0);
    const long ey = B.hi[1] - B.lo[1] + 1 + 2 * ng + (fd == 1);
    const long li = i - B.lo[0] + ng, lj = j - B.lo[1] + ng;
    const long lk = (dim == 3) ? (k - B.lo[2] + ng) : 0;
    return li + ex * (lj + ey * lk);
}

// ---------------------------------------------------------- cell_to_edge
__global__ void __launch_bounds__(ITPB) k_cell_to_edge(const double *__restrict__ c, int nr, double *__restrict__ e)
{
    for (int r = blockIdx.x * ITPB + threadIdx.x; r <= nr; r += gridDim.x * ITPB) {
        double v;
        if (r == 0) {
            v = c[0];
        } else if (r == 1) {
            v = 0.5 * (c[r - 1] + c[r]);
        } else if (r == nr) {
            v = c[r - 1];
        } else if (r == nr - 1) {
            v = 0.5 * (c[r] + c[r - 1]);
        } else {
            const double tmp = 7.0 / 12.0 * (c[r] + c[r - 1]) - 1.0 / 12.0 * (c[r + 1] + c[r - 2]);
            const double lo = fmin(c[r], c[r - 1]), hi = fmax(c[r], c[r - 1]);
            v = fmin(fmax(tmp, lo), hi);
        }
        e[r] = v;
    }
}

void launch_cell_to_edge(const double *c, int nr, double *e, hipStream_t s)
{
    hipLaunchKernelGGL(k_cell_to_edge, dim3((nr + ITPB) / ITPB), dim3(ITPB), 0, s, c, nr, e);
}

// ------------------------------------- 1-D radial profile on a 3D cell
// put_1d_array_on_cart_3d_sphr for a bin-centred, scalar profile: type 1
// piecewise constant, 2 piecewise linear, 3 quadratic (quad_interp,
// fill_3d_data.f90:535-546, limited to the range of its three points)
// What the interpolation takes from the cell's place (at), shared by the
// profiles interpolated there, and a profile's value (of).  Divisors are few (dr
// and differences of radii near it), so quotients are formed from their
// reciprocals (quot), five or six operations for a division's eleven or more.
struct SphrAt {
    int i0, i1, i2;
    bool one;           // s0[i0] itself
    double w0, w1;      // interp 2: weights of i0, i1; 3: radius - x0, radius - x1
    double d0, d1, d2;  // x1 - x0, x2 - x1, x2 - x0
    double r0, r1, r2;  // their reciprocals
};

// whether quot(n, d, r) is n / d: its correction steps round correctly while
// nothing under- or overflows, d being a radial spacing within 1e-40 .. 1e40
// (spacing_recip gives 0 for one outside)
__device__ __forceinline__ bool quot_range(double n)
{
    const double m = fabs(n);
    return (m > 1e-200 && m < 1e200) || n == 0.0;
}
__device__ __forceinline__ double spacing_recip(double d)
{
    return d > 1e-40 && d < 1e40 ? 1.0 / d : 0.0;
}

__device__ __forceinline__ SphrAt sphr_at(const SphrGeom &G, double x, double y, double z, double rdr)
{
    SphrAt A;
    const double radius = sqrt(x * x + y * y + z * z);
    const double dr = G.dr;
    const int nr = G.nr;
    int index = (int)(rdr != 0.0 && quot_range(radius) ? quot(radius, dr, rdr) : radius / dr);
    A.one = true;
    A.i0 = A.i1 = A.i2 = index;
    if (G.interp == 1) return A;
    if (G.interp == 2) {
        const double rc = ((double)index + 0.5) * dr;
        if (radius >= rc) {
            if (index >= nr - 1) {
                A.i0 = nr - 1;
                return A;
            }
            const double rc1 = ((double)(index + 1) + 0.5) * dr;
            A.i0 = index + 1;
            A.w0 = radius - rc;
            A.i1 = index;
            A.w1 = rc1 - radius;
        } else {
            if (index == 0) return A;
            if (index > nr - 1) {
                A.i0 = nr - 1;
                return A;
            }
            const double rcm = ((double)(index - 1) + 0.5) * dr;
            A.i0 = index;
            A.w0 = radius - rcm;
            A.i1 = index - 1;
            A.w1 = rc - radius;
        }
        A.one = false;
        A.d0 = dr;
        A.r0 = rdr;
        return A;
    }
    if (index == 0) index = 1;
    else if (index >= nr - 1) index = nr - 2;
    const double x0 = ((double)(index - 1) + 0.5) * dr, x1 = ((double)index + 0.5) * dr,
                 x2 = ((double)(index + 1) + 0.5) * dr;
    A.i0 = index - 1;
    A.i1 = index;
    A.i2 = index + 1;
    A.one = false;
    A.w0 = radius - x0;
    A.w1 = radius - x1;
    A.d0 = x1 - x0;
    A.d1 = x2 - x1;
    A.d2 = x2 - x0;
    A.r0 = spacing_recip(A.d0);
    A.r1 = spacing_recip(A.d1);
    A.r2 = spacing_recip(A.d2);
    return A;
}

// DIV: by division, what the other form takes where a quotient's operands are
// out of quot's range (one test per profile: no branch between its quotients)
template <bool DIV = false>
__device__ __forceinline__ double sphr_of(const SphrGeom &G, const SphrAt &A, const double *__restrict__ s0)
{
    const double y0 = s0[A.i0];
    if (A.one) return y0;
    bool ok = true;
    auto ratio = [&](double n, double d, double r) {
        if constexpr (DIV) return n / d;
        ok = ok && r != 0.0 && quot_range(n);
        return quot(n, d, r);
    };
    const double y1 = s0[A.i1];
    double v;
    if (G.interp == 2) {
        v = ratio(y0 * A.w0, A.d0, A.r0) + ratio(y1 * A.w1, A.d0, A.r0);
    } else {
        const double y2 = s0[A.i2];
        const double q = ratio(y1 - y0, A.d0, A.r0);
        v = y0 + q * A.w0 + ratio(ratio(y2 - y1, A.d1, A.r1) - q, A.d2, A.r2) * A.w0 * A.w1;
        const double mx = fmax(fmax(y0, y1), y2), mn = fmin(fmin(y0, y1), y2);
        if (v > mx) v = mx;
        if (v < mn) v = mn;
    }
    if constexpr (!DIV) {
        if (!ok) v = sphr_of<true>(G, A, s0);
    }
    return v;
}
__device__ __forceinline__ double sphr_x(const SphrGeom &G, int d, int i)
{
    return G.prob_lo[d] + ((double)i + 0.5) * G.dx[d] - G.center[d];
}

// ----------------------------------------------------------- make_macrhs
// One thread per column (i, j) of box blockIdx.y's valid cells and chunk of
// `planes` planes; blockIdx.x is a tile of NT columns and a chunk, the tiles first
// (with the chunks outermost of all a 256^3 planar call takes 310 us for 294).
// TAB: the radial profiles are copied to LDS first.  A row of cells reaches over
// as many cache lines of a profile as it has bins across, and a cell takes 15
// such gathers (five quadratic profiles).  Bound by the interpolations' FP64
// instructions and their latency: 256^3 cells, six arrays of 0.13 GB, take 255
// us; with the profiles in memory, a branch per quotient and the streams' loads
// after the interpolation 326, with a division per quotient and 64-bit index
// divisions per cell 336.  Blocks of 512 threads (three to a CU with 44 KB of
// profiles) 255, of 1024 (one) 269.
template <int DIM, bool SPH, bool TAB>
__global__ void __launch_bounds__(TAB ? 512 : ITPB) k_make_macrhs(MacrhsArgs A, int planes, int tiles)
{
    constexpr int NT = TAB ? 512 : ITPB;
    const int b = blockIdx.y;
    const BoxDev B = A.boxes[b];
    const int ex = B.hi[0] - B.lo[0] + 1, ey = B.hi[1] - B.lo[1] + 1;
    const int ez = (DIM == 3) ? B.hi[2] - B.lo[2] + 1 : 1;
    int chunk, p;
    if constexpr (SPH && !TAB) {   // small domains: no lanes left over at a chunk's end
        const int q = blockIdx.x * NT + threadIdx.x;
        chunk = q / (ex * ey);
        p = q - chunk * (ex * ey);
    } else {
        chunk = blockIdx.x / tiles;
        p = ((int)blockIdx.x - chunk * tiles) * NT + threadIdx.x;
    }
    const int k0 = chunk * planes, k1 = min(k0 + planes, ez);
    if (k0 >= ez) return;
    extern __shared__ double tab[];
    const int nr = A.geo.nr;
    if constexpr (TAB) {
        const int np = A.dpdt_on ? 5 : 2;
        for (int q = threadIdx.x; q < nr; q += NT) {
            tab[q] = A.beta0[q];
            tab[nr + q] = A.Sbar[q];
            if (np == 5) {
                tab[2 * nr + q] = A.gamma1bar[q];
                tab[3 * nr + q] = A.p0[q];
                tab[4 * nr + q] = A.rho0[q];
            }
        }
        __syncthreads();
    }
    if (p >= ex * ey) return;
    const int lj = p / ex, li = p - lj * ex;
    const int i = B.lo[0] + li, j = B.lo[1] + lj;
    const int J = j - A.dlo[1];
    double x = 0.0, y = 0.0, rdr = 0.0;
    if constexpr (SPH) {
        x = sphr_x(A.geo, 0, i - A.dlo[0]);
        y = sphr_x(A.geo, 1, J);
        rdr = spacing_recip(A.geo.dr);
    }
    const double *__restrict__ pS = A.S[b], *__restrict__ pdg = A.dg[b];
    const double *__restrict__ pdp = A.dpdt_on ? A.dp[b] : nullptr;
    double *__restrict__ pchi = A.dpdt_on ? A.dchi[b] : nullptr, *__restrict__ prhs = A.rhs[b];
    for (int l = k0; l < k1; ++l) {
        const int k = (DIM == 3) ? B.lo[2] + l : 0, K = (DIM == 3) ? k - A.dlo[2] : 0;
        // the streams' loads before the interpolation
        const double S = pS[box_index(B, A.ng_S, -1, DIM, i, j, k)];
        const double dg = pdg[box_index(B, A.ng_dg, -1, DIM, i, j, k)];
        double *dchi = nullptr, c = 0.0;
        if (A.dpdt_on) {
            dchi = pchi + box_index(B, A.ng_dchi, -1, DIM, i, j, k);
            if (!A.predictor) c = *dchi;
        }
        double b0, sb, g1 = 0.0, pp = 0.0;
        bool below;
        if constexpr (SPH) {
            const SphrAt at = sphr_at(A.geo, x, y, sphr_x(A.geo, 2, K), rdr);
            b0 = sphr_of(A.geo, at, TAB ? tab : A.beta0);
            sb = sphr_of(A.geo, at, TAB ? tab + 1 * nr : A.Sbar);
            double r0 = 0.0;
            if (A.dpdt_on) {
                g1 = sphr_of(A.geo, at, TAB ? tab + 2 * nr : A.gamma1bar);
                pp = sphr_of(A.geo, at, TAB ? tab + 3 * nr : A.p0);
                r0 = sphr_of(A.geo, at, TAB ? tab + 4 * nr : A.rho0);
            }
            below = r0 > A.cutoff_density;
        } else {
            const int r = (DIM == 3) ? K : J;
            b0 = A.beta0[r];
            sb = A.Sbar[r];
            if (A.dpdt_on) {
                g1 = A.gamma1bar[r];
                pp = A.p0[r];
            }
            below = r < A.cutoff_coord;
        }
        double v = b0 * (S - sb + dg);
        if (A.dpdt_on) {
            if (below) {
                const double dp = pdp[box_index(B, A.ng_dp, -1, DIM, i, j, k)];
                c = c + A.dpdt * dp / (A.dt * g1 * pp);
                v = v + b0 * c;
            }
            *dchi = c;
        }
        prhs[box_index(B, A.ng_rhs, -1, DIM, i, j, k)] = v;
    }
}

// the reference zeroes a predictor's delta_chi over the whole array, ghost
// cells included; the kernel above covers the valid cells
__global__ void __launch_bounds__(ITPB) k_zero_ghosts(MacrhsArgs A, int dim)
{
    const int b = blockIdx.y;
    const BoxDev B = A.boxes[b];
    const int ng = A.ng_dchi;
    const long ex = B.hi[0] - B.lo[0] + 1 + 2 * ng, ey = B.hi[1] - B.lo[1] + 1 + 2 * ng;
    const long ez = (dim == 3) ? B.hi[2] - B.lo[2] + 1 + 2 * ng : 1;
    for (long q = (long)blockIdx.x * ITPB + threadIdx.x; q < ex * ey * ez; q += (long)gridDim.x * ITPB) {
        const long li = q % ex, lj = (q / ex) % ey, lk = q / (ex * ey);
        const bool ghost = li < ng || li >= ex - ng || lj < ng || lj >= ey - ng ||
                           (dim == 3 && (lk < ng || lk >= ez - ng));
        if (ghost) A.dchi[b][q] = 0.0;
    }
}

// Planes of a chunk (spherical): as many as leave some 2048 blocks of 512
// threads, 16 at most (cells: of all boxes).  A thread's planes follow each other in a chain of square
// roots and interpolations, so a small domain wants them side by side, and the
// profiles from memory (a block of few cells does not repay the copy).  Calls in
// microseconds, by planes 1, 2, 4, 8, 16: 64^3 50, 50, 55, 63, 82 (profiles in memory,
// blocks of 256: 50, 51, 54, 63, 80), 96^3 77, 76, 77, 79, 98 (75, 74, 77, 82, 96), 128^3
// 96, 92, 90, 92, 99 (94, 91, 92, 96, 109), 256^3 467, 420, 398, 386, 387 (476 .. 486).
// A planar cell is a few loads and little else: one plane a chunk at every size.
void launch_make_macrhs(const MacrhsArgs &A, const int maxext[3], long cells, bool sph, hipStream_t s)
{
    const long cols = (long)maxext[0] * maxext[1];
    auto go = [&](auto k, int nt, size_t lds, int planes) {
        const long tiles = (cols + nt - 1) / nt;   // enough for either order
        const dim3 g((unsigned)(tiles * ((maxext[2] + planes - 1) / planes)), A.nboxes);
        hipLaunchKernelGGL(k, g, dim3(nt), lds, s, A, planes, (int)tiles);
    };
    if (A.dim == 3 && sph) {
        const long blocks = cells / 512;   // at one plane a chunk
        const int planes = blocks <= 1024 ? 1 : (int)std::max(2L, std::min(16L, (blocks + 2047) / 2048));
        // two blocks or more to a CU
        const size_t lds = sizeof(double) * (size_t)A.geo.nr * (A.dpdt_on ? 5 : 2);
        if (blocks > 2048 && lds <= 64 * 1024) go(k_make_macrhs<3, true, true>, 512, lds, planes);
        else go(k_make_macrhs<3, true, false>, ITPB, 0, planes);
    } else if (A.dim == 3) {
        go(k_make_macrhs<3, false, false>, ITPB, 0, 1);
    } else {
        go(k_make_macrhs<2, false, false>, ITPB, 0, 1);
    }
    if (A.dpdt_on && A.predictor && A.ng_dchi > 0)
        hipLaunchKernelGGL(k_zero_ghosts, dim3(64, A.nboxes, 1), dim3(ITPB), 0, s, A, A.dim);
}

// ------------------------------------------------------------ make_s0mac
// Box blockIdx.y's face arrays of the three directions (one ghost layer: every
// face of the grown box), each face the mean of its two cells, the cells
// clamped into the domain (first-order extrapolation outside it).  A block of
// NT threads marches a tile of R rows of W columns through `planes` planes, one
// thread per column: it interpolates the profile on its cell, gives the value to
// its neighbours in x and y through LDS and keeps it for the face above; the
// first row, column and plane only lead in.  W covers a whole row of the box up
// to 80 faces: long runs to write, and few of the threads only leading in.
//
// Bound by the interpolation and the faces' writes about equally: 256^3 cells
// (boxes of 64^3, 0.45 GB of faces) take 155 us; a pass for the cells (110 us)
// and one for the faces took 330.  TAB: the profile is copied to LDS (157 us
// and 163 without).
static constexpr int S0_ROW = 80;
template <bool TAB, int NT>
__global__ void __launch_bounds__(NT) k_make_s0mac(S0macArgs A, int planes)
{
    const int b = blockIdx.y;
    const BoxDev B = A.boxes[b];
    const int n[3] = {B.hi[0] - B.lo[0] + 1, B.hi[1] - B.lo[1] + 1, B.hi[2] - B.lo[2] + 1};
    // faces: n + 3 along their direction, n + 2 along the others
    const int nseg = (n[0] + 3 + S0_ROW - 1) / S0_ROW, w = (n[0] + 3 + nseg - 1) / nseg, W = w + 1;
    const int R = NT / W, rows = R - 1;
    const int nrow = (n[1] + 3 + rows - 1) / rows;
    const int tile = blockIdx.x;
    if (tile >= nseg * nrow) return;
    const int k0 = blockIdx.z * planes, k1 = min(k0 + planes, n[2] + 3);
    if (k0 >= n[2] + 3) return;
    extern __shared__ double tab[];   // the profile
    if constexpr (TAB) {
        for (int q = threadIdx.x; q < A.geo.nr; q += NT) tab[q] = A.s0[q];
        __syncthreads();
    }
    const int tr = tile / nseg, ts = tile - tr * nseg;
    const int r = threadIdx.x / W, m = threadIdx.x - r * W;
    // face (li, lj, k) of the grown box's arrays; cell g of the domain
    const int li = ts * w + m - 1, lj = tr * rows + r - 1;
    const bool live = r < R;
    auto clamp = [&](int d, int l) {
        const int g = B.lo[d] - 1 + l - A.dlo[d];
        return g < 0 ? 0 : (g > A.n[d] - 1 ? A.n[d] - 1 : g);
    };
    const double x = sphr_x(A.geo, 0, clamp(0, li)), y = sphr_x(A.geo, 1, clamp(1, lj));
    const double rdr = spacing_recip(A.geo.dr);
    const bool own = live && m > 0 && r > 0 && li < n[0] + 3 && lj < n[1] + 3;
    const bool wx = own && lj < n[1] + 2, wy = own && li < n[0] + 2, wz = wx && wy;
    double *__restrict__ fx = A.out[b * 3], *__restrict__ fy = A.out[b * 3 + 1], *__restrict__ fz = A.out[b * 3 + 2];
    const long ox = li + (long)(n[0] + 3) * lj, px = (long)(n[0] + 3) * (n[1] + 2);
    const long oy = li + (long)(n[0] + 2) * lj, py = (long)(n[0] + 2) * (n[1] + 3);
    const long pz = (long)(n[0] + 2) * (n[1] + 2);
    __shared__ double v[2][NT];
    const int t = threadIdx.x;
    double below = 0.0;
    for (int k = k0 - 1; k < k1; ++k) {
        const double c = sphr_of(A.geo, sphr_at(A.geo, x, y, sphr_x(A.geo, 2, clamp(2, k)), rdr), TAB ? tab : A.s0);
        v[k & 1][t] = c;
        __syncthreads();
        if (k >= k0) {
            if (k < n[2] + 2) {
                if (wx) fx[ox + px * k] = 0.5 * (c + v[k & 1][t - 1]);
                if (wy) fy[oy + py * k] = 0.5 * (c + v[k & 1][t - W]);
            }
            if (wz) fz[oy + pz * k] = 0.5 * (c + below);
        }
        below = c;
    }
}

// the most tiles of any box: a narrow box has fewer, longer ones in x and more
// rows to a tile
static long s0_tiles(const int maxext[3], int nt)
{
    long tiles = 0;
    for (int e = 1; e <= maxext[0]; ++e) {
        const int nseg = (e + 3 + S0_ROW - 1) / S0_ROW, W = (e + 3 + nseg - 1) / nseg + 1, rows = nt / W - 1;
        tiles = std::max(tiles, (long)nseg * ((maxext[1] + 3 + rows - 1) / rows));
    }
    return tiles;
}

// Planes of a chunk: as many as leave some 800 blocks of 512 threads, 16 at most
// (one more plane leads in).  Blocks of 1024 threads for chunks of 16 planes where
// their tiles fit the boxes as well.  Calls in microseconds, by planes 1, 2, 4, 8,
// 16: 64^3 35, 33, 33, 37, 45 (blocks of 1024: 35, 33, 36, 43, 56), 128^3 85, 70,
// 64, 59, 65, 256^3 in boxes of 64 455, 341, 291, 259, 246 (1024: 434 .. 234), of
// 32 978, 861, 804, 778, 774 (1141 .. 818).
void launch_make_s0mac(const S0macArgs &A, const int maxext[3], hipStream_t s)
{
    const long t512 = s0_tiles(maxext, 512), t1024 = s0_tiles(maxext, 1024);
    const int nz = maxext[2] + 3;
    const int planes = (int)std::min(16L, (t512 * nz * A.nboxes + 799) / 800);
    const size_t lds = sizeof(double) * (size_t)A.geo.nr;
    auto go = [&](auto k, long tiles, int nt, size_t bytes) {
        const dim3 g((unsigned)tiles, A.nboxes, (unsigned)((nz + planes - 1) / planes));
        hipLaunchKernelGGL(k, g, dim3(nt), bytes, s, A, planes);
    };
    const bool tab = lds <= 48 * 1024;
    if (planes == 16 && 2 * t1024 <= t512)
        tab ? go(k_make_s0mac<true, 1024>, t1024, 1024, lds) : go(k_make_s0mac<false, 1024>, t1024, 1024, 0);
    else
        tab ? go(k_make_s0mac<true, 512>, t512, 512, lds) : go(k_make_s0mac<false, 512>, t512, 512, 0);
}

}  // namespace mac
