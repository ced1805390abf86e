// mac_legs.hip -- the small levels of the multigrid cycle for gfx950.
//
// A level of some 10^5 cells is bound by latency: a kernel on it takes 4 to 7
// microseconds however little it does (start-up, one round trip to memory,
// drain), and a V-cycle made of single sweeps runs seven or more of them on
// each level.  Two forms replace them:
//   k_leg_down / k_leg_up   one level's way down (two red-black sweeps,
//       residual, restriction) or up (prolongation, two sweeps) in one launch.
//       A block holds a tile and a halo of 4 cells and repeats the halo's
//       updates, so that blocks need nothing from each other;
//   k_coarse                the cycle from the first level of at most 4096
//       cells down to the bottom solve, in one workgroup.
// Both keep the iterate in LDS split by colour.  A thread owns pairs of cells
// (2m, 2m+1) of a row, one red and one black: with the colours apart, the five
// neighbours that a cell takes from LDS lie at consecutive addresses over
// the lanes (no bank conflicts, 4 or 8 bytes a lane), the sixth is the pair's
// other cell in a register, and no lane idles in either colour.  The face
// weights, the diagonal and its reciprocal stay in registers.
//
// The arithmetic is that of the single operators (stencil, gs_value,
// apply_value, prolong_value of mac_internal.h) in the same order, so the
// results agree with them bit for bit.
#include <algorithm>

#include "mac_launch.h"

namespace mac {

// ---------------------------------------------------------------- helpers
template <typename T>
struct __align__(2 * sizeof(T)) Two {
    T a, b;
};

template <typename T>
__device__ __forceinline__ Two<T> load2(const T *p)
{
    return *reinterpret_cast<const Two<T> *>(p);
}

template <typename T>
__device__ __forceinline__ void store2(T *p, T a, T b)
{
    *reinterpret_cast<Two<T> *>(p) = Two<T>{a, b};
}

// n / d from r = 1 / d (both correctly rounded): a product and two correction
// steps, after which the quotient is the correctly rounded one (P. Markstein,
// IBM J. Res. Dev. 34 (1990) 111-119) away from under- and overflow, the value
// that the division of gs_value gives.  A cell is updated four times with one
// diagonal; five operations replace the division's eleven in FP64.
template <typename T>
__device__ __forceinline__ T quot(T n, T d, T r)
{
    T q = n * r;
    q = dfma(dfma(-d, q, n), r, q);
    return dfma(dfma(-d, q, n), r, q);
}

// numerator and denominator of gs_value
template <int DIM, typename T>
__device__ __forceinline__ T gs_num(const Lev<T> &L, const T *w, const T *p, T rhs)
{
    const T tx = dfma(w[0], p[0], w[1] * p[1]);
    const T ty = dfma(w[2], p[2], w[3] * p[3]);
    if constexpr (DIM == 3) {
        const T tz = dfma(w[4], p[4], w[5] * p[5]);
        return dfma(L.ih2x, tx, dfma(L.ih2y, ty, dfma(L.ih2z, tz, rhs)));
    } else {
        return dfma(L.ih2x, tx, dfma(L.ih2y, ty, rhs));
    }
}
template <int DIM, typename T>
__device__ __forceinline__ T gs_den(const Lev<T> &L, const T *w, T a)
{
    const T sx = w[0] + w[1], sy = w[2] + w[3];
    if constexpr (DIM == 3) return dfma(L.ih2x, sx, dfma(L.ih2y, sy, L.ih2z * (w[4] + w[5]))) + a;
    else return dfma(L.ih2x, sx, L.ih2y * sy) + a;
}
// A phi (apply_value) from 2 DIM weights
template <int DIM, typename T>
__device__ __forceinline__ T apply_w(const Lev<T> &L, const T *w, const T *p, T pc)
{
    T w6[6], p6[6];
#pragma unroll
    for (int s = 0; s < 6; ++s) {
        w6[s] = s < 2 * DIM ? w[s] : T(0);
        p6[s] = s < 2 * DIM ? p[s] : T(0);
    }
    return apply_value<DIM, T>(L, w6, p6, pc);
}

// A pair of cells: [0] the red one, [1] the black one.  Where j + k is odd the
// red cell is the right one.
template <int DIM, typename T>
struct Pair {
    T w[2][2 * DIM];
    T den[2], inv[2], rhs[2];
};

// the pair with left cell (i, j, k), i even, of a level with even nx
template <int DIM, typename T>
__device__ __forceinline__ Pair<DIM, T> load_pair(const Lev<T> &L, int i, int j, int k)
{
    const int nx = L.nx, ny = L.ny, nz = L.nz, plane = nx * ny;
    const int c = i + nx * (j + ny * k);
    const Two<T> xa = load2(L.bx + c);
    const T xh = (i + 2 < nx) ? L.bx[c + 2] : L.bxh[j + ny * k];
    const Two<T> yl = load2(L.by + c), yh = load2(j < ny - 1 ? L.by + c + nx : L.byh + i + nx * k);
    Two<T> zl{T(0), T(0)}, zh{T(0), T(0)}, al{T(-0.0), T(-0.0)};
    if constexpr (DIM == 3) {
        zl = load2(L.bz + c);
        zh = load2(k < nz - 1 ? L.bz + c + plane : L.bzh + i + nx * j);
    }
    const Two<T> r = load2(L.rhs + c);
    if (L.alpha) al = load2(L.alpha + c);
    T l[2 * DIM], h[2 * DIM];   // left and right cell
    l[0] = xa.a; l[1] = xa.b; l[2] = yl.a; l[3] = yh.a;
    h[0] = xa.b; h[1] = xh;   h[2] = yl.b; h[3] = yh.b;
    if constexpr (DIM == 3) {
        l[4] = zl.a; l[5] = zh.a;
        h[4] = zl.b; h[5] = zh.b;
    }
    const bool s = (j + k) & 1;
    Pair<DIM, T> P;
#pragma unroll
    for (int q = 0; q < 2 * DIM; ++q) {
        P.w[0][q] = s ? h[q] : l[q];
        P.w[1][q] = s ? l[q] : h[q];
    }
    P.rhs[0] = s ? r.b : r.a;
    P.rhs[1] = s ? r.a : r.b;
    P.den[0] = gs_den<DIM, T>(L, P.w[0], s ? al.b : al.a);
    P.den[1] = gs_den<DIM, T>(L, P.w[1], s ? al.a : al.b);
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2) P.inv[c2] = T(1) / P.den[c2];
    return P;
}

// a pair outside the domain: its cells stay zero through every update
template <int DIM, typename T>
__device__ __forceinline__ Pair<DIM, T> dead_pair()
{
    Pair<DIM, T> P;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
        for (int q = 0; q < 2 * DIM; ++q) P.w[c][q] = T(0);
        P.den[c] = P.inv[c] = T(1);
        P.rhs[c] = T(0);
    }
    return P;
}

// the six (four) neighbour values of the pair's cell of colour c: the pair's
// other cell `oth`, the x neighbour across the pair's end and the row and plane
// neighbours, all of the other colour, from its LDS array O.  x[0], x[1]:
// positions of the row's pairs left and right; y, z: of the rows and planes
// below and above
template <int DIM, typename T>
__device__ __forceinline__ void pair_nbrs(const T *O, bool s, int c, T oth, int xl, int xr, int ym, int yp, int zm,
                                          int zp, T *p)
{
    const bool right = s != (c == 1);   // whether this cell is the pair's right one
    const T xo = O[right ? xr : xl];
    p[0] = right ? oth : xo;
    p[1] = right ? xo : oth;
    p[2] = O[ym];
    p[3] = O[yp];
    if constexpr (DIM == 3) {
        p[4] = O[zm];
        p[5] = O[zp];
    }
}

template <int DIM, typename T>
__device__ __forceinline__ T pair_update(const Lev<T> &L, const Pair<DIM, T> &P, int c, const T *p, T old, bool sor,
                                         T omega)
{
    const T gs = quot(gs_num<DIM, T>(L, P.w[c], p, P.rhs[c]), P.den[c], P.inv[c]);
    return sor ? relax<true>(gs, old, omega) : gs;
}

// The coarse correction at the cells (i, j, k) and (i + 1, j, k), i even:
// prolong_value of both, which share their rows and one of the two x points.
// at(I, J, K): the coarse value
template <int DIM, typename T, typename At>
__device__ __forceinline__ Two<T> prolong_pair(int cnx, int cny, int cnz, const EllBC &bc, int i, int j, int k, At &&at)
{
    int P, ql, qr, y0, y1, z0 = 0, z1 = 0;
    T wp, wl, wr, wy0, wy1, wz0 = T(1), wz1 = T(0);
    lin_w<T>(i, cnx, bc.k[0][0], bc.k[0][1], P, ql, wp, wl);
    lin_w<T>(i + 1, cnx, bc.k[0][0], bc.k[0][1], P, qr, wp, wr);
    lin_w<T>(j, cny, bc.k[1][0], bc.k[1][1], y0, y1, wy0, wy1);
    if constexpr (DIM == 3) lin_w<T>(k, cnz, bc.k[2][0], bc.k[2][1], z0, z1, wz0, wz1);
    T vl[2], vr[2];
#pragma unroll
    for (int cz = 0; cz < (DIM == 3 ? 2 : 1); ++cz) {
        T rl[2], rr[2];
#pragma unroll
        for (int cy = 0; cy < 2; ++cy) {
            const int J = cy ? y1 : y0, K = cz ? z1 : z0;
            const T ep = at(P, J, K);
            rl[cy] = dfma(wl, at(ql, J, K), wp * ep);
            rr[cy] = dfma(wr, at(qr, J, K), wp * ep);
        }
        vl[cz] = dfma(wy1, rl[1], wy0 * rl[0]);
        vr[cz] = dfma(wy1, rr[1], wy0 * rr[0]);
    }
    if constexpr (DIM == 3) return Two<T>{dfma(wz1, vl[1], wz0 * vl[0]), dfma(wz1, vr[1], wz0 * vr[0])};
    else return Two<T>{vl[0], vr[0]};
}

// --------------------------------------------------------------- the legs
// A block's tile TX x TY x TZ with its halo, in pairs along x.  Two sweeps
// (four half-sweeps) and a residual need the four cells around the tile to be
// updated too (H = 4 down); up, without the residual, three would do (H = 3
// in y and z; pairs keep x at 4).  One more layer holds old values only.
template <int DIM, int TX, int TY, int TZ, int H>
struct LegTile {
    static constexpr int HX = TX / 2 + 4, RY = TY + 2 * H, RZ = DIM == 3 ? TZ + 2 * H : 1;
    static constexpr int PX = HX + 2, PY = RY + 2, PZ = DIM == 3 ? RZ + 2 : 1;
    static constexpr int NPAIR = HX * RY * RZ, NPOS = PX * PY * PZ;
    static constexpr int SY = PX, SZ = PX * PY;
};

// the domain's image of g; false outside a non-periodic side
__device__ __forceinline__ bool wrap_into(int &g, int n, int per)
{
    if (per) {
        while (g < 0) g += n;
        while (g >= n) g -= n;
        return true;
    }
    return g >= 0 && g < n;
}

// UP false: two sweeps of pin -> pout (MODE SWEEP_ZERO: pin is zero and not
// read), C.rhs = the averaged residual, C.phi = 0.  UP true: pin + P C.phi, two
// sweeps, -> pout.  pout must not be pin: a block reads pin beyond its tile.
template <int DIM, typename T, int TX, int TY, int TZ, int NTH, bool UP>
__global__ void __launch_bounds__(NTH) k_leg(Lev<T> L, const T *__restrict__ pin, T *__restrict__ pout, Lev<T> C,
                                             EllBC bc, int zero, int ntx, int nty, int total, int per_xcd)
{
    constexpr int H = UP ? 3 : 4;
    using G = LegTile<DIM, TX, TY, TZ, H>;
    constexpr int NP = (G::NPAIR + NTH - 1) / NTH;
    const int b = blockIdx.x;
    const int idx = (b & 7) * per_xcd + (b >> 3);   // neighbouring tiles on one XCD
    if (idx >= total) return;
    const int tz = idx / (ntx * nty), tr = idx - tz * (ntx * nty), ty = tr / ntx, tx = tr - ty * ntx;
    const int x0 = tx * TX - 4, y0 = ty * TY - H, z0 = DIM == 3 ? tz * TZ - H : 0;   // the region's low corner
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    __shared__ T S[2][G::NPOS];
    // ---- pair weights of the region, all loads in flight together
    Pair<DIM, T> P[NP];
    int pos[NP];
    bool s[NP];
#pragma unroll
    for (int a = 0; a < NP; ++a) {
        const int q = threadIdx.x + a * NTH;
        const int m = q % G::HX, r = q / G::HX, jj = r % G::RY, kk = r / G::RY;
        pos[a] = (m + 1) + G::PX * (jj + 1) + (DIM == 3 ? G::SZ * (kk + 1) : 0);
        int gi = x0 + 2 * m, gj = y0 + jj, gk = z0 + kk;
        s[a] = (gj + gk) & 1;
        bool live = q < G::NPAIR;
        live = wrap_into(gi, nx, L.perx) && live;
        live = wrap_into(gj, ny, L.pery) && live;
        if constexpr (DIM == 3) live = wrap_into(gk, nz, L.perz) && live;
        if (live) P[a] = load_pair<DIM, T>(L, gi, gj, gk);
        else P[a] = dead_pair<DIM, T>();
        if (q >= G::NPAIR) pos[a] = 0;   // a ring corner that no cell reads
    }
    // ---- the iterate of the region and its ring
    for (int q = threadIdx.x; q < G::NPOS; q += NTH) {
        const int m = q % G::PX, r = q / G::PX, jj = r % G::PY, kk = r / G::PY;
        int gi = x0 - 2 + 2 * m, gj = y0 - 1 + jj, gk = DIM == 3 ? z0 - 1 + kk : 0;
        const bool sq = (gj + gk) & 1;
        Two<T> v{T(0), T(0)};
        if (UP || !zero) {
            bool live = wrap_into(gi, nx, L.perx);
            live = wrap_into(gj, ny, L.pery) && live;
            if constexpr (DIM == 3) live = wrap_into(gk, nz, L.perz) && live;
            if (live) {
                v = load2(pin + gi + nx * (gj + ny * gk));
                if constexpr (UP) {
                    const T *e = C.phi;
                    const Two<T> d = prolong_pair<DIM, T>(C.nx, C.ny, C.nz, bc, gi, gj, gk, [&](int I, int J, int K) {
                        return e[I + C.nx * (J + C.ny * K)];
                    });
                    v.a = v.a + d.a;
                    v.b = v.b + d.b;
                }
            }
        }
        S[0][q] = sq ? v.b : v.a;
        S[1][q] = sq ? v.a : v.b;
    }
    __syncthreads();
    T v[NP][2];
#pragma unroll
    for (int a = 0; a < NP; ++a) {
        v[a][0] = S[0][pos[a]];
        v[a][1] = S[1][pos[a]];
    }
    const bool sor = L.omega != T(1);
    // ---- two sweeps: a half-sweep reads the other colour only and writes its
    // own, so one barrier each is enough
#pragma unroll 1
    for (int it = 0; it < 2; ++it) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
#pragma unroll
            for (int a = 0; a < NP; ++a) {
                if (threadIdx.x + a * NTH < G::NPAIR) {
                    T p[2 * DIM];
                    const int q = pos[a];
                    pair_nbrs<DIM, T>(S[1 - c], s[a], c, v[a][1 - c], q - 1, q + 1, q - G::SY, q + G::SY, q - G::SZ,
                                      q + G::SZ, p);
                    v[a][c] = pair_update<DIM, T>(L, P[a], c, p, v[a][c], sor, L.omega);
                    S[c][q] = v[a][c];
                }
            }
            __syncthreads();
        }
    }
    // ---- the tile's new iterate, and going down its residual
    constexpr int CX = TX / 2;
    __shared__ T rs[UP ? 1 : CX * TY * TZ];   // left + right residual of a pair
#pragma unroll
    for (int a = 0; a < NP; ++a) {
        const int q = threadIdx.x + a * NTH;
        const int m = q % G::HX, r = q / G::HX, jj = r % G::RY, kk = r / G::RY;
        const int gi = x0 + 2 * m, gj = y0 + jj, gk = z0 + kk;   // not wrapped: the tile lies in the domain
        const bool in = q < G::NPAIR && m >= 2 && m < 2 + CX && jj >= H && jj < H + TY &&
                        (DIM == 2 || (kk >= H && kk < H + TZ)) && gi < nx && gj < ny && gk < nz;
        if (!in) continue;
        const int c0 = gi + nx * (gj + ny * gk);
        store2(pout + c0, s[a] ? v[a][1] : v[a][0], s[a] ? v[a][0] : v[a][1]);
        if constexpr (!UP) {
            T res[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                T p[2 * DIM];
                const int o = pos[a];
                pair_nbrs<DIM, T>(S[1 - c], s[a], c, v[a][1 - c], o - 1, o + 1, o - G::SY, o + G::SY, o - G::SZ,
                                  o + G::SZ, p);
                T ap = apply_w<DIM, T>(L, P[a].w[c], p, v[a][c]);
                if (L.alpha) ap = dfma(L.alpha[c0 + (s[a] != (c == 1) ? 1 : 0)], v[a][c], ap);
                res[c] = P[a].rhs[c] - ap;
            }
            rs[(m - 2) + CX * ((jj - H) + TY * (DIM == 3 ? kk - H : 0))] = res[0] + res[1];
        }
    }
    if constexpr (!UP) {
        __syncthreads();
        constexpr int CY = TY / 2, CZ = DIM == 3 ? TZ / 2 : 1;
        for (int q = threadIdx.x; q < CX * CY * CZ; q += NTH) {
            const int ci = q % CX, r = q / CX, cj = r % CY, ck = r / CY;
            const int I = tx * CX + ci, J = ty * CY + cj, K = DIM == 3 ? tz * CZ + ck : 0;
            if (I >= C.nx || J >= C.ny || K >= C.nz) continue;
            const T *a = rs + ci + CX * (2 * cj + TY * 2 * ck);
            const int o = I + C.nx * (J + C.ny * K);
            if constexpr (DIM == 3) C.rhs[o] = T(0.125) * ((a[0] + a[CX]) + (a[CX * TY] + a[CX * TY + CX]));
            else C.rhs[o] = T(0.25) * (a[0] + a[CX]);
            C.phi[o] = T(0);
        }
    }
}

template <int DIM, typename T, int TX, int TY, int TZ, int NTH, bool UP>
static void launch_leg_t(const Lev<T> &L, const T *pin, T *pout, const Lev<T> &C, const EllBC &bc, bool zero,
                         hipStream_t s)
{
    const int ntx = (L.nx + TX - 1) / TX, nty = (L.ny + TY - 1) / TY, ntz = DIM == 3 ? (L.nz + TZ - 1) / TZ : 1;
    const int total = ntx * nty * ntz, per = (total + 7) / 8;
    hipLaunchKernelGGL((k_leg<DIM, T, TX, TY, TZ, NTH, UP>), dim3((unsigned)(8 * per)), dim3(NTH), 0, s, L, pin, pout,
                       C, bc, (int)zero, ntx, nty, total, per);
}

template <typename T>
bool leg_ok(int dim, const Lev<T> &L)
{
    if (!L.phi2 || (L.nx & 1) || (L.ny & 1) || (dim == 3 && (L.nz & 1))) return false;
    const long n = (long)L.nx * L.ny * L.nz;
    return n <= (dim == 3 ? LEG_MAX_3D : LEG_MAX_2D);
}

template <typename T, bool UP>
static void launch_leg(int dim, const Lev<T> &L, const T *pin, T *pout, const Lev<T> &C, const EllBC &bc, bool zero,
                       hipStream_t s)
{
    const long n = (long)L.nx * L.ny * L.nz;
    if (dim == 2) {
        launch_leg_t<2, T, 32, 32, 1, 832, UP>(L, pin, pout, C, bc, zero, s);
    } else if (n <= LEG_SMALL_3D) {
        launch_leg_t<3, T, 4, 4, 4, 896, UP>(L, pin, pout, C, bc, zero, s);
    } else if constexpr (sizeof(T) == 4) {
        launch_leg_t<3, T, 16, 8, 8, 1024, UP>(L, pin, pout, C, bc, zero, s);
    } else {
        launch_leg_t<3, T, 8, 8, 8, 1024, UP>(L, pin, pout, C, bc, zero, s);
    }
}

template <typename T>
void launch_leg_down(int dim, const Lev<T> &L, const T *pin, T *pout, bool zero, const Lev<T> &C, hipStream_t s)
{
    launch_leg<T, false>(dim, L, pin, pout, C, EllBC{}, zero, s);
}

template <typename T>
void launch_leg_up(int dim, const Lev<T> &L, const T *pin, T *pout, const Lev<T> &C, const EllBC &bc, hipStream_t s)
{
    launch_leg<T, true>(dim, L, pin, pout, C, bc, false, s);
}

// -------------------------------------------------------- wave operations
// lane i ^ MASK of the wave, by data-parallel primitives (a few cycles, where
// a shuffle through LDS takes over a hundred)
template <int CTRL>
__device__ __forceinline__ int dpp(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int MASK>
__device__ __forceinline__ int lane_xor(int v)
{
    static_assert(MASK == 1 || MASK == 2 || MASK == 4 || MASK == 8, "within a row of 16 lanes");
    if constexpr (MASK == 1) return dpp<0xB1>(v);        // quad_perm 1 0 3 2
    else if constexpr (MASK == 2) return dpp<0x4E>(v);   // quad_perm 2 3 0 1
    else if constexpr (MASK == 4) return dpp<0x1B>(dpp<0x141>(v));   // i ^ 7 (row_half_mirror), then i ^ 3
    else return dpp<0x128>(v);                           // row_ror:8
}
template <int MASK>
__device__ __forceinline__ float lane_xor(float v)
{
    return __int_as_float(lane_xor<MASK>(__float_as_int(v)));
}
template <int MASK>
__device__ __forceinline__ double lane_xor(double v)
{
    return __hiloint2double(lane_xor<MASK>(__double2hiint(v)), lane_xor<MASK>(__double2loint(v)));
}

// sum over the 64 lanes in a fixed order (butterfly): every lane holds the
// same, deterministic result
__device__ __forceinline__ double wsum(double v)
{
    v += __shfl_xor(v, 32, 64);
    v += __shfl_xor(v, 16, 64);
    v += lane_xor<8>(v);
    v += lane_xor<4>(v);
    v += lane_xor<2>(v);
    v += lane_xor<1>(v);
    return v;
}
__device__ __forceinline__ double wmax(double v)
{
    v = fmax(v, __shfl_xor(v, 32, 64));
    v = fmax(v, __shfl_xor(v, 16, 64));
    v = fmax(v, lane_xor<8>(v));
    v = fmax(v, lane_xor<4>(v));
    v = fmax(v, lane_xor<2>(v));
    return fmax(v, lane_xor<1>(v));
}

// ------------------------------------------------------- the bottom solve
// One cell per thread: nub red-black sweeps, FP64 CG or BiCGStab on A x = rhs
// (- mean on singular problems) to eps, nub sweeps.  The three forms differ
// in how neighbours and sums reach a thread; X provides
//   nbrs(v, p)      the 2 DIM neighbours' values of v (0 outside)
//   sum(v), max(v)  over all cells, the same in every thread, fixed order
// and says which threads hold a cell (live).
template <int DIM, typename T, typename X>
__device__ __forceinline__ T bottom_solve(const Lev<T> &L, X &x_, const T *w, T acell, int colour, T phi, T rhs,
                                          const CoarseOpts &o, int n)
{
    const bool live = x_.live;
    const T den = gs_den<DIM, T>(L, w, acell), inv = T(1) / den;
    auto sweeps = [&](int count) {
        for (int it = 0; it < count; ++it)
            for (int c = 0; c < 2; ++c) {
                T p[2 * DIM];
                x_.nbrs(phi, p);
                const T v = quot(gs_num<DIM, T>(L, w, p, rhs), den, inv);
                if (live && colour == c) phi = v;
            }
    };
    sweeps(o.nub);
    if (o.bottom == MAC_BOTTOM_SMOOTH) {
        sweeps(o.nub);
        return phi;
    }
    Lev<double> D;
    D.ih2x = L.ih2x; D.ih2y = L.ih2y; D.ih2z = L.ih2z;
    double wd[2 * DIM];
#pragma unroll
    for (int s = 0; s < 2 * DIM; ++s) wd[s] = (double)w[s];
    auto apply = [&](double v) -> double {
        double p[2 * DIM];
        x_.nbrs(v, p);
        if (!live) return 0.0;
        const double ap = apply_w<DIM, double>(D, wd, p, v);
        return L.alpha ? fma((double)acell, v, ap) : ap;
    };
    const double nd = (double)n;
    const double m = o.singular ? x_.sum(live ? (double)rhs : 0.0) / nd : 0.0;
    double x = live ? (double)phi : 0.0;
    const double ax = apply(x);
    double r = live ? ((double)rhs - m) - ax : 0.0;
    auto project = [&]() {   // the mean off r on singular problems
        if (o.singular) {
            const double rm = x_.sum(r) / nd;
            if (live) r -= rm;
        }
    };
    project();
    const double r0 = x_.max(fabs(r));
    if (r0 > 0.0 && o.bottom == MAC_BOTTOM_BICGSTAB) {
        // van der Vorst, SIAM J. Sci. Stat. Comput. 13 (1992) 631-644
        // (FBoxLib's default, mg_bottom_solver = 1, mg.tex:242-243)
        const double rh = r;
        double p = 0.0, v = 0.0, rho_old = 1.0, al = 1.0, om = 1.0;
        for (int it = 0; it < o.bottom_maxit; ++it) {
            const double rho = x_.sum(rh * r);
            if (rho == 0.0) break;
            if (it == 0) p = r;
            else p = r + ((rho / rho_old) * (al / om)) * (p - om * v);
            v = apply(p);
            const double rv = x_.sum(rh * v);
            if (rv == 0.0) break;
            al = rho / rv;
            r -= al * v;
            project();
            if (x_.max(fabs(r)) <= o.bottom_eps * r0) {
                x += al * p;
                break;
            }
            const double t = apply(r);
            const double tt = x_.sum(t * t);
            if (!(tt > 0.0)) {
                x += al * p;
                break;
            }
            om = x_.sum(t * r) / tt;
            x += al * p + om * r;
            r -= om * t;
            project();
            rho_old = rho;
            if (x_.max(fabs(r)) <= o.bottom_eps * r0 || om == 0.0) break;
        }
    } else if (r0 > 0.0) {
        double p = r;
        double rr = x_.sum(r * r);
        for (int it = 0; it < o.bottom_maxit; ++it) {
            const double Ap = apply(p);
            const double pap = x_.sum(p * Ap);
            if (!(pap > 0.0)) break;
            const double alpha = rr / pap;
            x += alpha * p;
            r -= alpha * Ap;
            project();
            const double am = x_.max(fabs(r));
            const double rr1 = x_.sum(r * r);
            if (am <= o.bottom_eps * r0) break;
            const double beta = rr1 / rr;
            rr = rr1;
            p = r + beta * p;
        }
    }
    phi = live ? (T)x : T(0);
    sweeps(o.nub);
    return phi;
}

// 2 cells per direction (2 x 2 x 2, or 2 x 2 in 2D): every group of 8 (4)
// lanes of the wave solves the same problem, neighbours and sums by
// data-parallel primitives.  The sums pair the lanes in the butterfly's order
template <int DIM>
struct BottomTwos {
    bool live = true, in[2 * DIM];   // whether there is a neighbour on each side
    template <typename V>
    __device__ __forceinline__ void nbrs(V v, V *p) const
    {
        V o[3];
        o[0] = lane_xor<1>(v);
        o[1] = lane_xor<2>(v);
        if constexpr (DIM == 3) o[2] = lane_xor<4>(v);
#pragma unroll
        for (int s = 0; s < 2 * DIM; ++s) p[s] = in[s] ? o[s >> 1] : V(0);
    }
    __device__ __forceinline__ double sum(double v) const
    {
        if constexpr (DIM == 3) v += lane_xor<4>(v);
        v += lane_xor<2>(v);
        return v + lane_xor<1>(v);
    }
    __device__ __forceinline__ double max(double v) const
    {
        if constexpr (DIM == 3) v = fmax(v, lane_xor<4>(v));
        v = fmax(v, lane_xor<2>(v));
        return fmax(v, lane_xor<1>(v));
    }
};

// at most 64 cells: one wave, neighbours by lane shuffles
template <int DIM>
struct BottomWave {
    bool live;
    int nb[2 * DIM];   // neighbour lanes, -1 outside
    template <typename V>
    __device__ __forceinline__ void nbrs(V v, V *p) const
    {
#pragma unroll
        for (int s = 0; s < 2 * DIM; ++s) {
            const V t = __shfl(v, nb[s] < 0 ? 0 : nb[s], 64);
            p[s] = nb[s] < 0 ? V(0) : t;
        }
    }
    __device__ __forceinline__ double sum(double v) const { return wsum(v); }
    __device__ __forceinline__ double max(double v) const { return wmax(v); }
};

// up to a block of cells: neighbours and sums through LDS, one barrier each
// (two slots in turn, so a slot is written again only after a barrier that
// all its readers have passed)
template <int DIM>
struct BottomBlock {
    bool live;
    int nb[2 * DIM];      // neighbour cells; outside: the zero cell n
    double *xs, *sh;      // two exchange arrays of n + 1 values; 2 x 32 partial sums
    int n, flip, fs;
    template <typename V>
    __device__ __forceinline__ void nbrs(V v, V *p)
    {
        V *a = reinterpret_cast<V *>(xs + flip * (n + 1));
        flip ^= 1;
        if (live) a[threadIdx.x] = v;
        if ((int)threadIdx.x == n || (n == (int)blockDim.x && threadIdx.x == 0)) a[n] = V(0);
        __syncthreads();
        if (live) {
#pragma unroll
            for (int s = 0; s < 2 * DIM; ++s) p[s] = a[nb[s]];
        } else {
#pragma unroll
            for (int s = 0; s < 2 * DIM; ++s) p[s] = V(0);
        }
    }
    __device__ __forceinline__ double *post(double v)
    {
        double *a = sh + 32 * fs;
        fs ^= 1;
        if ((threadIdx.x & 63) == 0) a[threadIdx.x >> 6] = v;
        __syncthreads();
        return a;
    }
    __device__ __forceinline__ double sum(double v)
    {
        const double *a = post(wsum(v));
        double s = 0.0;
        for (int w = 0; w < (n + 63) >> 6; ++w) s += a[w];
        return s;
    }
    __device__ __forceinline__ double max(double v)
    {
        const double *a = post(wmax(v));
        double s = 0.0;
        for (int w = 0; w < (n + 63) >> 6; ++w) s = fmax(s, a[w]);
        return s;
    }
};

// the neighbours of cell q of level L, `none` outside a non-periodic side
template <int DIM, typename T>
__device__ __forceinline__ void cell_nbrs(const Lev<T> &L, int q, int none, int *nb)
{
    const int nx = L.nx, ny = L.ny, nz = L.nz, sz = nx * ny;
    const int i = q % nx, r = q / nx, j = r % ny, k = r / ny;
    nb[0] = i > 0 ? q - 1 : (L.perx ? q + nx - 1 : none);
    nb[1] = i < nx - 1 ? q + 1 : (L.perx ? q - (nx - 1) : none);
    nb[2] = j > 0 ? q - nx : (L.pery ? q + (ny - 1) * nx : none);
    nb[3] = j < ny - 1 ? q + nx : (L.pery ? q - (ny - 1) * nx : none);
    if constexpr (DIM == 3) {
        nb[4] = k > 0 ? q - sz : (L.perz ? q + (nz - 1) * sz : none);
        nb[5] = k < nz - 1 ? q + sz : (L.perz ? q - (nz - 1) * sz : none);
    }
}

// ---------------------------------------------------------- the coarse cycle
// LDS image, offsets in units of T: level 0 of the cycle (`lc` of the
// hierarchy) takes its pair weights from global memory, into registers, on
// its way down and again up; each level between it and the bottom has its
// pairs' fields (weights, diagonals, reciprocals, rhs) as arrays over the
// pairs; all have the iterate by colour (with a zero at the
// end of each colour for neighbours outside) and, below level 0, as a plain
// array for the prolongation.  The bottom: weights, alpha and rhs by cell.
struct CoarseMap {
    int nl;                    // levels in the cycle
    int S[COARSE_LEVELS], F[COARSE_LEVELS], E[COARSE_LEVELS];
    int rs, bw, br, xs, sh;    // pair residuals; bottom weights, rhs, exchange, sums
    int bytes;
};

template <typename T>
struct CoarseLevs {
    Lev<T> l[COARSE_LEVELS];
};

template <int DIM>
static constexpr int pair_fields() { return 2 * (2 * DIM + 3); }

// positions of a pair's neighbours within a colour array of hx x ny x nz pairs
struct PairPos {
    int q, xl, xr, ym, yp, zm, zp;
};
template <int DIM, typename T>
__device__ __forceinline__ PairPos pair_pos(const Lev<T> &L, int q)
{
    const int hx = L.nx >> 1, ny = L.ny, nz = L.nz, sz = hx * ny, none = sz * nz;
    const int m = q % hx, r = q / hx, j = r % ny, k = r / ny;
    PairPos o;
    o.q = q;
    o.xl = m > 0 ? q - 1 : (L.perx ? q + hx - 1 : none);
    o.xr = m < hx - 1 ? q + 1 : (L.perx ? q - (hx - 1) : none);
    o.ym = j > 0 ? q - hx : (L.pery ? q + (ny - 1) * hx : none);
    o.yp = j < ny - 1 ? q + hx : (L.pery ? q - (ny - 1) * hx : none);
    o.zm = o.zp = none;
    if constexpr (DIM == 3) {
        o.zm = k > 0 ? q - sz : (L.perz ? q + (nz - 1) * sz : none);
        o.zp = k < nz - 1 ? q + sz : (L.perz ? q - (nz - 1) * sz : none);
    }
    return o;
}

// One cycle (V, W or F) over the levels of LV, the first of at most
// COARSE_CELLS cells, the last the bottom.  zero: the first level's iterate is
// zero and is not read.
template <int DIM, typename T, bool VC>
__global__ void __launch_bounds__(COARSE_THREADS) k_coarse(CoarseLevs<T> LV, CoarseMap M, CoarseOpts o, int zero)
{
    extern __shared__ __align__(16) char smem_[];
    T *sm = reinterpret_cast<T *>(smem_);
    constexpr int NT = COARSE_THREADS, NP = COARSE_CELLS / 2 / NT, NF = pair_fields<DIM>();
    const int t = threadIdx.x, bot = M.nl - 1;
    // ---- stage: the iterate of level 0, the deeper levels' pairs and the
    // bottom's weights into LDS
    const Lev<T> &L0 = LV.l[0];
    {
        if (bot > 0) {
            const int hx = L0.nx >> 1, h = hx * L0.ny * L0.nz;
#pragma unroll
            for (int a = 0; a < NP; ++a) {
                const int q = t + a * NT;
                if (q < h) {
                    const int r = q / hx;
                    const bool s = (r % L0.ny + r / L0.ny) & 1;
                    Two<T> v{T(0), T(0)};
                    if (!zero) v = load2(L0.phi + 2 * q);
                    sm[M.S[0] + q] = s ? v.b : v.a;
                    sm[M.S[0] + h + 1 + q] = s ? v.a : v.b;
                }
            }
            if (t < 2) sm[M.S[0] + (t + 1) * (h + 1) - 1] = T(0);
        }
        int first = 0;   // the flattened pairs of the levels between
        for (int l = 1; l < bot; ++l) {
            const Lev<T> &L = LV.l[l];
            const int hx = L.nx >> 1, h = hx * L.ny * L.nz;
            const int q = t - first;
            first = (first + h) % NT;
            // h <= NT / 2 pairs, laid over the threads one level after the other
            const int qq = q < 0 ? q + NT : q;
            if (qq < h) {
                const int m = qq % hx, r = qq / hx, j = r % L.ny, k = r / L.ny;
                const Pair<DIM, T> P = load_pair<DIM, T>(L, 2 * m, j, k);
                T *f = sm + M.F[l] + qq;
#pragma unroll
                for (int c = 0; c < 2; ++c) {
#pragma unroll
                    for (int d = 0; d < 2 * DIM; ++d) f[(c * (2 * DIM + 3) + d) * h] = P.w[c][d];
                    f[(c * (2 * DIM + 3) + 2 * DIM) * h] = P.den[c];
                    f[(c * (2 * DIM + 3) + 2 * DIM + 1) * h] = P.inv[c];
                }
            }
            if (t < 2) sm[M.S[l] + (t + 1) * (h + 1) - 1] = T(0);   // the zero cells
        }
        {
            const Lev<T> &L = LV.l[bot];
            const int n = L.nx * L.ny * L.nz, nx = L.nx, ny = L.ny, nz = L.nz;
            for (int q = NT - 1 - t; q < n; q += NT) {   // from the last thread: the first hold other levels' pairs
                const int i = q % nx, r = q / nx, j = r % ny, k = r / ny;
                T *f = sm + M.bw + q;
                f[0] = L.bx[q];
                f[n] = (i < nx - 1) ? L.bx[q + 1] : L.bxh[j + ny * k];
                f[2 * n] = L.by[q];
                f[3 * n] = (j < ny - 1) ? L.by[q + nx] : L.byh[i + nx * k];
                if constexpr (DIM == 3) {
                    f[4 * n] = L.bz[q];
                    f[5 * n] = (k < nz - 1) ? L.bz[q + nx * ny] : L.bzh[i + nx * j];
                }
                f[2 * DIM * n] = alpha_at(L, q);
                if (bot == 0) {
                    sm[M.br + q] = L.rhs[q];
                    sm[M.E[0] + q] = zero ? T(0) : L.phi[q];
                }
            }
        }
    }
    __syncthreads();

    // `count` sweeps of one pair set; v: the pairs' values, also in LDS
    auto sweeps = [&](const Lev<T> &L, const auto &P, const auto &pos, const auto &s, const auto &on, auto &v, T *S, int h,
                      int count, bool sor) {
        constexpr int N = sizeof(P) / sizeof(P[0]);
        for (int it = 0; it < count; ++it)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                T *own = S + c * (h + 1), *oth = S + (1 - c) * (h + 1);
#pragma unroll
                for (int a = 0; a < N; ++a)
                    if (on[a]) {
                        T p[2 * DIM];
                        pair_nbrs<DIM, T>(oth, s[a], c, v[a][1 - c], pos[a].xl, pos[a].xr, pos[a].ym, pos[a].yp,
                                          pos[a].zm, pos[a].zp, p);
                        v[a][c] = pair_update<DIM, T>(L, P[a], c, p, v[a][c], sor, L.omega);
                        own[pos[a].q] = v[a][c];
                    }
                __syncthreads();
            }
    };
    // the pairs' residuals into rs, then (after a barrier) the next level's
    // right side and zero iterate
    auto resid = [&](const Lev<T> &L, const auto &P, const auto &pos, const auto &s, const auto &on, const auto &v,
                     const T *S, int h) {
        constexpr int N = sizeof(P) / sizeof(P[0]);
#pragma unroll
        for (int a = 0; a < N; ++a)
            if (on[a]) {
                T res[2];
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    T p[2 * DIM];
                    pair_nbrs<DIM, T>(S + (1 - c) * (h + 1), s[a], c, v[a][1 - c], pos[a].xl, pos[a].xr, pos[a].ym,
                                      pos[a].yp, pos[a].zm, pos[a].zp, p);
                    T ap = apply_w<DIM, T>(L, P[a].w[c], p, v[a][c]);
                    if (L.alpha) ap = dfma(L.alpha[2 * pos[a].q + (s[a] != (c == 1) ? 1 : 0)], v[a][c], ap);
                    res[c] = P[a].rhs[c] - ap;
                }
                sm[M.rs + pos[a].q] = res[0] + res[1];
            }
        __syncthreads();
    };
    auto restricted = [&](const Lev<T> &F, int I, int J, int K) -> T {   // coarse cell from rs
        const int hx = F.nx >> 1;
        const T *a = sm + M.rs + I + hx * (2 * J + (DIM == 3 ? F.ny * 2 * K : 0));
        if constexpr (DIM == 3) {
            const int sz = hx * F.ny;
            return T(0.125) * ((a[0] + a[hx]) + (a[sz] + a[sz + hx]));
        } else {
            return T(0.25) * (a[0] + a[hx]);
        }
    };
    auto to_level = [&](int l) {   // right side and zero iterate of level l > 0
        const Lev<T> &F = LV.l[l - 1], &C = LV.l[l];
        if (l == bot) {
            const int n = C.nx * C.ny * C.nz;
            for (int q = t; q < n; q += NT) {
                const int r = q / C.nx;
                sm[M.br + q] = restricted(F, q % C.nx, r % C.ny, r / C.ny);
                sm[M.E[l] + q] = T(0);
            }
            __syncthreads();   // the bottom reads other threads' cells
        } else {
            const int hx = C.nx >> 1, h = hx * C.ny * C.nz;
            if (t < h) {   // read again by this thread only, and S after the sweep's barrier
                const int m = t % hx, r = t / hx, j = r % C.ny, k = r / C.ny;
                const bool s = (j + k) & 1;
                const T a = restricted(F, 2 * m, j, k), b = restricted(F, 2 * m + 1, j, k);
                T *f = sm + M.F[l] + t;
                f[(2 * DIM + 2) * h] = s ? b : a;
                f[(2 * DIM + 3 + 2 * DIM + 2) * h] = s ? a : b;
                sm[M.S[l] + t] = T(0);
                sm[M.S[l] + h + 1 + t] = T(0);
            }
            __syncthreads();
        }
    };
    // the pair of level l that this thread holds, from LDS
    auto pair_of = [&](int l, int h) -> Pair<DIM, T> {
        Pair<DIM, T> P;
        const T *f = sm + M.F[l] + t;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
#pragma unroll
            for (int d = 0; d < 2 * DIM; ++d) P.w[c][d] = f[(c * (2 * DIM + 3) + d) * h];
            P.den[c] = f[(c * (2 * DIM + 3) + 2 * DIM) * h];
            P.inv[c] = f[(c * (2 * DIM + 3) + 2 * DIM + 1) * h];
            P.rhs[c] = f[(c * (2 * DIM + 3) + 2 * DIM + 2) * h];
        }
        return P;
    };
    // level l < bot: down (sweeps, residual, restriction) or up (prolongation, sweeps)
    auto leg = [&](int l, bool up) {
        const Lev<T> &L = LV.l[l];
        const int h = (L.nx >> 1) * L.ny * L.nz;
        T *S = sm + M.S[l];
        auto go = [&](const auto &P, const auto &pos, const auto &s, const auto &on) {
            constexpr int N = sizeof(P) / sizeof(P[0]);
            T v[N][2];
#pragma unroll
            for (int a = 0; a < N; ++a) {
                v[a][0] = v[a][1] = T(0);
                if (!on[a]) continue;
                v[a][0] = S[pos[a].q];
                v[a][1] = S[h + 1 + pos[a].q];
                if (up) {
                    const int hx = L.nx >> 1, m = pos[a].q % hx, r = pos[a].q / hx;
                    const Lev<T> &C = LV.l[l + 1];
                    const T *e = sm + M.E[l + 1];
                    const Two<T> d = prolong_pair<DIM, T>(C.nx, C.ny, C.nz, o.bc, 2 * m, r % L.ny, r / L.ny,
                                                          [&](int I, int J, int K) { return e[I + C.nx * (J + C.ny * K)]; });
                    v[a][0] = v[a][0] + (s[a] ? d.b : d.a);
                    v[a][1] = v[a][1] + (s[a] ? d.a : d.b);
                    S[pos[a].q] = v[a][0];   // read and written by this thread only until the barrier
                    S[h + 1 + pos[a].q] = v[a][1];
                }
            }
            if (up) __syncthreads();
            const bool sor = l == 0 && L.omega != T(1);
            sweeps(L, P, pos, s, on, v, S, h, up ? o.nu2 : o.nu1, sor);
            if (!up) {
                resid(L, P, pos, s, on, v, S, h);
                return;
            }
#pragma unroll
            for (int a = 0; a < N; ++a)
                if (on[a]) {
                    const T lo = s[a] ? v[a][1] : v[a][0], hi = s[a] ? v[a][0] : v[a][1];
                    if (l == 0) store2(L.phi + 2 * pos[a].q, lo, hi);
                    else store2(sm + M.E[l] + 2 * pos[a].q, lo, hi);
                }
            if (l > 0) __syncthreads();
        };
        if (l == 0) {
            // from global memory on each visit (L2): held in registers through
            // the deeper levels they would spill
            Pair<DIM, T> P[NP];
            PairPos pos[NP];
            bool s[NP], on[NP];
#pragma unroll
            for (int a = 0; a < NP; ++a) {
                const int q = t + a * NT;
                P[a] = dead_pair<DIM, T>();
                pos[a] = PairPos{0, 0, 0, 0, 0, 0, 0};
                s[a] = false;
                on[a] = q < h;
                if (on[a]) {
                    const int hx = L.nx >> 1, m = q % hx, r = q / hx, j = r % L.ny, k = r / L.ny;
                    P[a] = load_pair<DIM, T>(L, 2 * m, j, k);
                    pos[a] = pair_pos<DIM, T>(L, q);
                    s[a] = (j + k) & 1;
                }
            }
            go(P, pos, s, on);
        } else {
            Pair<DIM, T> P[1] = {dead_pair<DIM, T>()};
            PairPos pos[1] = {PairPos{0, 0, 0, 0, 0, 0, 0}};
            bool s[1] = {false}, on[1] = {t < h};
            if (on[0]) {
                P[0] = pair_of(l, h);
                pos[0] = pair_pos<DIM, T>(L, t);
                const int r = t / (L.nx >> 1);
                s[0] = (r % L.ny + r / L.ny) & 1;
            }
            go(P, pos, s, on);
        }
        if (!up) to_level(l + 1);
    };
    auto bottom = [&]() {
        const Lev<T> &L = LV.l[bot];
        const int n = L.nx * L.ny * L.nz;
        T *E = sm + M.E[bot];
        auto cell = [&](int q, T *w, T &a, int &colour) {
            const T *f = sm + M.bw + q;
#pragma unroll
            for (int d = 0; d < 2 * DIM; ++d) w[d] = f[d * n];
            a = f[2 * DIM * n];
            const int r = q / L.nx;
            colour = (q % L.nx + r % L.ny + r / L.ny) & 1;
        };
        T w[2 * DIM], a;
        int colour;
        if (n == (1 << DIM) && L.nx == 2 && L.ny == 2) {
            if (t < 64) {
                const int q = t & (n - 1);
                cell(q, w, a, colour);
                BottomTwos<DIM> X;
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    const bool hi = (q >> d) & 1, per = d == 0 ? L.perx : (d == 1 ? L.pery : L.perz);
                    X.in[2 * d] = hi || per;
                    X.in[2 * d + 1] = !hi || per;
                }
                const T v = bottom_solve<DIM, T>(L, X, w, a, colour, E[q], sm[M.br + q], o, n);
                if (t < n) E[t] = v;
            }
        } else if (n <= 64) {
            if (t < 64) {
                const bool live = t < n;
                const int q = live ? t : 0;
                cell(q, w, a, colour);
                BottomWave<DIM> X;
                X.live = live;
                cell_nbrs<DIM, T>(L, q, -1, X.nb);
                const T v = bottom_solve<DIM, T>(L, X, w, a, colour, live ? E[q] : T(0), live ? sm[M.br + q] : T(0), o, n);
                if (live) E[t] = v;
            }
        } else {
            const bool live = t < n;
            const int q = live ? t : 0;
            cell(q, w, a, colour);
            BottomBlock<DIM> X;
            X.live = live;
            X.n = n;
            X.flip = X.fs = 0;
            X.xs = reinterpret_cast<double *>(smem_ + M.xs);
            X.sh = reinterpret_cast<double *>(smem_ + M.sh);
            cell_nbrs<DIM, T>(L, q, n, X.nb);
            const T v = bottom_solve<DIM, T>(L, X, w, a, colour, live ? E[q] : T(0), live ? sm[M.br + q] : T(0), o, n);
            if (live) E[t] = v;
        }
        __syncthreads();
    };
    if constexpr (VC) {
        for (int l = 0; l < bot; ++l) leg(l, false);
        bottom();
        for (int l = bot - 1; l >= 0; --l) leg(l, true);
    } else {
        // W and F cycles, without recursion.  Going down, each level owes a
        // second visit of the next coarser level (bit l of `again`; bit l of
        // `again_w`: that visit is a W, else a V); going up, a level that
        // owes one turns back down before its prolongation.  The first visit
        // has the shape of the visiting level.  The masks are the same in
        // every thread, so the block stays in step.
        unsigned again = 0u, again_w = 0u;
        bool w = o.cycle == MAC_CYCLE_W;   // shape of the current visit (W, or F/V below)
        bool v = false;                     // the current visit is a V
        int l = 0;
        for (;;) {
            for (; l < bot; ++l) {
                leg(l, false);
                if (!v) {
                    again |= 1u << l;
                    if (w) again_w |= 1u << l;
                    else again_w &= ~(1u << l);
                }
            }
            bottom();
            bool down = false;
            while (l > 0) {
                --l;
                if (again & (1u << l)) {   // second visit of level l + 1
                    again &= ~(1u << l);
                    w = (again_w >> l) & 1u;
                    v = !w;
                    ++l;
                    down = true;
                    break;
                }
                leg(l, true);
            }
            if (!down) break;
        }
    }
    if (bot == 0) {
        const int n = L0.nx * L0.ny * L0.nz;
        for (int q = t; q < n; q += NT) L0.phi[q] = sm[M.E[0] + q];
    }
}

// the LDS image of a cycle over levs[lc .. nlev - 1]; false if it has none
template <typename T>
static bool coarse_map(int dim, const Lev<T> *levs, int lc, int nlev, CoarseMap &M)
{
    M = CoarseMap{};
    M.nl = nlev - lc;
    if (M.nl < 1 || M.nl > COARSE_LEVELS) return false;
    const int NF = dim == 3 ? pair_fields<3>() : pair_fields<2>();
    long off = 0;
    auto take = [&](long cnt) {
        const long r = off;
        off += (cnt + 3) / 4 * 4;   // 16-byte steps at least
        return (int)r;
    };
    for (int a = 0; a < M.nl; ++a) {
        const Lev<T> &L = levs[lc + a];
        const long n = (long)L.nx * L.ny * L.nz;
        const bool bottom = a == M.nl - 1;
        if (n > (bottom ? COARSE_BOTTOM : COARSE_CELLS)) return false;
        if (bottom) {
            M.bw = take((2 * dim + 1) * n);
            M.br = take(n);
            M.E[a] = take(n);
            continue;
        }
        if ((L.nx & 1) || (L.ny & 1) || (dim == 3 && (L.nz & 1))) return false;
        if (a > 0 && n / 2 > COARSE_THREADS) return false;
        M.S[a] = take(2 * (n / 2 + 1));
        if (a > 0) {
            M.F[a] = take(NF * (n / 2));
            M.E[a] = take(n);
        } else {
            M.rs = take(n / 2);
        }
    }
    const Lev<T> &B = levs[nlev - 1];
    const long nb = (long)B.nx * B.ny * B.nz;
    long bytes = (off * (long)sizeof(T) + 15) / 16 * 16;
    M.xs = (int)bytes;
    if (nb > 64) bytes += 2 * (nb + 1) * 8;
    M.sh = (int)bytes;
    if (nb > 64) bytes += 64 * 8;
    M.bytes = (int)bytes;
    return bytes <= COARSE_LDS;
}

template <typename T>
int coarse_first(int dim, const Lev<T> *levs, int nlev)
{
    for (int l = 0; l < nlev; ++l) {
        CoarseMap M;
        if (coarse_map<T>(dim, levs, l, nlev, M)) return l;
    }
    return -1;
}

template <typename T>
bool launch_coarse(int dim, const Lev<T> *levs, int lc, int nlev, const CoarseOpts &o, bool zero, hipStream_t s)
{
    CoarseMap M;
    if (!coarse_map<T>(dim, levs, lc, nlev, M)) return false;
    CoarseLevs<T> LV;
    for (int a = 0; a < M.nl; ++a) LV.l[a] = levs[lc + a];
    const dim3 g(1), b(COARSE_THREADS);
    auto go = [&](auto D, auto V) {
        hipLaunchKernelGGL((k_coarse<decltype(D)::value, T, decltype(V)::value>), g, b, (unsigned)M.bytes, s, LV, M, o,
                           (int)zero);
    };
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    const bool v = o.cycle == MAC_CYCLE_V;
    if (dim == 3) v ? go(I3{}, std::true_type{}) : go(I3{}, std::false_type{});
    else v ? go(I2{}, std::true_type{}) : go(I2{}, std::false_type{});
    return true;
}

#define INST(T)                                                                                                       \
    template bool leg_ok<T>(int, const Lev<T> &);                                                                     \
    template void launch_leg_down<T>(int, const Lev<T> &, const T *, T *, bool, const Lev<T> &, hipStream_t);         \
    template void launch_leg_up<T>(int, const Lev<T> &, const T *, T *, const Lev<T> &, const EllBC &, hipStream_t);  \
    template int coarse_first<T>(int, const Lev<T> *, int);                                                           \
    template bool launch_coarse<T>(int, const Lev<T> *, int, int, const CoarseOpts &, bool, hipStream_t);
INST(double)
INST(float)
#undef INST

}  // namespace mac
