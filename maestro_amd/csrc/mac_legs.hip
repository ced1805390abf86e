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

// A copy of x that stays in a register.  A kernel argument used in a loop with
// barriers is otherwise loaded again in each round, at 100 to 200 cycles in a
// chain of some 300.
template <typename T>
__device__ __forceinline__ T held(T x)
{
    asm volatile("" : "+v"(x));
    return x;
}
template <typename T>
__device__ __forceinline__ Lev<T> held_ih2(const Lev<T> &L)
{
    Lev<T> H = L;
    H.ih2x = held(L.ih2x);
    H.ih2y = held(L.ih2y);
    H.ih2z = held(L.ih2z);
    return H;
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
// tiny: the cell's weights, diagonal and right side are scaled by tiny_up().
template <int DIM, typename T>
struct Pair {
    T w[2][2 * DIM];
    T den[2], inv[2], rhs[2];
    bool tiny[2];
};

// what a pair is made of, as loaded
template <int DIM, typename T>
struct PairRaw {
    Two<T> x, yl, yh, zl, zh, r, al;
    T xh;
};

// of the pair with left cell (i, j, k), i even, of a level with even nx
template <int DIM, typename T>
__device__ __forceinline__ PairRaw<DIM, T> load_raw(const Lev<T> &L, int i, int j, int k)
{
    const int nx = L.nx, ny = L.ny, nz = L.nz, plane = nx * ny;
    const int c = i + nx * (j + ny * k);
    PairRaw<DIM, T> R;
    R.x = load2(L.bx + c);
    R.xh = *((i + 2 < nx) ? L.bx + c + 2 : L.bxh + j + ny * k);
    R.yl = load2(L.by + c);
    R.yh = load2(j < ny - 1 ? L.by + c + nx : L.byh + i + nx * k);
    if constexpr (DIM == 3) {
        R.zl = load2(L.bz + c);
        R.zh = load2(k < nz - 1 ? L.bz + c + plane : L.bzh + i + nx * j);
    }
    R.r = load2(L.rhs + c);
    R.al = Two<T>{T(-0.0), T(-0.0)};
    if (L.alpha) R.al = load2(L.alpha + c);
    return R;
}

// to be called when a thread's loads are on their way: the branch waits for the
// diagonals (called pair by pair it cost a round trip to memory, 0.3 us a leg)
template <int DIM, typename T>
__device__ __forceinline__ void scale_tiny(Pair<DIM, T> &P)
{
    P.tiny[0] = is_tiny(P.den[0]);
    P.tiny[1] = is_tiny(P.den[1]);
    if (__builtin_expect(__ballot(P.tiny[0] || P.tiny[1]) != 0, 0)) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const T f = P.tiny[c] ? tiny_up<T>() : T(1);
#pragma unroll
            for (int q = 0; q < 2 * DIM; ++q) P.w[c][q] *= f;
            P.den[c] *= f;
            P.rhs[c] *= f;
            P.inv[c] = T(1) / P.den[c];
        }
    }
}

// the right sides r of the pair and its ap = A phi without that scale (one
// branch for both: it parts the loads before it from those behind)
template <int DIM, typename T>
__device__ __forceinline__ void true_scale(const Pair<DIM, T> &P, T *r, T *ap)
{
    r[0] = P.rhs[0];
    r[1] = P.rhs[1];
    if (__builtin_expect(__ballot(P.tiny[0] || P.tiny[1]) != 0, 0)) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const T f = P.tiny[c] ? tiny_down<T>() : T(1);
            ap[c] *= f;
            r[c] *= f;
        }
    }
}

// s: j + k is odd
template <int DIM, typename T>
__device__ __forceinline__ Pair<DIM, T> make_pair(const Lev<T> &L, const PairRaw<DIM, T> &R, bool s)
{
    T l[2 * DIM], h[2 * DIM];   // left and right cell
    l[0] = R.x.a; l[1] = R.x.b; l[2] = R.yl.a; l[3] = R.yh.a;
    h[0] = R.x.b; h[1] = R.xh;  h[2] = R.yl.b; h[3] = R.yh.b;
    if constexpr (DIM == 3) {
        l[4] = R.zl.a; l[5] = R.zh.a;
        h[4] = R.zl.b; h[5] = R.zh.b;
    }
    Pair<DIM, T> P;
#pragma unroll
    for (int q = 0; q < 2 * DIM; ++q) {
        P.w[0][q] = s ? h[q] : l[q];
        P.w[1][q] = s ? l[q] : h[q];
    }
    P.rhs[0] = s ? R.r.b : R.r.a;
    P.rhs[1] = s ? R.r.a : R.r.b;
    P.den[0] = gs_den<DIM, T>(L, P.w[0], s ? R.al.b : R.al.a);
    P.den[1] = gs_den<DIM, T>(L, P.w[1], s ? R.al.a : R.al.b);
#pragma unroll
    for (int c = 0; c < 2; ++c) P.inv[c] = T(1) / P.den[c];
    return P;
}

template <int DIM, typename T>
__device__ __forceinline__ Pair<DIM, T> load_pair(const Lev<T> &L, int i, int j, int k)
{
    return make_pair<DIM, T>(L, load_raw<DIM, T>(L, i, j, k), (j + k) & 1);
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
    // coarse rows and planes that a way up reads: the parents of the ring's
    // cells and one more on each side
    static constexpr int RYC = PY / 2 + 2, RZC = DIM == 3 ? PZ / 2 + 2 : 1;
};

// lin_w for a row or plane index that is not wrapped: the periodic image of
// Q stands at Q itself
template <typename T>
__device__ __forceinline__ void row_w(int g, int nc, int kind_lo, int kind_hi, int &P, int &Q, T &wp, T &wq)
{
    const int p = g >> 1, q = (g & 1) ? p + 1 : p - 1;
    const int kind = q < 0 ? kind_lo : (q >= nc ? kind_hi : ELL_PER);
    P = p;
    Q = kind == ELL_PER ? q : p;
    wp = T(0.75);
    wq = kind == ELL_DIR ? T(-0.25) : T(0.25);
}

// the domain's image of g; false outside a non-periodic side.  per: 0 not
// periodic, 1 one period reaches (selects), 2 the region spans several
__device__ __forceinline__ bool wrap_into(int &g, int n, int per)
{
    if (per) {
        g = g < 0 ? g + n : g;
        g = g >= n ? g - n : g;
        if (per == 2) {
            while (g < 0) g += n;
            while (g >= n) g -= n;
        }
    }
    return (unsigned)g < (unsigned)n;
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
    // a tile starts inside the domain, so an extent of at least a tile and its
    // halo (coarse rows: half of both) is wrapped once
    const int px = L.perx ? (nx < TX + 8 ? 2 : 1) : 0, py = L.pery ? (ny < TY + 8 ? 2 : 1) : 0;
    const int pz = L.perz ? (nz < TZ + 8 ? 2 : 1) : 0;
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
        live = wrap_into(gi, nx, px) && live;
        live = wrap_into(gj, ny, py) && live;
        if constexpr (DIM == 3) live = wrap_into(gk, nz, pz) && live;
        if (live) P[a] = load_pair<DIM, T>(L, gi, gj, gk);
        else P[a] = dead_pair<DIM, T>();
        if (q >= G::NPAIR) pos[a] = 0;   // a ring corner that no cell reads
    }
    // ---- going up: the coarse rows that the region touches, interpolated in x
    // to its pairs (both cells), so a cell reads 4 values instead of 12
    const int JB = (y0 - 1) / 2 - 1, KB = DIM == 3 ? (z0 - 1) / 2 - 1 : 0;   // y0 - 1, z0 - 1 are even
    __shared__ Two<T> xr[UP ? G::PX * G::RYC * G::RZC : 1];
    if constexpr (UP) {
        for (int q = threadIdx.x; q < G::PX * G::RYC * G::RZC; q += NTH) {
            const int m = q % G::PX, r = q / G::PX;
            int gi = x0 - 2 + 2 * m, J = JB + r % G::RYC, K = KB + r / G::RYC;
            bool live = wrap_into(gi, nx, px);
            live = wrap_into(J, C.ny, py) && live;
            if constexpr (DIM == 3) live = wrap_into(K, C.nz, pz) && live;
            Two<T> v{T(0), T(0)};
            if (live) {
                int pc, ql, qr;
                T wp, wl, wr;
                lin_w<T>(gi, C.nx, bc.k[0][0], bc.k[0][1], pc, ql, wp, wl);
                lin_w<T>(gi + 1, C.nx, bc.k[0][0], bc.k[0][1], pc, qr, wp, wr);
                const T *e = C.phi + C.nx * (J + C.ny * K);
                const T ep = wp * e[pc];
                v.a = dfma(wl, e[ql], ep);
                v.b = dfma(wr, e[qr], ep);
            }
            xr[q] = v;
        }
        __syncthreads();
    }
    // ---- the iterate of the region and its ring
    for (int q = threadIdx.x; q < G::NPOS; q += NTH) {
        const int m = q % G::PX, r = q / G::PX, jj = r % G::PY, kk = r / G::PY;
        int gi = x0 - 2 + 2 * m, gj = y0 - 1 + jj, gk = DIM == 3 ? z0 - 1 + kk : 0;
        const bool sq = (gj + gk) & 1;
        Two<T> v{T(0), T(0)};
        if (UP || !zero) {
            const int uj = gj, uk = gk;   // not wrapped
            bool live = wrap_into(gi, nx, px);
            live = wrap_into(gj, ny, py) && live;
            if constexpr (DIM == 3) live = wrap_into(gk, nz, pz) && live;
            if (live) {
                v = load2(pin + gi + nx * (gj + ny * gk));
                if constexpr (UP) {
                    // y and z of prolong_value from the rows' x parts
                    int y0r, y1r, z0r = 0, z1r = 0;
                    T wy0, wy1, wz0 = T(1), wz1 = T(0);
                    row_w(uj, C.ny, bc.k[1][0], bc.k[1][1], y0r, y1r, wy0, wy1);
                    if constexpr (DIM == 3) row_w(uk, C.nz, bc.k[2][0], bc.k[2][1], z0r, z1r, wz0, wz1);
                    const Two<T> *e = xr + m - G::PX * (JB + (DIM == 3 ? G::RYC * KB : 0));
                    T vl[2], vr[2];
#pragma unroll
                    for (int cz = 0; cz < (DIM == 3 ? 2 : 1); ++cz) {
                        const int kr = DIM == 3 ? G::RYC * (cz ? z1r : z0r) : 0;
                        const Two<T> a = e[G::PX * (y0r + kr)], d = e[G::PX * (y1r + kr)];
                        vl[cz] = dfma(wy1, d.a, wy0 * a.a);
                        vr[cz] = dfma(wy1, d.b, wy0 * a.b);
                    }
                    if constexpr (DIM == 3) {
                        v.a = v.a + dfma(wz1, vl[1], wz0 * vl[0]);
                        v.b = v.b + dfma(wz1, vr[1], wz0 * vr[0]);
                    } else {
                        v.a = v.a + vl[0];
                        v.b = v.b + vr[0];
                    }
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
        scale_tiny(P[a]);
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
            T r[2], ap[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                T p[2 * DIM];
                const int o = pos[a];
                pair_nbrs<DIM, T>(S[1 - c], s[a], c, v[a][1 - c], o - 1, o + 1, o - G::SY, o + G::SY, o - G::SZ,
                                  o + G::SZ, p);
                ap[c] = apply_w<DIM, T>(L, P[a].w[c], p, v[a][c]);
            }
            true_scale(P[a], r, ap);
            if (L.alpha) {
#pragma unroll
                for (int c = 0; c < 2; ++c) ap[c] = dfma(L.alpha[c0 + (s[a] != (c == 1) ? 1 : 0)], v[a][c], ap[c]);
            }
            rs[(m - 2) + CX * ((jj - H) + TY * (DIM == 3 ? kk - H : 0))] = (r[0] - ap[0]) + (r[1] - ap[1]);
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

// The tile: the smallest that gives at most one block per CU (256), else the
// largest.  A larger tile repeats less of its halo, a smaller one spreads a
// small level over more CUs.  Down / up, microseconds: 32^3 FP32 8 x 4 x 4
// (256 blocks) 6.0 / 6.2, 4 x 4 x 4 (512) 8.9 / 9.3, 8 x 8 x 8 (64) 7.2 / 8.1;
// 64^3 FP32 16 x 8 x 8 (256) 10.8 / 11.5, 8 x 8 x 8 (512) 11.9 / 16.7, FP64
// 8 x 8 x 8 18.9 / 19.9, 16 x 8 x 4 (512) 21.5 / 22.6.
template <typename T, bool UP>
static void launch_leg(int dim, const Lev<T> &L, const T *pin, T *pout, const Lev<T> &C, const EllBC &bc, bool zero,
                       hipStream_t s)
{
    auto tiles = [&](int tx, int ty, int tz) {
        return (long)((L.nx + tx - 1) / tx) * ((L.ny + ty - 1) / ty) * ((L.nz + tz - 1) / tz);
    };
    if (dim == 2)
        launch_leg_t<2, T, 32, 32, 1, 832, UP>(L, pin, pout, C, bc, zero, s);
    else if (tiles(8, 4, 4) <= 256)
        launch_leg_t<3, T, 8, 4, 4, sizeof(T) == 4 ? 1024 : 640, UP>(L, pin, pout, C, bc, zero, s);
    else if (sizeof(T) == 8 || tiles(8, 8, 8) <= 256)
        launch_leg_t<3, T, 8, 8, 8, 1024, UP>(L, pin, pout, C, bc, zero, s);
    else if constexpr (sizeof(T) == 4)
        launch_leg_t<3, T, 16, 8, 8, 1024, UP>(L, pin, pout, C, bc, zero, s);
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

// v of lane i plus (or max with) v of lane i ^ 32, i ^ 16: the swap
// instructions exchange the upper and lower halves (odd and even rows of 16)
// of two registers, here of two copies of v
template <int MASK, typename F>
__device__ __forceinline__ double swap_op(double v, F &&f)
{
    static_assert(MASK == 32 || MASK == 16, "halves or rows");
    const unsigned hi = (unsigned)__double2hiint(v), lo = (unsigned)__double2loint(v);
    if constexpr (MASK == 32) {
        const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
        const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
        return f(__hiloint2double((int)h[0], (int)l[0]), __hiloint2double((int)h[1], (int)l[1]));
    } else {
        const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        return f(__hiloint2double((int)h[0], (int)l[0]), __hiloint2double((int)h[1], (int)l[1]));
    }
}
// over the 64 lanes in a fixed order (butterfly): every lane holds the same,
// deterministic result
template <typename F>
__device__ __forceinline__ double wave_all(double v, F &&f)
{
    v = swap_op<32>(v, f);
    v = swap_op<16>(v, f);
    v = f(v, lane_xor<8>(v));
    v = f(v, lane_xor<4>(v));
    v = f(v, lane_xor<2>(v));
    return f(v, lane_xor<1>(v));
}
__device__ __forceinline__ double wsum(double v)
{
    return wave_all(v, [](double a, double b) { return a + b; });
}
__device__ __forceinline__ double wmax(double v)
{
    return wave_all(v, [](double a, double b) { return fmax(a, b); });
}

// ------------------------------------------------------- the bottom solve
// One cell per thread: nub red-black sweeps, FP64 CG or BiCGStab on A x = rhs
// (- mean on singular problems) to eps, nub sweeps.  The three forms differ
// in how neighbours and sums reach a thread; X provides
//   nbrs(v, p)      the 2 DIM neighbours' values of v (0 outside)
//   nbrs_any(v, p)  the same, where has(s) is false any finite value
//   sum(v), max(v), sum_max(s, m)  over all cells, the same in every thread,
//                   fixed order
// and says which threads hold a cell (live).
template <int DIM, typename T, typename X>
__device__ __forceinline__ T bottom_solve(const Lev<T> &L_, X &x_, const T *w, T acell, int colour, T phi, T rhs,
                                          const CoarseOpts &o, int n)
{
    const bool live = x_.live;
    const Lev<T> L = held_ih2(L_);
    const bool has_alpha = held((int)(L_.alpha != nullptr));
    const int n_sweeps = held(o.nub), singular = held(o.singular);
    const double eps = held(o.bottom_eps);
    // for the sweeps: the weights of the neighbours, the diagonal and the right
    // side, scaled as a pair's where the diagonal is tiny
    T wn[2 * DIM], den = gs_den<DIM, T>(L, w, acell), rn = rhs;
#pragma unroll
    for (int s = 0; s < 2 * DIM; ++s) wn[s] = x_.has(s) ? w[s] : T(0);
    if (__builtin_expect(__ballot(live && is_tiny(den)) != 0, 0)) {
        const T f = is_tiny(den) ? tiny_up<T>() : T(1);
#pragma unroll
        for (int s = 0; s < 2 * DIM; ++s) wn[s] *= f;
        den *= f;
        rn *= f;
    }
    const T inv = T(1) / den;
    // the mean of a sum over the cells
    auto mean = [&](double v) -> double { return X::POW2 ? v * (1.0 / n) : v / (double)n; };
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
        return has_alpha ? fma((double)acell, v, ap) : ap;
    };
#pragma unroll 1
    for (int part = 0; part < 2; ++part) {
#pragma unroll 1
        for (int h = 0; h < 2 * n_sweeps; ++h) {
            T p[2 * DIM];
            x_.nbrs_any(phi, p);
            const T v = quot(gs_num<DIM, T>(L, wn, p, rn), den, inv);
            if (live && colour == (h & 1)) phi = v;
        }
        if (part == 1 || o.bottom == MAC_BOTTOM_SMOOTH) continue;
        const double m = singular ? mean(x_.sum(live ? (double)rhs : 0.0)) : 0.0;
        double x = live ? (double)phi : 0.0;
        const double ax = apply(x);
        double r = live ? ((double)rhs - m) - ax : 0.0;
        auto project = [&]() {   // the mean off r on singular problems
            if (singular) {
                const double rm = mean(x_.sum(r));
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
#pragma unroll 1
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
                if (x_.max(fabs(r)) <= eps * r0) {
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
                if (x_.max(fabs(r)) <= eps * r0 || om == 0.0) break;
            }
        } else if (r0 > 0.0) {
            double p = r;
            double rr = x_.sum(r * r);
#pragma unroll 1
            for (int it = 0; it < o.bottom_maxit; ++it) {
                const double irr = 1.0 / rr;   // off the chain of the step
                const double Ap = apply(p);
                const double pap = x_.sum(p * Ap);
                if (!(pap > 0.0)) break;
                const double alpha = rr / pap;
                x += alpha * p;
                r -= alpha * Ap;
                project();
                double rr1 = r * r, am = fabs(r);
                x_.sum_max(rr1, am);
                if (am <= eps * r0) break;
                double beta = quot(rr1, rr, irr);
                if (__builtin_expect(__ballot(!__builtin_isnormal(irr)) != 0, 0)) beta = rr1 / rr;
                rr = rr1;
                p = r + beta * p;
            }
        }
        phi = live ? (T)x : T(0);
    }
    return phi;
}

// 2 cells per direction (2 x 2 x 2, or 2 x 2 in 2D): every group of 8 (4)
// lanes of the wave solves the same problem, neighbours and sums by
// data-parallel primitives.  In a sweep a side without a neighbour is left out
// by a zero weight, so no value is selected.  The sums pair the lanes in the
// butterfly's order
// lane i ^ 4 where lanes 8 apart hold the same: a rotation by 4 in the row
__device__ __forceinline__ float group_xor4(float v) { return __int_as_float(dpp<0x124>(__float_as_int(v))); }
__device__ __forceinline__ double group_xor4(double v)
{
    return __hiloint2double(dpp<0x124>(__double2hiint(v)), dpp<0x124>(__double2loint(v)));
}
template <int DIM>
struct BottomTwos {
    static constexpr bool POW2 = true;   // 4 or 8 cells: 1 / n is exact
    bool live = true, in[2 * DIM];       // whether there is a neighbour on each side
    __device__ __forceinline__ bool has(int s) const { return in[s]; }
    template <typename V>
    __device__ __forceinline__ void nbrs_any(V v, V *p) const
    {
        V o[3];
        o[0] = lane_xor<1>(v);
        o[1] = lane_xor<2>(v);
        if constexpr (DIM == 3) o[2] = group_xor4(v);
#pragma unroll
        for (int s = 0; s < 2 * DIM; ++s) p[s] = o[s >> 1];
    }
    template <typename V>
    __device__ __forceinline__ void nbrs(V v, V *p) const
    {
        nbrs_any(v, p);
#pragma unroll
        for (int s = 0; s < 2 * DIM; ++s) p[s] = in[s] ? p[s] : V(0);
    }
    __device__ __forceinline__ double sum(double v) const
    {
        if constexpr (DIM == 3) v += group_xor4(v);
        v += lane_xor<2>(v);
        return v + lane_xor<1>(v);
    }
    __device__ __forceinline__ double max(double v) const
    {
        if constexpr (DIM == 3) v = fmax(v, group_xor4(v));
        v = fmax(v, lane_xor<2>(v));
        return fmax(v, lane_xor<1>(v));
    }
    __device__ __forceinline__ void sum_max(double &s, double &m) const
    {
        s = sum(s);
        m = max(m);
    }
};

// at most 64 cells: one wave, neighbours by lane shuffles
template <int DIM>
struct BottomWave {
    static constexpr bool POW2 = false;
    __device__ __forceinline__ bool has(int) const { return true; }
    template <typename V>
    __device__ __forceinline__ void nbrs_any(V v, V *p)
    {
        nbrs(v, p);
    }
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
    __device__ __forceinline__ void sum_max(double &s, double &m) const
    {
        s = wsum(s);
        m = wmax(m);
    }
};

// up to a block of cells: neighbours and sums through LDS, one barrier each
// (two slots in turn, so a slot is written again only after a barrier that
// all its readers have passed).  Only the waves that hold cells run the solve;
// the others wait at its barriers (idle), since their instructions would take
// the busy waves' turns: 6 x 5 x 7 cells FP64, 3100 -> 2150 cycles a CG step.
template <int DIM, bool FOLD>   // FOLD: more than 512 cells
struct BottomBlock {
    static constexpr bool POW2 = false;
    bool live;
    int nb[2 * DIM];      // neighbour cells; outside: -1, the zeros before an array
    double *xs, *sh;      // two exchange arrays of 1 + n values; 2 x 32 partial results
    volatile int *last;   // number of the last barrier, set before it
    int n, flip, fs, bar; // bar: barriers passed
    __device__ __forceinline__ bool has(int) const { return true; }
    __device__ __forceinline__ void sync()
    {
        ++bar;
        __syncthreads();
    }
    // the barriers of a solve, for a wave without cells; each compares its own
    // count, so a late look at `last` cannot end it early
    __device__ __forceinline__ void idle() const
    {
        for (int k = 1;; ++k) {
            __syncthreads();
            if (*last == k) break;
        }
    }
    __device__ __forceinline__ void finish()
    {
        if (threadIdx.x == 0) *last = bar + 1;
        sync();
    }
    template <typename V>
    __device__ __forceinline__ void nbrs_any(V v, V *p)
    {
        nbrs(v, p);
    }
    template <typename V>
    __device__ __forceinline__ void nbrs(V v, V *p)
    {
        V *a = reinterpret_cast<V *>(xs + (flip ? n + 2 : 1));
        flip ^= 1;
        if (live) a[threadIdx.x] = v;
        sync();
        if (live) {
#pragma unroll
            for (int s = 0; s < 2 * DIM; ++s) p[s] = a[nb[s]];
        } else {
#pragma unroll
            for (int s = 0; s < 2 * DIM; ++s) p[s] = V(0);
        }
    }
    // over the waves' partial results in order, four reads at a time (those
    // of idle waves are zero)
    template <typename F>
    __device__ __forceinline__ double over(const double *a, F &&f) const
    {
        double s = 0.0;
#pragma unroll 1
        for (int w = 0; w < n; w += 256, a += 4) {
            const double a0 = a[0], a1 = a[1], a2 = a[2], a3 = a[3];
            s = f(f(f(f(s, a0), a1), a2), a3);
        }
        return s;
    }
    __device__ __forceinline__ double *slot()
    {
        double *a = sh + 32 * fs;
        fs ^= 1;
        return a;
    }
    // Beyond 512 cells a sum takes cells t and t + 512 together, then the waves
    // in order, as a block of 512 threads does (k_bottom).  A singular bottom's
    // constant mode is whatever the rounding of its sums leaves in it, and phi's
    // constant with it: with another order it moved by up to 1e-5 of phi's range
    // (192 x 80 x 256).  The tests hold the solution up to that constant, and its
    // bits from call to call; nothing compares the order itself.
    __device__ __forceinline__ double folded(double v)
    {
        if constexpr (!FOLD) return v;
        double *a = xs + (flip ? n + 2 : 1);
        flip ^= 1;
        const int t = threadIdx.x;
        if (live && t >= 512) a[t] = v;
        sync();
        if (t >= 512) return 0.0;
        return t + 512 < n ? v + a[t + 512] : v;
    }
    __device__ __forceinline__ double sum(double v)
    {
        v = folded(v);
        double *a = slot();
        v = wsum(v);
        if ((threadIdx.x & 63) == 0) a[threadIdx.x >> 6] = v;
        sync();
        return over(a, [](double x, double y) { return x + y; });
    }
    __device__ __forceinline__ double max(double v)
    {
        double *a = slot();
        v = wmax(v);
        if ((threadIdx.x & 63) == 0) a[threadIdx.x >> 6] = v;
        sync();
        return over(a, [](double x, double y) { return fmax(x, y); });
    }
    __device__ __forceinline__ void sum_max(double &s, double &m)   // one barrier for both
    {
        s = folded(s);
        double *a = slot();
        s = wsum(s);
        m = wmax(m);
        if ((threadIdx.x & 63) == 0) {
            a[threadIdx.x >> 6] = s;
            a[16 + (threadIdx.x >> 6)] = m;
        }
        sync();
        s = over(a, [](double x, double y) { return x + y; });
        m = over(a + 16, [](double x, double y) { return fmax(x, y); });
    }
};

// q / d for q d < 2^32: the high word of q times m = floor(2^32 / d) + 1 (0: d = 1)
__device__ __forceinline__ int fast_div(int q, unsigned m)
{
    return m ? (int)__umulhi((unsigned)q, m) : q;
}
static unsigned fast_div_factor(int d)
{
    return d == 1 ? 0u : (unsigned)(4294967296.0 / d) + 1u;
}
// position q of a row-major array of rows of nx in planes of ny rows
struct Ijk {
    int i, j, k;
};
__device__ __forceinline__ Ijk ijk_of(int q, int nx, int ny, unsigned mx, unsigned my)
{
    const int r = fast_div(q, mx), k = fast_div(r, my);
    return Ijk{q - r * nx, r - k * ny, k};
}

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
// LDS image, offsets in bytes.  Level 0 of the cycle (`lc` of the hierarchy)
// has its iterate by colour at 0, its pairs' weights come from global memory
// on the way down and again up.  A pair of a level between it and the bottom
// belongs to one thread throughout, which keeps the weights in registers; LDS
// holds the iterate by colour and, for the prolongation, as a plain array.  A
// colour array ends in a zero cell for neighbours outside; colour 1 lies a
// constant stride behind colour 0, so an access is one address and an
// immediate offset.  The bottom: weights, alpha, rhs and iterate by cell.
struct CoarseMap {
    int nl;                    // levels in the cycle
    int S[COARSE_LEVELS], E[COARSE_LEVELS];
    int rs, bw, br, xs, sh;    // pair residuals; bottom weights, rhs, exchange, sums
    int park, mid;             // waiting pairs of the levels between, their number
    // factors of fast_div by a row's pairs (the bottom: cells) and by the rows
    unsigned mx[COARSE_LEVELS], my[COARSE_LEVELS];
    int bytes;
};

// pairs of all levels between the first and the bottom: one thread each
static constexpr int COARSE_MID = COARSE_CELLS / 8 + 1;   // of one level, and the zero cell
template <typename T> static constexpr int colour0() { return (COARSE_CELLS / 2 + 2) * (int)sizeof(T); }
template <typename T> static constexpr int colour_mid() { return (COARSE_MID + 1) * (int)sizeof(T); }

template <typename T>
struct CoarseLevs {
    Lev<T> l[COARSE_LEVELS];
};

// a pair: its place among its level's pairs and the LDS offsets (colour 0) of
// itself, of the x neighbours across its ends (x[c]: colour c's) and of its
// row and plane neighbours
struct PairPos {
    int q, m, j, k;
    int at, x[2], ym, yp, zm, zp;
    bool s, on;
};
template <int DIM, typename T>
__device__ __forceinline__ PairPos pair_pos(const Lev<T> &L, int q, int S, unsigned mx, unsigned my)
{
    const int hx = L.nx >> 1, ny = L.ny, nz = L.nz, sz = hx * ny, none = sz * nz;
    PairPos o;
    o.on = q < none;
    if (!o.on) q = 0;
    const Ijk c = ijk_of(q, hx, ny, mx, my);
    o.q = q; o.m = c.i; o.j = c.j; o.k = c.k;
    o.s = (c.j + c.k) & 1;
    auto off = [&](int p) { return S + p * (int)sizeof(T); };
    o.at = off(q);
    const int xl = off(c.i > 0 ? q - 1 : (L.perx ? q + hx - 1 : none));
    const int xr = off(c.i < hx - 1 ? q + 1 : (L.perx ? q - (hx - 1) : none));
    o.x[0] = o.s ? xr : xl;   // the red cell is the right one where s
    o.x[1] = o.s ? xl : xr;
    o.ym = off(c.j > 0 ? q - hx : (L.pery ? q + (ny - 1) * hx : none));
    o.yp = off(c.j < ny - 1 ? q + hx : (L.pery ? q - (ny - 1) * hx : none));
    o.zm = o.zp = 0;
    if constexpr (DIM == 3) {
        o.zm = off(c.k > 0 ? q - sz : (L.perz ? q + (nz - 1) * sz : none));
        o.zp = off(c.k < nz - 1 ? q + sz : (L.perz ? q - (nz - 1) * sz : none));
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
    constexpr int NT = COARSE_THREADS, NP = COARSE_CELLS / 2 / NT;
    constexpr int C0 = colour0<T>(), CM = colour_mid<T>();
    const int t = threadIdx.x, bot = M.nl - 1;
    auto arr = [&](int off) -> T * { return reinterpret_cast<T *>(smem_ + off); };
    auto ref = [&](int off) -> T & { return *reinterpret_cast<T *>(smem_ + off); };
    const Lev<T> &L0 = LV.l[0];
    // in 3D and FP64 (or the W and F shapes) the pairs of the levels between
    // wait in LDS and come into registers for a leg: they would spill
    constexpr bool PARK = DIM == 3 && (sizeof(T) == 8 || !VC);
    Pair<DIM, T> Pm;      // the pair of a level between that this thread owns
    PairPos om;
    int lm = 0, qm = 0;   // that level (0: none), the pair's place in it
    bool tiny0 = false, tiny1 = false;   // Pair::tiny of Pm
    // the deeper levels' pairs, the bottom's weights and level 0's iterate
    // (pairs at o0): every load issued before the first is waited for
    auto stage = [&](const PairPos(&o0)[NP]) {
        Two<T> v0[NP];
#pragma unroll
        for (int a = 0; a < NP; ++a) {
            v0[a] = Two<T>{T(0), T(0)};
            if (bot > 0 && !zero) v0[a] = load2(L0.phi + 2 * o0[a].q);
        }
        PairRaw<DIM, T> Rm;
        int first = 0;
        for (int l = 1; l < bot; ++l) {
            const Lev<T> &L = LV.l[l];
            const int h = (L.nx >> 1) * L.ny * L.nz;
            if (t >= first && t < first + h) {
                lm = l;
                qm = t - first;
                om = pair_pos<DIM, T>(L, qm, M.S[l], M.mx[l], M.my[l]);
                Rm = load_raw<DIM, T>(L, 2 * om.m, om.j, om.k);
            }
            first += h;
            if (t < 2) ref(M.S[l] + h * (int)sizeof(T) + t * CM) = T(0);   // the zero cells
        }
        const Lev<T> &L = LV.l[bot];
        const int n = L.nx * L.ny * L.nz, nx = L.nx, ny = L.ny, nz = L.nz;
        for (int q = NT - 1 - t; q < n; q += NT) {   // from the last thread: the first own other levels' pairs
            const Ijk c = ijk_of(q, nx, ny, M.mx[bot], M.my[bot]);
            const int i = c.i, j = c.j, k = c.k;
            T *f = arr(M.bw) + q;
            T g[2 * DIM + 1], r = T(0), p = T(0);
            g[0] = L.bx[q];
            g[1] = *((i < nx - 1) ? L.bx + q + 1 : L.bxh + j + ny * k);
            g[2] = L.by[q];
            g[3] = *((j < ny - 1) ? L.by + q + nx : L.byh + i + nx * k);
            if constexpr (DIM == 3) {
                g[4] = L.bz[q];
                g[5] = *((k < nz - 1) ? L.bz + q + nx * ny : L.bzh + i + nx * j);
            }
            g[2 * DIM] = alpha_at(L, q);
            if (bot == 0) {
                r = L.rhs[q];
                if (!zero) p = L.phi[q];
            }
#pragma unroll
            for (int d = 0; d < 2 * DIM + 1; ++d) f[d * n] = g[d];
            if (bot == 0) {
                arr(M.br)[q] = r;
                arr(M.E[0])[q] = p;
            }
        }
        if (lm) {
            Pm = make_pair<DIM, T>(LV.l[lm], Rm, om.s);
            scale_tiny(Pm);
            tiny0 = Pm.tiny[0];
            tiny1 = Pm.tiny[1];
            if constexpr (PARK) {
                T *f = arr(M.park) + t;
#pragma unroll
                for (int c = 0; c < 2; ++c) {
#pragma unroll
                    for (int d = 0; d < 2 * DIM; ++d) f[(c * 2 * DIM + d) * M.mid] = Pm.w[c][d];
                    f[(4 * DIM + c) * M.mid] = Pm.den[c];
                    f[(4 * DIM + 2 + c) * M.mid] = Pm.inv[c];
                }
            }
        }
        if (bot > 0) {
#pragma unroll
            for (int a = 0; a < NP; ++a)
                if (o0[a].on) {
                    ref(o0[a].at) = o0[a].s ? v0[a].b : v0[a].a;
                    ref(o0[a].at + C0) = o0[a].s ? v0[a].a : v0[a].b;
                }
            const int none = ((L0.nx >> 1) * L0.ny * L0.nz) * (int)sizeof(T);
            if (t < 2) ref(none + t * C0) = T(0);
        }
        __syncthreads();
    };

    // the neighbours of the pair's cell of colour c, in an iterate whose colours lie CS apart
    auto nbrs = [&](const PairPos &o_, int c, int CS, T oth, T *p) {
        const int d = (1 - c) * CS;
        const bool right = o_.s != (c == 1);
        const T xo = ref(o_.x[c] + d);
        p[0] = right ? oth : xo;
        p[1] = right ? xo : oth;
        p[2] = ref(o_.ym + d);
        p[3] = ref(o_.yp + d);
        if constexpr (DIM == 3) {
            p[4] = ref(o_.zm + d);
            p[5] = ref(o_.zp + d);
        }
    };
    // coarse cell (I, J, K) from the residuals of level F's pairs
    auto restricted = [&](const Lev<T> &F, int I, int J, int K) -> T {
        const int hx = F.nx >> 1;
        const T *a = arr(M.rs) + I + hx * (2 * J + (DIM == 3 ? F.ny * 2 * K : 0));
        if constexpr (DIM == 3) {
            const int sz = hx * F.ny;
            return T(0.125) * ((a[0] + a[hx]) + (a[sz] + a[sz + hx]));
        } else {
            return T(0.25) * (a[0] + a[hx]);
        }
    };
    // right side and zero iterate of level l > 0 (and a barrier)
    auto to_level = [&](int l) {
        const Lev<T> &F = LV.l[l - 1], &C = LV.l[l];
        if (l == bot) {
            const int n = C.nx * C.ny * C.nz;
            for (int q = t; q < n; q += NT) {
                const Ijk c = ijk_of(q, C.nx, C.ny, M.mx[l], M.my[l]);
                arr(M.br)[q] = restricted(F, c.i, c.j, c.k);
                arr(M.E[l])[q] = T(0);
            }
        } else if (lm == l) {
            PairPos pos;
            if constexpr (PARK) pos = pair_pos<DIM, T>(C, qm, M.S[l], M.mx[l], M.my[l]);
            else pos = om;
            const T a = restricted(F, 2 * pos.m, pos.j, pos.k), b = restricted(F, 2 * pos.m + 1, pos.j, pos.k);
            const T r0 = (pos.s ? b : a) * (tiny0 ? tiny_up<T>() : T(1));
            const T r1 = (pos.s ? a : b) * (tiny1 ? tiny_up<T>() : T(1));
            if constexpr (PARK) {
                arr(M.park)[(4 * DIM + 4) * M.mid + t] = r0;
                arr(M.park)[(4 * DIM + 5) * M.mid + t] = r1;
            } else {
                Pm.rhs[0] = r0;
                Pm.rhs[1] = r1;
            }
            ref(pos.at) = T(0);
            ref(pos.at + CM) = T(0);
        }
        __syncthreads();
    };
    // The pairs P of level l (N a thread, colours CS apart) down: `nu1` sweeps,
    // the residual, the next level's right side; or up: the prolongation of
    // level l + 1, nu2 sweeps, the values for the level above
    auto leg = [&](int l, bool up, auto CSt, auto &P, const auto &pos, auto &&on) {
        constexpr int N = sizeof(P) / sizeof(P[0]), CS = decltype(CSt)::value;
        const Lev<T> L = held_ih2(LV.l[l]);
        T v[N][2];
#pragma unroll
        for (int a = 0; a < N; ++a) {
            v[a][0] = v[a][1] = T(0);
            if (!on(a)) continue;
            v[a][0] = ref(pos[a].at);
            v[a][1] = ref(pos[a].at + CS);
            if (up) {
                const Lev<T> &C = LV.l[l + 1];
                const T *e = arr(M.E[l + 1]);
                auto at = [&](int I, int J, int K) { return e[I + C.nx * (J + C.ny * K)]; };
                const Two<T> d =
                    prolong_pair<DIM, T>(C.nx, C.ny, C.nz, o.bc, 2 * pos[a].m, pos[a].j, pos[a].k, at);
                v[a][0] = v[a][0] + (pos[a].s ? d.b : d.a);
                v[a][1] = v[a][1] + (pos[a].s ? d.a : d.b);
                ref(pos[a].at) = v[a][0];   // read and written by this thread only until the barrier
                ref(pos[a].at + CS) = v[a][1];
            }
        }
        if (up) __syncthreads();
        const T omega = l == 0 ? L.omega : T(1);
        const bool sor = omega != T(1);
        const int count = up ? o.nu2 : o.nu1;
        for (int it = 0; it < count; ++it)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
#pragma unroll
                for (int a = 0; a < N; ++a)
                    if (on(a)) {
                        T p[2 * DIM];
                        nbrs(pos[a], c, CS, v[a][1 - c], p);
                        v[a][c] = pair_update<DIM, T>(L, P[a], c, p, v[a][c], sor, omega);
                        ref(pos[a].at + c * CS) = v[a][c];
                    }
                __syncthreads();
            }
#pragma unroll
        for (int a = 0; a < N; ++a) {
            if (!on(a)) continue;
            if (up) {
                const T lo = pos[a].s ? v[a][1] : v[a][0], hi = pos[a].s ? v[a][0] : v[a][1];
                if (l == 0) store2(L.phi + 2 * pos[a].q, lo, hi);
                else store2(arr(M.E[l]) + 2 * pos[a].q, lo, hi);
                continue;
            }
            T r[2], ap[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                T p[2 * DIM];
                nbrs(pos[a], c, CS, v[a][1 - c], p);
                ap[c] = apply_w<DIM, T>(L, P[a].w[c], p, v[a][c]);
            }
            true_scale(P[a], r, ap);
            if (L.alpha) {
#pragma unroll
                for (int c = 0; c < 2; ++c)
                    ap[c] = dfma(L.alpha[2 * pos[a].q + (pos[a].s != (c == 1) ? 1 : 0)], v[a][c], ap[c]);
            }
            arr(M.rs)[pos[a].q] = (r[0] - ap[0]) + (r[1] - ap[1]);
        }
        if (!up || l > 0) __syncthreads();
        if (!up) to_level(l + 1);
    };
    auto leg_mid = [&](int l, bool up) {
        if constexpr (PARK) {
            Pair<DIM, T> P[1] = {dead_pair<DIM, T>()};
            const PairPos pos[1] = {pair_pos<DIM, T>(LV.l[l], lm == l ? qm : 0, M.S[l], M.mx[l], M.my[l])};
            if (lm == l) {
                const T *f = arr(M.park) + t;
#pragma unroll
                for (int c = 0; c < 2; ++c) {
#pragma unroll
                    for (int d = 0; d < 2 * DIM; ++d) P[0].w[c][d] = f[(c * 2 * DIM + d) * M.mid];
                    P[0].den[c] = f[(4 * DIM + c) * M.mid];
                    P[0].inv[c] = f[(4 * DIM + 2 + c) * M.mid];
                    P[0].rhs[c] = f[(4 * DIM + 4 + c) * M.mid];
                }
                P[0].tiny[0] = tiny0;
                P[0].tiny[1] = tiny1;
            }
            leg(l, up, std::integral_constant<int, CM>{}, P, pos, [&](int) { return lm == l; });
        } else {
            Pair<DIM, T>(&P)[1] = *reinterpret_cast<Pair<DIM, T>(*)[1]>(&Pm);
            const PairPos(&pos)[1] = *reinterpret_cast<const PairPos(*)[1]>(&om);
            leg(l, up, std::integral_constant<int, CM>{}, P, pos, [&](int) { return lm == l; });
        }
    };
    auto bottom = [&]() {
        const Lev<T> &L = LV.l[bot];
        const int n = L.nx * L.ny * L.nz;
        T *E = arr(M.E[bot]);
        const T *R = arr(M.br);
        auto cell = [&](int q, T *w, T &a, int &colour) {
            const T *f = arr(M.bw) + q;
#pragma unroll
            for (int d = 0; d < 2 * DIM; ++d) w[d] = f[d * n];
            a = f[2 * DIM * n];
            const Ijk c = ijk_of(q, L.nx, L.ny, M.mx[bot], M.my[bot]);
            colour = (c.i + c.j + c.k) & 1;
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
                const T v = bottom_solve<DIM, T>(L, X, w, a, colour, E[q], R[q], o, n);
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
                const T v = bottom_solve<DIM, T>(L, X, w, a, colour, live ? E[q] : T(0), live ? R[q] : T(0), o, n);
                if (live) E[t] = v;
            }
        } else {
            const bool live = t < n;
            const int q = live ? t : 0;
            cell(q, w, a, colour);
            auto block = [&](auto FC) __attribute__((always_inline)) {
                BottomBlock<DIM, decltype(FC)::value> X;
                X.live = live;
                X.n = held(n);
                X.flip = X.fs = X.bar = 0;
                X.xs = reinterpret_cast<double *>(smem_ + M.xs);
                X.sh = reinterpret_cast<double *>(smem_ + M.sh);
                X.last = reinterpret_cast<int *>(X.sh + 64);
                if (t == 0) X.xs[0] = X.xs[n + 1] = 0.0;
                if (t == 0) *X.last = 0;
                if (t < 64) X.sh[t] = 0.0;
                if ((t & ~63) < n) {
                    cell_nbrs<DIM, T>(L, q, -1, X.nb);
                    X.sync();   // the zeros above
                    const T v = bottom_solve<DIM, T>(L, X, w, a, colour, live ? E[q] : T(0), live ? R[q] : T(0), o, n);
                    if (live) E[t] = v;
                    X.finish();
                } else {
                    X.idle();
                }
            };
            if (n > 512) block(std::true_type{});
            else block(std::false_type{});
        }
        __syncthreads();
    };
    // Level 0's pairs, from global memory (L2) on the way down and up: held in
    // registers through the levels below they would spill.  In FP32 they load
    // together with the rest of the stage; FP64 has no registers for that.
    {
        PairRaw<DIM, T> R0[NP];
        Pair<DIM, T> P0[NP];
        PairPos o0[NP];
#pragma unroll
        for (int a = 0; a < NP; ++a) o0[a] = pair_pos<DIM, T>(L0, t + a * NT, 0, M.mx[0], M.my[0]);
        auto load0 = [&]() {
#pragma unroll
            for (int a = 0; a < NP; ++a) R0[a] = load_raw<DIM, T>(L0, 2 * o0[a].m, o0[a].j, o0[a].k);
        };
        if (sizeof(T) == 4 && bot > 0) load0();
        stage(o0);
        if (bot > 0) {
            if (sizeof(T) == 8) load0();
#pragma unroll
            for (int a = 0; a < NP; ++a) P0[a] = make_pair<DIM, T>(L0, R0[a], o0[a].s);
#pragma unroll
            for (int a = 0; a < NP; ++a) scale_tiny(P0[a]);
            leg(0, false, std::integral_constant<int, C0>{}, P0, o0, [&](int a) { return o0[a].on; });
        }
    }
    if constexpr (VC) {
        for (int l = 1; l < bot; ++l) leg_mid(l, false);
        bottom();
        for (int l = bot - 1; l > 0; --l) leg_mid(l, true);
    } else {
        // W and F cycles, without recursion.  Going down, each level owes a
        // second visit of the next coarser level (bit l of `again`; bit l of
        // `again_w`: that visit is a W, else a V); going up, a level that
        // owes one turns back down before its prolongation.  The first visit
        // has the shape of the visiting level.  The masks are the same in
        // every thread, so the block stays in step.
        bool w = o.cycle == MAC_CYCLE_W;   // shape of the current visit (W, or F/V below)
        bool v = false;                     // the current visit is a V
        unsigned again = 1u, again_w = w ? 1u : 0u;
        int l = min(1, bot);
        for (;;) {
            for (; l < bot; ++l) {
                leg_mid(l, false);
                if (!v) {
                    again |= 1u << l;
                    if (w) again_w |= 1u << l;
                    else again_w &= ~(1u << l);
                }
            }
            bottom();
            bool down = false;
            for (--l; l >= 0; --l) {
                if (again & (1u << l)) {   // second visit of level l + 1
                    again &= ~(1u << l);
                    w = (again_w >> l) & 1u;
                    v = !w;
                    ++l;
                    down = true;
                    break;
                }
                if (l > 0) leg_mid(l, true);
            }
            if (!down) break;
        }
    }
    if (bot > 0) {
        int tp = t;
        asm volatile("" : "+v"(tp));   // positions and addresses made again, not kept
        Pair<DIM, T> P0[NP];
        PairPos o0[NP];
#pragma unroll
        for (int a = 0; a < NP; ++a) {
            o0[a] = pair_pos<DIM, T>(L0, tp + a * NT, 0, M.mx[0], M.my[0]);
            P0[a] = load_pair<DIM, T>(L0, 2 * o0[a].m, o0[a].j, o0[a].k);
        }
#pragma unroll
        for (int a = 0; a < NP; ++a) scale_tiny(P0[a]);
        leg(0, true, std::integral_constant<int, C0>{}, P0, o0, [&](int a) { return o0[a].on; });
    } else {
        const int n = L0.nx * L0.ny * L0.nz;
        for (int q = t; q < n; q += NT) L0.phi[q] = arr(M.E[0])[q];
    }
}

// the LDS image of a cycle over levs[lc .. nlev - 1]; false if it has none
template <typename T>
static bool coarse_map(int dim, const Lev<T> *levs, int lc, int nlev, CoarseMap &M)
{
    M = CoarseMap{};
    M.nl = nlev - lc;
    if (M.nl < 1 || M.nl > COARSE_LEVELS) return false;
    long off = 0, mid = 0;
    auto take = [&](long bytes) {
        const long r = off;
        off += (bytes + 15) / 16 * 16;
        return (int)r;
    };
    const long sz = sizeof(T);
    for (int a = 0; a < M.nl; ++a) {
        const Lev<T> &L = levs[lc + a];
        const long n = (long)L.nx * L.ny * L.nz;
        const bool bottom = a == M.nl - 1;
        if (n > (bottom ? COARSE_BOTTOM : COARSE_CELLS)) return false;
        M.mx[a] = fast_div_factor(bottom ? L.nx : std::max(1, L.nx / 2));
        M.my[a] = fast_div_factor(L.ny);
        if (bottom) {
            M.bw = take((2 * dim + 1) * n * sz);
            M.br = take(n * sz);
            M.E[a] = take(n * sz);
            continue;
        }
        if ((L.nx & 1) || (L.ny & 1) || (dim == 3 && (L.nz & 1))) return false;
        if (a == 0) {
            M.S[0] = take(2 * colour0<T>());
            M.rs = take(n / 2 * sz);
            continue;
        }
        mid += n / 2;
        if (n / 2 >= COARSE_MID || mid > COARSE_THREADS) return false;   // a thread per pair
        M.S[a] = take(2 * colour_mid<T>());
        M.E[a] = take(n * sz);
    }
    const Lev<T> &B = levs[nlev - 1];
    const long nb = (long)B.nx * B.ny * B.nz;
    M.xs = take(nb > 64 ? 2 * (nb + 1) * 8 : 0);
    M.sh = take(nb > 64 ? 65 * 8 : 0);
    M.mid = (int)mid;
    M.park = take(dim == 3 ? 18 * mid * sz : 0);   // 12 weights, diagonals, reciprocals, right sides
    M.bytes = (int)off;
    return off <= COARSE_LDS;
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
