// mac_sweep2.hip -- two red-black sweeps of a large 3D level in one pass over
// memory (gfx950).
//
// A sweep reads an iterate, three weights and the right side and writes an
// iterate; on levels beyond the caches the single-sweep kernels run at 75 to 85%
// of what this card's memory gives, so the way to a faster pair of sweeps is
// to read everything once for both.  k_sweep2 marches a column tile through z
// with the four half-sweeps (red, black, red, black) one plane behind each
// other: at step k the first red half-sweep updates plane k, the first black
// one plane k - 1, the second red one k - 2 and the second black one k - 3, which
// is then final.  Each half-sweep needs, in its plane, only the other colour
// as the half-sweep before left it one step earlier, so one barrier a step
// orders all four.  Tiles overlap by 4 cells in x and y (and chunks by 3
// planes in z), where the updates are repeated; the arithmetic per cell is
// gs_value's, so the result equals two single sweeps bit for bit.
//
// Layout: a thread holds the pair of columns (2m, 2m + 1), one red and one
// black on every plane, with the weights of the four planes in flight in
// registers; the diagonal is inverted once for the two updates it serves.
// LDS holds, per half-sweep and split by colour, the plane that the next one
// reads (two buffers each): neighbours in x and y lie at consecutive addresses
// and immediate offsets.  The lanes of a wave hold rows of one parity, so
// which column is red is uniform in a wave and known at compile time in the
// march (two instances of it, by the parity of row + plane).
//
// Measured: a pair on 512^3 FP32 takes 1.19 ms for the 3.2 GB it cannot do
// without (2.7 TB/s; two single sweeps 2.19 ms), on 256^3 FP64 0.28 ms for 0.81
// GB (2.9 TB/s; 0.35 ms).  Bound by the chain of a step, the waves waiting for
// 47% (512^3 FP32) and 56% (256^3 FP64) of their cycles: the four updates follow each other through LDS and one
// barrier, and the registers for the weights of four planes leave room for one
// block per CU.  Loads by 64-bit address instead of buffer descriptors took
// 1.47 ms at 512^3.
#include <algorithm>

#include "mac_launch.h"

namespace mac {

struct Sweep2Grid {
    int ntx, nty;    // column tiles
    int tz;          // planes per chunk
    int total, per_xcd;
};

// c ? a : b of values (the operator on two variables selects an address, which
// would keep them in memory)
template <typename T>
__device__ __forceinline__ T pick(bool c, T a, T b)
{
    return c ? a : b;
}

// 1 / d of a diagonal: the hardware's approximation and Newton steps, the last
// of which gives the correctly rounded value (P. Markstein, IBM J. Res. Dev.
// 34 (1990) 111-119; a d with all mantissa bits set may be one off, which quot
// makes good).  A division does the same with scaling for the ends of the
// exponent range; there (quot_ok) the march divides.
__device__ __forceinline__ float recip(float d)
{
    const float r = __builtin_amdgcn_rcpf(d);
    return dfma(dfma(-d, r, 1.0f), r, r);
}
__device__ __forceinline__ double recip(double d)
{
    double r = __builtin_amdgcn_rcp(d);
    r = dfma(dfma(-d, r, 1.0), r, r);
    return dfma(dfma(-d, r, 1.0), r, r);
}

template <typename T>
struct __align__(2 * sizeof(T)) Cols {
    T a, b;
};

// HX pairs x RY rows per block (the tile and its halo), one thread each.
// ZERO: the old iterate is zero and not read.  AL: the level has alpha.
template <typename T, int HX, int RY, bool ZERO, bool AL, bool SOR>
__global__ void __launch_bounds__(HX *RY) k_sweep2(Lev<T> L, const T *__restrict__ pin, T *__restrict__ pout,
                                                   Sweep2Grid G)
{
    using T2 = Cols<T>;
    constexpr int NW = HX * RY / 64, RW = 64 / HX;          // waves, rows of a wave
    static_assert(NW % 2 == 0 && NW * RW == RY, "the rows of a wave have one parity");
    constexpr int TX = 2 * HX - 8, TY = RY - 8;
    constexpr int PX = HX + 2, NPOS = PX * (RY + 2);
    constexpr unsigned ES = sizeof(T);
    const int b = blockIdx.x, idx = (b & 7) * G.per_xcd + (b >> 3);   // neighbouring tiles on one XCD
    if (idx >= G.total) return;
    const int nt = G.ntx * G.nty, chunk = idx / nt, tile = idx - chunk * nt;
    const int tyi = tile / G.ntx, txi = tile - tyi * G.ntx;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const unsigned plane = (unsigned)nx * (unsigned)ny;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m = lane % HX, j = wv + NW * (lane / HX);
    const int gi = txi * TX - 4 + 2 * m, gj = tyi * TY - 4 + j;
    // the column's image in the domain (a tile may span several periods)
    int wi = gi, wj = gj;
    if (L.perx) {
        while (wi < 0) wi += nx;
        while (wi >= nx) wi -= nx;
    }
    if (L.pery) {
        while (wj < 0) wj += ny;
        while (wj >= ny) wj -= ny;
    }
    const bool live = (unsigned)wi < (unsigned)nx && (unsigned)wj < (unsigned)ny;
    if (!live) wi = wj = 0;
    const bool out = m >= 2 && m < 2 + TX / 2 && j >= 4 && j < 4 + TY && gi < nx && gj < ny;
    const bool xend = wi + 2 == nx, yend = wj == ny - 1;
    const bool any_dead = __any(!live), any_xend = __any(xend), any_yend = __any(yend);
    const int z0 = chunk * G.tz, z1 = min(z0 + G.tz, nz), ks = z0 - 3;
    // byte offsets within a plane
    const unsigned col = (unsigned)wi + (unsigned)nx * (unsigned)wj;
    const unsigned vc = col * ES, vx2 = (xend ? col : col + 2) * ES, vyn = (yend ? col : col + (unsigned)nx) * ES;
    const unsigned vxh = (unsigned)wj * ES, vyh = (unsigned)wi * ES;
    const __amdgpu_buffer_rsrc_t Rx = buf_rsrc(L.bx), Ry = buf_rsrc(L.by), Rz = buf_rsrc(L.bz), Rr = buf_rsrc(L.rhs);
    const __amdgpu_buffer_rsrc_t Rp = buf_rsrc(pin), Ro = buf_rsrc(pout), Rxh = buf_rsrc(L.bxh), Ryh = buf_rsrc(L.byh);
    const T ih2x = L.ih2x, ih2y = L.ih2y, ih2z = L.ih2z, omega = L.omega;
    __shared__ T A[4][2][NPOS];   // [half-sweep that reads it][buffer]
    for (int q = threadIdx.x; q < 8 * NPOS; q += HX * RY) (&A[0][0][0])[q] = T(0);
    const int pos = (m + 1) + PX * (j + 1);

    // A plane's place in memory, stepped one plane at a time: wrapped where z
    // is periodic, plane 0 standing in for one outside (ok false)
    struct Pl {
        int k, kw;
        bool ok, top;
        unsigned o;   // byte offset of a cell array's plane
    };
    const int perz = L.perz;
    const bool below = !perz && z0 == 0;   // the march starts outside the domain
    auto place = [&](Pl &q) {
        q.ok = perz || (unsigned)q.k < (unsigned)nz;
        const int kw = perz ? q.kw : (q.ok ? q.k : 0);
        q.top = q.ok && kw == nz - 1;
        q.o = (unsigned)kw * plane * ES;
    };
    auto first = [&](int k) -> Pl {
        Pl q;
        q.k = k;
        q.kw = ((k % nz) + nz) % nz;
        place(q);
        return q;
    };
    auto next = [&](const Pl &q) -> Pl {
        Pl r;
        r.k = q.k + 1;
        r.kw = q.kw + 1 == nz ? 0 : q.kw + 1;
        place(r);
        return r;
    };
    auto load_z = [&](const Pl &q) -> T2 { return ld_rs<T2>(Rz, vc, q.o); };
    auto load_p = [&](const Pl &q) -> T2 {
        T2 v{T(0), T(0)};
        if constexpr (!ZERO) {
            v = ld_rs<T2>(Rp, vc, q.o);
            if (any_dead || !q.ok) {
                const bool in = live && q.ok;
                v.a = pick(in, v.a, T(0));
                v.b = pick(in, v.b, T(0));
            }
        }
        return v;
    };
    // the weights of a plane as loaded
    T2 rx, ryl, ryh, rr, ra{T(-0.0), T(-0.0)};
    T rx2;
    auto load_w = [&](const Pl &q) __attribute__((always_inline)) {
        rx = ld_rs<T2>(Rx, vc, q.o);
        rx2 = ld_rs<T>(Rx, vx2, q.o);
        ryl = ld_rs<T2>(Ry, vc, q.o);
        ryh = ld_rs<T2>(Ry, vyn, q.o);
        rr = ld_rs<T2>(Rr, vc, q.o);
        if constexpr (AL) ra = ld_rs<T2>(buf_rsrc(L.alpha), vc, q.o);
        if (any_xend || any_yend) {   // the domain's high faces
            const unsigned kw = (unsigned)(perz ? q.kw : (q.ok ? q.k : 0));
            const T hx = ld_rs<T>(Rxh, vxh, kw * (unsigned)ny * ES);
            const T2 hy = ld_rs<T2>(Ryh, vyh, kw * (unsigned)nx * ES);
            rx2 = pick(xend, hx, rx2);
            ryh.a = pick(yend, hy.a, ryh.a);
            ryh.b = pick(yend, hy.b, ryh.b);
        }
    };
    // per plane in flight: x faces, y faces (low, high; left, right column),
    // low z faces, rhs, diagonal and its reciprocal
    struct W {
        T x0, x1, x2, yl[2], yh[2], zl[2], r[2], d[2], i[2];
    };
    W wq[4];      // planes k .. k - 3, plane p of step ks + m + S in slot S
    T v[4][2];    // their values
    T last0 = T(0), last1 = T(0), top0, top1;   // plane k - 4; the domain's high z faces
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        wq[q].x0 = wq[q].x1 = wq[q].x2 = T(0);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            wq[q].yl[c] = wq[q].yh[c] = wq[q].zl[c] = wq[q].r[c] = v[q][c] = T(0);
            wq[q].d[c] = wq[q].i[c] = T(1);
        }
    }
    {
        const T2 t = ld_rs<T2>(buf_rsrc(L.bzh), vc, 0u);
        top0 = pick(live, t.a, T(0));
        top1 = pick(live, t.b, T(0));
    }
    Pl q0 = first(ks), q1 = next(q0), q2 = next(q1);   // planes k, k + 1, k + 2
    {
        const T2 t = load_p(first(ks - 1));
        v[3][0] = t.a;
        v[3][1] = t.b;
    }
    T2 pc = load_p(q0), pn = load_p(q1);   // old values of planes k, k + 1
    T2 zc = load_z(q0), zn = load_z(q1);   // low z faces of planes k, k + 1
    unsigned long long by_div = 0;   // the lanes where quot does not serve a diagonal so far
    bool tp1 = false, tp2 = false, tp3 = false;   // whether planes k - 1, k - 2, k - 3 are the domain's top
    load_w(q0);
    __syncthreads();

    auto run = [&](auto PBC) {
        constexpr int PB = decltype(PBC)::value;   // parity of gj + ks
        auto step = [&](auto SC, int mm) __attribute__((always_inline)) {
            constexpr int S = decltype(SC)::value, B = S & 1;
            constexpr int S1 = (S + 3) & 3, S2 = (S + 2) & 3, S3 = (S + 1) & 3;   // planes k - 1, k - 2, k - 3
            constexpr int R0 = (PB + S) & 1;                                     // plane k's red column
            constexpr int R1 = R0 ^ 1, R2 = R0, R3 = R0 ^ 1;                     // of planes k - 1 .. k - 3
            const int k = ks + mm + S;
            // ---- plane k enters; loads for the next step
            last0 = v[S][0];
            last1 = v[S][1];
            v[S][0] = pc.a;
            v[S][1] = pc.b;
            pc = pn;
            W &w = wq[S];
            w.x0 = rx.a; w.x1 = rx.b; w.x2 = rx2;
            w.yl[0] = ryl.a; w.yl[1] = ryl.b;
            w.yh[0] = ryh.a; w.yh[1] = ryh.b;
            w.zl[0] = zc.a; w.zl[1] = zc.b;
            w.r[0] = rr.a; w.r[1] = rr.b;
            const bool tp0 = q0.top;
            T zh0 = pick(tp0, top0, zn.a), zh1 = pick(tp0, top1, zn.b);
            w.d[0] = dfma(ih2x, w.x0 + w.x1, dfma(ih2y, w.yl[0] + w.yh[0], ih2z * (w.zl[0] + zh0))) + ra.a;
            w.d[1] = dfma(ih2x, w.x1 + w.x2, dfma(ih2y, w.yl[1] + w.yh[1], ih2z * (w.zl[1] + zh1))) + ra.b;
            if (any_dead || !q0.ok) {   // cells outside stay zero
                const bool in = live && q0.ok;
                zh0 = pick(in, zh0, T(0));
                zh1 = pick(in, zh1, T(0));
                w.x0 = pick(in, w.x0, T(0)); w.x1 = pick(in, w.x1, T(0)); w.x2 = pick(in, w.x2, T(0));
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    w.yl[c] = pick(in, w.yl[c], T(0));
                    w.yh[c] = pick(in, w.yh[c], T(0));
                    w.zl[c] = pick(in, w.zl[c], T(0));
                    w.r[c] = pick(in, w.r[c], T(0));
                    w.d[c] = pick(in, w.d[c], T(1));
                }
            }
            w.i[0] = recip(w.d[0]);
            w.i[1] = recip(w.d[1]);
            by_div |= __ballot(!quot_ok(w.d[0], w.d[1]));
            zc = zn;
            load_w(q1);
            zn = load_z(q2);
            pn = load_p(q2);
            q0 = q1;
            q1 = q2;
            q2 = next(q2);
            // ---- the old black values of plane k
            A[0][B][pos] = v[S][R0 ^ 1];
            __syncthreads();
            // the update of column C of plane p: O its plane's other colour in
            // LDS, zm, zp the column's values below and above, zh its high z face
            auto update = [&](auto CC, auto DC, const W &q, const T *O, T own, T oth, T zm, T zp, T zh) -> T {
                constexpr int C = decltype(CC)::value;
                constexpr bool DIV = decltype(DC)::value;
                const T xo = O[C ? pos + 1 : pos - 1];
                const T tx = dfma(C ? T(q.x1) : T(q.x0), C ? T(oth) : T(xo),
                                  (C ? T(q.x2) : T(q.x1)) * (C ? T(xo) : T(oth)));
                const T ty = dfma(q.yl[C], O[pos - PX], q.yh[C] * O[pos + PX]);
                const T tz = dfma(q.zl[C], zm, zh * zp);
                const T num = dfma(ih2x, tx, dfma(ih2y, ty, dfma(ih2z, tz, q.r[C])));
                return relax<SOR>(DIV ? num / q.d[C] : quot(num, q.d[C], q.i[C]), own, omega);
            };
            using CA = std::integral_constant<int, R0>;
            using CB = std::integral_constant<int, R0 ^ 1>;
            // high z faces of plane k - b: the next plane's low ones or the
            // domain's; none on a plane below the domain, whose cells stay zero
            auto zhi = [&](int b, bool t, T above) -> T {
                const T a = pick(t, R0 ? T(top1) : T(top0), above);
                return pick(below && k - b < 0, T(0), a);
            };
            auto halves = [&](auto DC) __attribute__((always_inline)) {
                // first red half-sweep, plane k, column R0
                v[S][R0] = update(CA{}, DC, w, A[0][B], v[S][R0], v[S][R0 ^ 1], v[S1][R0], R0 ? T(pc.b) : T(pc.a),
                                  R0 ? T(zh1) : T(zh0));
                A[1][B][pos] = v[S][R0];
                // first black half-sweep, plane k - 1: its black column is R1 ^ 1 = R0
                v[S1][R0] = update(CA{}, DC, wq[S1], A[1][B ^ 1], v[S1][R0], v[S1][R1], v[S2][R0], v[S][R0],
                                   zhi(1, tp1, w.zl[R0]));
                A[2][B ^ 1][pos] = v[S1][R0];
                // second red, plane k - 2, column R2 = R0
                v[S2][R2] = update(CA{}, DC, wq[S2], A[2][B], v[S2][R2], v[S2][R2 ^ 1], v[S3][R2], v[S1][R2],
                                   zhi(2, tp2, wq[S1].zl[R0]));
                A[3][B][pos] = v[S2][R2];
                // second black, plane k - 3, column R3 ^ 1 = R0
                v[S3][R0] = update(CA{}, DC, wq[S3], A[3][B ^ 1], v[S3][R0], v[S3][R3], R0 ? T(last1) : T(last0),
                                   v[S2][R0], zhi(3, tp3, wq[S2].zl[R0]));
            };
            // a scalar branch on the ballot keeps the second form out of the march
            // (0.5 us a launch; a branch on a lane mask 1.5, a test in each update
            // 1.5% of a 256^3 FP64 pair)
            if (__builtin_expect(by_div != 0, 0)) halves(std::true_type{});
            else halves(std::false_type{});
            tp3 = tp2;
            tp2 = tp1;
            tp1 = tp0;
            const int kd = k - 3;
            if (out && kd >= z0 && kd < z1)
                st_rs<T2, CPOL_NT>(Ro, vc, (unsigned)kd * plane * ES, T2{v[S3][0], v[S3][1]});
        };
        const int n = z1 + 3 - ks;
        for (int mm = 0; mm < n; mm += 4) {
            step(std::integral_constant<int, 0>{}, mm);
            step(std::integral_constant<int, 1>{}, mm);
            step(std::integral_constant<int, 2>{}, mm);
            step(std::integral_constant<int, 3>{}, mm);
        }
    };
    if ((tyi * TY - 4 + wv + ks) & 1) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 0>{});
}

// Chunks in z: the fewest steps in the longest chain of blocks on one of the
// device's block slots, a block taking its planes, the 6 of the pipeline and
// about 4 to start.
static int chunk_planes(int nz, int tiles, int slots)
{
    long best = -1;
    int best_tz = nz;
    for (int zc = 1; zc <= std::max(1, nz / 4); ++zc) {
        const int tz = (nz + zc - 1) / zc, n = (nz + tz - 1) / tz;
        const long rounds = ((long)tiles * n + slots - 1) / slots, steps = (tz + 6 + 3) / 4 * 4;
        const long cost = rounds * (steps + 4);
        if (best < 0 || cost < best) {
            best = cost;
            best_tz = tz;
        }
    }
    return best_tz;
}

template <typename T, int HX, int RY>
static void launch_sweep2_t(const Lev<T> &L, const T *pin, T *pout, int mode, hipStream_t s)
{
    static const int slots = [] {   // one block per CU (registers)
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
            cus = 256;
        return cus;
    }();
    Sweep2Grid G;
    G.ntx = (L.nx + 2 * HX - 9) / (2 * HX - 8);
    G.nty = (L.ny + RY - 9) / (RY - 8);
    G.tz = chunk_planes(L.nz, G.ntx * G.nty, slots);
    G.total = G.ntx * G.nty * ((L.nz + G.tz - 1) / G.tz);
    G.per_xcd = (G.total + 7) / 8;
    const dim3 g((unsigned)(8 * G.per_xcd)), b(HX * RY);
    auto go = [&](auto ZC, auto AC, auto SC) {
        hipLaunchKernelGGL((k_sweep2<T, HX, RY, decltype(ZC)::value, decltype(AC)::value, decltype(SC)::value>), g, b, 0,
                           s, L, pin, pout, G);
    };
    using Y = std::true_type;
    using N = std::false_type;
    const bool z = mode == SWEEP_ZERO, a = L.alpha != nullptr, o = L.omega != T(1);
    if (z) a ? (o ? go(Y{}, Y{}, Y{}) : go(Y{}, Y{}, N{})) : (o ? go(Y{}, N{}, Y{}) : go(Y{}, N{}, N{}));
    else a ? (o ? go(N{}, Y{}, Y{}) : go(N{}, Y{}, N{})) : (o ? go(N{}, N{}, Y{}) : go(N{}, N{}, N{}));
}

// Where a pair goes this way: wherever its layout holds it (pairs of columns;
// byte offsets within an array of 32 bits; a colour that holds across a
// periodic face), but for FP32 at nx = 128, which k_gsrb_rows sweeps out of the
// caches where the level is no larger than 128^3: there a pair takes 34.0 us in
// single sweeps and 33.4 here, from a zero iterate 30.8 and 32.6, and whole solves
// with such a level are 1 to 3% faster with the single sweeps.  The rule looks at
// nx alone; longer domains of such rows, levels with alpha and fewer than 8 planes
// (k_gsrb_deep) have not been measured either way.
// Two single sweeps (k_gsrb_rows at 128 and 256, k_gsrb_deep) and one pass,
// microseconds:
//   FP32  192^3 129, 66   256^3 215, 178   512^3 2190, 1194
//         320 x 224 x 256 352, 183   96^3 34, 24   512^3 from zero 1981, 1223
//   FP64  128^3 71, 45   192^3 258, 115   256^3 346, 278
//         320 x 224 x 256 659, 366   96 x 80 x 112 45, 27
template <typename T>
bool launch_sweep2(const Lev<T> &L, const T *pin, T *pout, int mode, hipStream_t s)
{
    if ((L.nx & 1) || (L.pery && (L.ny & 1)) || (L.perz && (L.nz & 1))) return false;
    if ((double)L.nx * L.ny * L.nz * sizeof(T) >= 4294967296.0) return false;
    if (sizeof(T) == 4 && L.nx == 128) return false;
    launch_sweep2_t<T, sizeof(T) == 4 ? 32 : 16, 32>(L, pin, pout, mode, s);
    return true;
}
template bool launch_sweep2<double>(const Lev<double> &, const double *, double *, int, hipStream_t);
template bool launch_sweep2<float>(const Lev<float> &, const float *, float *, int, hipStream_t);

}  // namespace mac
