// grid.hip -- the time-stepping kernels of the hot path on gfx950, FP64.
//
//   k_ghost_fill   periodic 2-layer face copy            comm.cpp:277-323 (serial branch)
//   k_ansatz       A[q][cell] = exp(alpha.m_q) (M_N) or alpha.m_q (P_N) on all cells
//                                                        flux_kinetic.cpp:20-37, 116-123
//   k_stencil      limited upwind differences, sum_q m_q (Fx/dx+Fy/dy+Fz/dz), optionally
//                  fused with the Euler stage             flux_kinetic.cpp:45-60, 126-196,
//                                                        update.cpp:21-37
//   k_flux_moment  P_N Fromm flux with half-range operators (nm <= 9)
//                                                        flux_moment.cpp:30-104
//   k_moment_stage the same flux, alone (nm > 9) or with the Euler stage and the RK2 average
//                                                        flux_moment.cpp:30-104,
//                                                        update.cpp:21-37, 268-274
//   k_euler        Euler stage with isotropic scattering update.cpp:21-37
//   k_rk2          uOld <- u / u <- (u + uOld)/2          update.cpp:206-212, 268-274
//   k_make_batch   synthetic closure batch (SplitMix64 counter RNG)
//
// Layout: the reference's AoS grid (src/global.h:15-16), cells (nx+4)(ny+4)(nz+4) with z
// fastest, nm moments contiguous per cell.  The ansatz is materialised ordinate-major,
// A[q*Ng + cell], so every stencil load of a wavefront is one contiguous segment.
// Every expression keeps the reference's evaluation order (no FMA contraction), so the
// results match the CPU code bit for bit whenever the exponentials agree.
#include <algorithm>
#include <cfloat>
#include <cmath>

#include "c3d_detmath.h"
#include "c3d_internal.h"
#include "c3d_tile.h"

#pragma clang fp contract(off)

namespace c3d {
namespace {

// ---------------------------------------------------------------- ghost fill
// u2, if not null, receives the same ghosts
__global__ void k_ghost_fill(Grid G, int nm, double *u, double *u2)
{
    // three slab families of 2 x 2 x (face area) cells, each copies nm moments
    const int64_t ax = (int64_t)2 * G.ny * G.nz, ay = (int64_t)2 * G.nx * G.nz,
                  az = (int64_t)2 * G.nx * G.ny;
    const int64_t total = (ax + ay + az) * 2 * nm;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total;
         t += (int64_t)gridDim.x * blockDim.x) {
        int m = (int)(t % nm);
        int64_t c = t / nm;
        int side = (int)(c & 1);  // 0: low ghosts <- high interior, 1: high <- low
        c >>= 1;
        size_t dst, src;
        if (c < ax) {
            int l = (int)(c / ((int64_t)G.ny * G.nz));
            int64_t rem = c % ((int64_t)G.ny * G.nz);
            int j = 2 + (int)(rem / G.nz), k = 2 + (int)(rem % G.nz);
            if (side == 0) {
                dst = G.idx(l, j, k);
                src = G.idx(G.nx + l, j, k);
            } else {
                dst = G.idx(G.nx + 2 + l, j, k);
                src = G.idx(2 + l, j, k);
            }
        } else if (c < ax + ay) {
            c -= ax;
            int l = (int)(c / ((int64_t)G.nx * G.nz));
            int64_t rem = c % ((int64_t)G.nx * G.nz);
            int i = 2 + (int)(rem / G.nz), k = 2 + (int)(rem % G.nz);
            if (side == 0) {
                dst = G.idx(i, l, k);
                src = G.idx(i, G.ny + l, k);
            } else {
                dst = G.idx(i, G.ny + 2 + l, k);
                src = G.idx(i, 2 + l, k);
            }
        } else {
            c -= ax + ay;
            int l = (int)(c / ((int64_t)G.nx * G.ny));
            int64_t rem = c % ((int64_t)G.nx * G.ny);
            int i = 2 + (int)(rem / G.ny), j = 2 + (int)(rem % G.ny);
            if (side == 0) {
                dst = G.idx(i, j, l);
                src = G.idx(i, j, G.nz + l);
            } else {
                dst = G.idx(i, j, G.nz + 2 + l);
                src = G.idx(i, j, 2 + l);
            }
        }
        const double v = u[src * nm + m];
        u[dst * nm + m] = v;
        if (u2)
            u2[dst * nm + m] = v;
    }
}

// ------------------------------------------------------------------- ansatz
// Row q of the ordinate table the flux kernels read as scalar operands: xi, eta, mu, w, then
// M's row.  Its loads are issued a piece ahead of their use: scalar loads return in any order,
// so a wait is for all of them, and use_s() waits for one piece before the next is issued.
constexpr int ord_row(int nm) { return 4 + nm; }
__device__ __forceinline__ void use_s(double x) { asm volatile("" ::"s"(x)); }
template <int N>
__device__ __forceinline__ void use_s(const double (&x)[N])
{
#pragma unroll
    for (int i = 0; i < N; ++i)
        use_s(x[i]);
}

// One thread per cell (all cells, ghosts included) and blockIdx.y's share of the ordinates;
// the ansatz argument keeps flux_kinetic.cpp:23-24's sequential order.  Bound by the vector
// unit (the argument without FMA contraction, then exp) and the store of A.  M's rows are
// uniform and come as scalar operands, half a row ahead; from LDS they took longer than the
// vector work at M_4.  Small grids share out the ordinates over the blocks.
// *wild is set where a value is not a number, exceeds kTame, or is not zero but below tiny (see
// k_stencil), in a cell that some stencil reads; of an exponential the argument is tested instead,
// |x - ra| <= rb, which is one comparison (M_3 61x45x77: 1% of the flux).
constexpr double kTame = 1e290;
template <int NM>
__global__ __launch_bounds__(kTB) __attribute__((amdgpu_waves_per_eu(NM == 25 ? 5 : 1))) void k_ansatz(Grid G, int64_t ng, int nq, int nqPer,
                                                 const double *__restrict__ ord,
                                                 const double *__restrict__ alpha, double *A,
                                                 int isPn, double ra, double rb, int *wild)
{
    constexpr int HA = (NM + 1) / 2, HB = NM - HA;
    const int64_t cell = (int64_t)blockIdx.x * kTB + threadIdx.x;
    const bool have = cell < ng;
    double a[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m)
        a[m] = have ? alpha[cell * NM + m] : 0.0;
    const int q0 = blockIdx.y * nqPer, q1 = min(q0 + nqPer, nq);
    if (q0 >= q1)
        return;
    const double *row = ord + (size_t)q0 * ord_row(NM) + 4;
    double *At = A + (size_t)q0 * ng + cell;
    double mA[HA];
    bool bad = false;
#pragma unroll
    for (int m = 0; m < HA; ++m)
        mA[m] = row[m];
#pragma unroll 1
    for (int q = q0; q < q1; ++q) {
        double mB[HB], kin = 0.0;
        __builtin_amdgcn_sched_barrier(0);
        use_s(mA);
#pragma unroll
        for (int m = 0; m < HB; ++m)
            mB[m] = row[HA + m];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < HA; ++m)
            kin += a[m] * mA[m];
        __builtin_amdgcn_sched_barrier(0);
        use_s(mB);
        row += ord_row(NM);  // past the last row: padding
#pragma unroll
        for (int m = 0; m < HA; ++m)
            mA[m] = row[m];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < HB; ++m)
            kin += a[HA + m] * mB[m];
        const double v = isPn == 1 ? kin : (isPn == 2 ? det_exp(kin) : exp(kin));
        if (isPn == 1)
            bad |= !(fabs(v) <= rb) || (fabs(v) < ra && v != 0.0);
        else
            bad |= !(fabs(kin - ra) <= rb);
        if (have)
            *At = v;
        At += ng;
    }
    if (have && bad && stencil_reads(G, (unsigned)cell))
        *wild = 1;
}
__global__ void k_clear_int(int *p) { *p = 0; }

__device__ __forceinline__ double sgn1(double x) { return x >= 0.0 ? 1.0 : -1.0; }
__device__ __forceinline__ double mmin(double a, double b) { return a < b ? a : b; }
__device__ __forceinline__ double mmax(double a, double b) { return a > b ? a : b; }
// flux_kinetic.cpp:45-49
__device__ __forceinline__ double minmod(double x, double y)
{
    return sgn1(x) * mmax(0.0, mmin(fabs(x), y * sgn1(x)));
}
// flux_kinetic.cpp:55-60.  TH1: theta == 1 (the minmod limiter), where th * x == x exactly.
template <bool TH1>
__device__ __forceinline__ double slopefit(double l, double c, double r, double th)
{
    if constexpr (TH1)
        return minmod(r - c, minmod(0.5 * (r - l), c - l));
    else
        return minmod(th * (r - c), minmod(0.5 * (r - l), th * (c - l)));
}
// one axis of flux_kinetic.cpp:141-191; A at offsets -2..+2 along the axis
template <bool TH1>
__device__ __forceinline__ double axis_flux(double am2, double am1, double a0, double ap1,
                                            double ap2, double dir, double wq, double th)
{
    double f;
    if (dir > 0) {
        f = a0 + 0.5 * slopefit<TH1>(am1, a0, ap1, th) - am1 -
            0.5 * slopefit<TH1>(am2, am1, a0, th);
    } else {
        f = ap1 - 0.5 * slopefit<TH1>(a0, ap1, ap2, th) - a0 +
            0.5 * slopefit<TH1>(am1, a0, ap1, th);
    }
    return f * dir * wq;
}

struct StencilArgs {
    Grid G;
    int nq;
    double dx, dy, dz, theta, dt;
    int fuseEuler;
    double rdx, rdy, rdz;  // 1/dx, ...
    int general;           // take the general path whatever the ansatz holds
};

// x / d == x * (1/d) exactly, for every x, iff d is a power of two
bool exact_reciprocal(double d)
{
    int e = 0;
    return d > 0.0 && std::isfinite(d) && std::frexp(d, &e) == 0.5 && e > -1021 && e < 1022;
}
bool exact_reciprocals(double dx, double dy, double dz)
{
    return exact_reciprocal(dx) && exact_reciprocal(dy) && exact_reciprocal(dz);
}
// the least magnitude of the ansatz that k_stencil's fast path takes
constexpr double kTinyDiv = 1e-200, kTinyP2 = 1e-270;

typedef const __attribute__((address_space(1))) double GlobalDouble;
typedef const __attribute__((address_space(1))) char GlobalByte;

// The three-way minmod that slopefit's nested one is for ordinary numbers (the common sign's
// smallest magnitude, else 0): y limited to what x and z of one sign leave of [n, p].
__device__ __forceinline__ double minmod3(double x, double y, double z)
{
    const double p = fmax(0.0, fmin(x, z)), n = fmin(0.0, fmax(x, z));
    return fmax(n, fmin(p, y));
}
// axis_flux on the four values it reads: u2, u1 upwind of the centre, a0, and d1 downwind.
// For dir <= 0 the axis is mirrored, which negates both slopes exactly.  The halves are
// moved through the minima (a factor of two commutes with every operation) to where one
// fused multiply-add, whose product is exact, adds the limited half slope.  th2 = 2 theta.
template <bool TH1>
__device__ __forceinline__ double upwind_flux(double u2, double u1, double a0, double d1,
                                              double dir, bool pos, double wq, double th2)
{
    double zA = u1 - u2, zB = a0 - u1, zC = d1 - a0, yA = a0 - u2, yB = d1 - u1;
    if constexpr (TH1) {
        yA = 0.5 * yA;
        yB = 0.5 * yB;
    } else {
        zA = th2 * zA;
        zB = th2 * zB;
        zC = th2 * zC;
    }
    constexpr double h = TH1 ? 0.5 : 0.25;
    const double sA = minmod3(zB, yA, zA), sB = minmod3(zC, yB, zB);
    double f;
    if (pos)
        f = fma(-h, sA, fma(h, sB, a0) - u1);
    else
        f = fma(-h, sB, fma(h, sA, u1) - a0);
    return f * dir * wq;
}
// x / d from the correctly rounded r = 1 / d: one residual correction gives the correctly
// rounded quotient (P. Markstein, IBM J. Res. Dev. 34, 1990) away from the ends of the
// exponent range; three operations instead of the dozen of a division.
__device__ __forceinline__ double div_by(double x, double d, double r)
{
    const double q = x * r;
    return fma(fma(-q, d, x), r, q);
}

// sum_q m_q (Fx/dx + Fy/dy + Fz/dz) for one interior cell per thread, optionally with the Euler
// stage.  Bound by the vector unit: at theta != 1 and general spacings about 105 operations for
// the three axes and 2 NM for the moments, per cell and ordinate.  What keeps it there:
//   - upwind_flux: the limiter as minima and maxima, four values an axis, the differences of
//     its two slopes shared (the nested minmod with its sign products took twice as many);
//   - div_by instead of division (or, P2: every spacing a power of two, the exact reciprocal);
//   - D ordinates' values in flight per thread: 2 where waves enough hide the latency, 4 on
//     grids that leave the chip mostly idle;
//   - the ordinate table as scalar operands, issued a stage ahead;
//   - the tiling of c3d_tile.h, for the L2.
// All of it gives the general path's bits as long as the ansatz is zero or within [tiny, kTame]
// and spacings, theta and the ordinates are within reason (launch_stencil): a value outside of
// that, or a NaN, anywhere (*wild, from k_ansatz) sends the whole call down the general path.
//
// Why tiny: every difference of ansatz values is a multiple of e = ulp(tiny), and a limited
// slope one of e / 2 (theta = 1) or of 2^-53 |theta| e, so that an axis's flux is zero or at
// least a quarter of that times |direction| and weight.  With |theta| >= 1e-15 and directions
// and weights >= 1e-20, tiny = 1e-200 leaves it above 1e-290, where div_by's residual is exact;
// without a division (P2), 1e-270 keeps the slopes' factors of two exact.
//
// Measured, ansatz and stencil together, against a kernel with 13 loads, the nested limiter and
// divisions: M_3 Q = 12 theta = 2 61x45x77: 945 -> 760 us; 96x128x128: 5.64 -> 4.50 ms; 16x12x20:
// 545 -> 207 us; M_2 Q = 8 20^3 218 -> 79 us, 128^3 3.02 -> 2.53 ms.  At M_2 128^3 (theta 1, powers of
// two) it issues 97 vector instructions per cell and ordinate, the vector unit busy 46% of the
// time; the L1 serves 10 unaligned rows per cell and ordinate.
// The waves of a SIMD that the fast path's registers leave room for (D = 2), for the general path
// and the Euler stage to keep to.
constexpr int stencil_waves(int nm, int d) { return d > 2 ? 1 : (nm <= 9 ? 5 : 4); }
template <int NM, bool P2, bool TH1, int D>
__global__ __launch_bounds__(kTB) __attribute__((amdgpu_waves_per_eu(stencil_waves(NM, D)))) void k_stencil(StencilArgs S, const double *__restrict__ A,
                                                  const double *__restrict__ ord,
                                                  const int *__restrict__ sgn,
                                                  const int *__restrict__ wild, double *flux,
                                                  double *u, const double *__restrict__ sigT,
                                                  const double *__restrict__ sigS)
{
    constexpr int OR = ord_row(NM);
    constexpr int TB = D > 2 ? kTBSmall : kTB;  // as launched
    const Grid &G = S.G;
    Tile T;
    if (!tile_of(G, blockIdx.x, gridDim.x, TB, T))
        return;
    // lanes past the run's end work on its last cell and write nothing; waves past it leave
    const TileCell tc = tile_cell(G, T, threadIdx.x);
    const bool have = tc.have;
    if (__ballot(have) == 0)
        return;
    const size_t ng = (size_t)G.NX * G.NY * G.NZ;
    // cells from the start of the tile's first plane
    const unsigned in =
        ((unsigned)tc.di * (unsigned)G.NY + (unsigned)tc.j) * (unsigned)G.NZ + (unsigned)tc.k;
    const ptrdiff_t sx = (ptrdiff_t)G.NY * G.NZ, sy = G.NZ;
    double fl[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m)
        fl[m] = 0.0;
    if (!S.general && *wild == 0) {
        const double *plane = A + (size_t)T.i * sx;
        // the values of the ordinate at plane b whose direction signs are sg (bits x, y, z; set:
        // positive)
        auto load = [&](double(&v)[10], const double *b, int sg) {
            unsigned off = 8u * in;
            asm("" : "+v"(off));  // widened here, next to the loads
            auto at = [&](ptrdiff_t o) {
                // the base stays scalar: one register offset serves every load
                uint64_t base = (uint64_t)(b + o);
                asm("" : "+s"(base));
                return *(GlobalDouble *)((GlobalByte *)base + off);
            };
            v[0] = at(0);
#pragma unroll
            for (int ax = 0; ax < 3; ++ax) {
                const ptrdiff_t st = ax == 0 ? sx : (ax == 1 ? sy : 1);
                const ptrdiff_t up = (sg >> ax) & 1 ? -st : st;
                v[1 + 3 * ax] = at(2 * up);
                v[2 + 3 * ax] = at(up);
                v[3 + 3 * ax] = at(-up);
            }
        };
        double v[D][10], dirs[4];
        int sNow[D], sNext;  // signs of the ordinates in v; of the one loaded next
#pragma unroll
        for (int d = 0; d < D; ++d) {
            sNow[d] = sgn[d];
            load(v[d], plane, sNow[d]);
            plane += d + 1 < S.nq ? ng : 0;
            __builtin_amdgcn_sched_barrier(0);  // in order, as the counted waits need them
        }
        sNext = sgn[D];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            dirs[e] = ord[e];
        const double *row = ord;
        // the scalar registers are for the ordinate table: the constants go to vector ones
        double th2 = 2.0 * S.theta, hx = S.dx, hy = S.dy, hz = S.dz, rx = S.rdx, ry = S.rdy,
               rz = S.rdz;
        asm("" : "+v"(th2), "+v"(hx), "+v"(hy), "+v"(hz), "+v"(rx), "+v"(ry), "+v"(rz));
        auto ordinate = [&](int d, int q) {
            // M's row in pieces of at most nine, for the scalar registers; a piece is issued
            // before the one ahead of it is used
            constexpr int PS = NM <= 9 ? NM : (NM == 16 ? 8 : 9), NP = (NM + PS - 1) / PS;
            double m[2][PS];
            auto piece = [&](int p) {
#pragma unroll
                for (int i = 0; i < PS; ++i)
                    m[p & 1][i] = p * PS + i < NM ? row[4 + p * PS + i] : 0.0;
            };
            __builtin_amdgcn_sched_barrier(0);
            use_s(dirs);
            asm volatile("" ::"s"(sNext));
            piece(0);
            __builtin_amdgcn_sched_barrier(0);
            const int sg = sNow[d];
            const double(&w)[10] = v[d];
            const double wq = dirs[3];
            const double fX = upwind_flux<TH1>(w[1], w[2], w[0], w[3], dirs[0], sg & 1, wq, th2);
            const double fY = upwind_flux<TH1>(w[4], w[5], w[0], w[6], dirs[1], sg & 2, wq, th2);
            const double fZ = upwind_flux<TH1>(w[7], w[8], w[0], w[9], dirs[2], sg & 4, wq, th2);
            double s;
            if constexpr (P2)
                s = fX * rx + fY * ry + fZ * rz;
            else
                s = div_by(fX, hx, rx) + div_by(fY, hy, ry) + div_by(fZ, hz, rz);
            __builtin_amdgcn_sched_barrier(0);
            sNow[d] = sNext;
            // unconditional (at the end again the last plane), so that the waits for the values
            // in flight can be counted
            load(v[d], plane, sNow[d]);
            plane += q + D + 1 < S.nq ? ng : 0;
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                use_s(m[p & 1]);
                if (p + 1 < NP) {
                    piece(p + 1);
                } else {
                    row += OR;  // past the last row: padding
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        dirs[e] = row[e];
                    sNext = sgn[q + 1 + D];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < PS && p * PS + i < NM; ++i)
                    fl[p * PS + i] += m[p & 1][i] * s;
                if (p + 1 < NP)
                    __builtin_amdgcn_sched_barrier(0);
            }
        };
        int q0 = 0;
#pragma unroll 1
        for (; q0 + D <= S.nq; q0 += D) {
#pragma unroll
            for (int d = 0; d < D; ++d)
                ordinate(d, q0 + d);
        }
        if constexpr (D > 2) {  // nq is even
#pragma unroll 1
            for (int d = 0; q0 + d < S.nq; ++d) {
                ordinate(0, q0 + d);
#pragma unroll
                for (int e = 0; e < 10; ++e)
                    v[0][e] = v[1][e];
                sNow[0] = sNow[1];
            }
        }
    } else {
        // the 13 values of the cell's stencil: the centre, then -2, -1, +1, +2 along x, y and z;
        // up to nm = 16 the next ordinate's are in flight while this one's are used (at nm = 25
        // there are no registers for them beside the fast path's waves)
        constexpr bool kAhead = NM <= 16;
        const ptrdiff_t off[13] = {0,       -2 * sx, -sx, sx, 2 * sx, -2 * sy, -sy,
                                   sy,      2 * sy,  -2,  -1, 1,      2};
        const double *a = A + (size_t)T.i * sx + in, *row = ord;
        double v[13], nv[13];
#pragma unroll
        for (int e = 0; e < 13; ++e)
            v[e] = a[off[e]];
        for (int q = 0; q < S.nq; ++q) {
            a += q + 1 < S.nq ? ng : 0;
            if constexpr (kAhead) {
#pragma unroll
                for (int e = 0; e < 13; ++e)
                    nv[e] = a[off[e]];
            }
            const double wq = row[3];
            const double fX = axis_flux<TH1>(v[1], v[2], v[0], v[3], v[4], row[0], wq, S.theta);
            const double fY = axis_flux<TH1>(v[5], v[6], v[0], v[7], v[8], row[1], wq, S.theta);
            const double fZ =
                axis_flux<TH1>(v[9], v[10], v[0], v[11], v[12], row[2], wq, S.theta);
            double s;
            if constexpr (P2)
                s = fX * S.rdx + fY * S.rdy + fZ * S.rdz;
            else
                s = fX / S.dx + fY / S.dy + fZ / S.dz;
#pragma unroll
            for (int m = 0; m < NM; ++m)
                fl[m] += row[4 + m] * s;
#pragma unroll
            for (int e = 0; e < 13; ++e)
                v[e] = kAhead ? nv[e] : a[off[e]];
            row += OR;
        }
    }
    if (!have)
        return;
    const size_t c = (size_t)T.i * sx + in;
    if (S.fuseEuler) {
        // update.cpp:28-35
        const double dt = S.dt, st = sigT[c], ss = sigS[c];
        double *uc = u + c * NM;
        uc[0] = uc[0] * (1.0 + dt * ss - dt * st) - dt * fl[0];
#pragma unroll
        for (int m = 1; m < NM; ++m) {
            uc[m] = uc[m] * (1.0 - dt * st) - dt * fl[m];
            if (m % 12 == 0)  // not all of u in registers beside the flux
                __builtin_amdgcn_sched_barrier(0);
        }
    } else {
#pragma unroll
        for (int m = 0; m < NM; ++m)
            flux[c * NM + m] = fl[m];
    }
}

__global__ void k_zero_ghost_flux(Grid G, int nm, double *flux)
{
    const int64_t ng = (int64_t)G.NX * G.NY * G.NZ;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < ng * nm;
         t += (int64_t)gridDim.x * blockDim.x) {
        int64_t c = t / nm;
        int k = (int)(c % G.NZ), j = (int)((c / G.NZ) % G.NY), i = (int)(c / ((int64_t)G.NZ * G.NY));
        bool interior = i >= 2 && i < G.nx + 2 && j >= 2 && j < G.ny + 2 && k >= 2 && k < G.nz + 2;
        if (!interior)
            flux[t] = 0.0;
    }
}

// -------------------------------------------------------------- moment flux
enum : int { kMomFlux = 0, kMomStage1 = 1, kMomStage2 = 2 };

__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ long long uniform_i64(long long v)
{
    const unsigned lo = __builtin_amdgcn_readfirstlane((int)(v & 0xffffffffll));
    const int hi = __builtin_amdgcn_readfirstlane((int)(v >> 32));
    return ((long long)hi << 32) | lo;
}

// operators are read kOpRun doubles at a time (the table is padded by as many)
constexpr int kOpRun = 16;
typedef double op8 __attribute__((ext_vector_type(8), aligned(8)));
typedef double op4 __attribute__((ext_vector_type(4), aligned(8)));
struct OpRun {
    op8 lo, hi;
};

// The flux alone up to nm = 9, one thread per interior cell on its own moments, the operators'
// columns broadcast from LDS.  k_moment_stage's runs, LDS turns and scalar operands are a longer
// chain of waits, which pays where they save the passes of a whole step and from nm = 16 on, but
// not here.  Measured, k_moment_stage -> this: P_1 64^3 12.4 -> 10.7 us, 128^3 65 -> 51; P_2 20^3
// 15.8 -> 11.2, 64^3 34 -> 31, 80^3 65 -> 51, 128^3 271 -> 211.
template <int NM>
__global__ __launch_bounds__(kTB) void k_flux_moment(Grid G, const double *__restrict__ u,
                                                      double *flux,
                                                      const double *__restrict__ opsT, double dx,
                                                      double dy, double dz)
{
    __shared__ double sO[6 * NM * NM];
    for (int e = threadIdx.x; e < 6 * NM * NM; e += blockDim.x)
        sO[e] = opsT[e];
    __syncthreads();
    Tile T;
    if (!tile_of(G, blockIdx.x, gridDim.x, blockDim.x, T))
        return;
    const TileCell tc = tile_cell(G, T, threadIdx.x);
    if (!tc.have)
        return;
    const size_t c = G.idx(T.i + tc.di, tc.j, tc.k);
    const size_t strides[3] = {(size_t)G.NY * G.NZ, (size_t)G.NZ, 1};
    const double hs[3] = {dx, dy, dz};
    double out[NM];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        const size_t s = strides[ax];
        const double *um2 = u + (c - 2 * s) * NM, *um1 = u + (c - s) * NM, *u0 = u + c * NM,
                     *up1 = u + (c + s) * NM, *up2 = u + (c + 2 * s) * NM;
        const double *Op = sO + (2 * ax) * NM * NM, *Om = Op + NM * NM;
        double temp[NM], F[NM];
#pragma unroll
        for (int m = 0; m < NM; ++m)
            temp[m] = 0.25 * up1[m] + 0.75 * u0[m] - 1.25 * um1[m] + 0.25 * um2[m];
#pragma unroll
        for (int r = 0; r < NM; ++r)
            F[r] = 0.0;
#pragma unroll
        for (int q = 0; q < NM; ++q)
#pragma unroll
            for (int r = 0; r < NM; ++r)
                F[r] += Op[q * NM + r] * temp[q];
#pragma unroll
        for (int m = 0; m < NM; ++m)
            temp[m] = -0.25 * up2[m] + 1.25 * up1[m] - 0.75 * u0[m] - 0.25 * um1[m];
#pragma unroll
        for (int q = 0; q < NM; ++q)
#pragma unroll
            for (int r = 0; r < NM; ++r)
                F[r] += Om[q * NM + r] * temp[q];
        // flux = xF/dx + yF/dy + zF/dz, accumulated left to right
#pragma unroll
        for (int m = 0; m < NM; ++m)
            out[m] = ax == 0 ? F[m] / hs[0] : out[m] + F[m] / hs[ax];
    }
#pragma unroll
    for (int m = 0; m < NM; ++m)
        flux[c * NM + m] = out[m];
}

template <int NM, int KIND>
constexpr int moment_lds()
{
    return kWave * ((NM | 1) + (KIND == kMomFlux ? 0 : 2));
}

// One thread per interior cell.  Bound by the vector unit (six NM x NM products without FMA
// contraction) and, close behind, by HBM.  A lane that reads its own cell's moments touches a
// cache line of its own per load (36 lines a load at nm = 9), so each
// wave reads the 64 cells of a stencil offset as one contiguous run, forms the differences on
// the runs (they are elementwise) and turns only those to a cell per lane through its own LDS
// rows.  opsT holds the operators' columns: uniform over the wave, they come as scalar
// operands (broadcast reads from LDS would take twice the vector unit's time), a run of them
// at a time, the next run's loads in flight while one is used.
//   kMomFlux    dst = flux
//   kMomStage1  dst = Euler(src, flux(src))
//   kMomStage2  dst = (Euler(src, flux(src)) + dst) / 2
// so that a two-stage step (u -> b, b -> u) neither copies u nor stores a flux.  Measured at
// 128^3, nm = 9: a step 447 us, against 1272 with flux, Euler, copy and average apart.
// P2: every spacing a power of two (division is multiplication by the exact reciprocal).
template <int NM, int KIND, bool P2>
__global__ __launch_bounds__(kTB) __attribute__((amdgpu_waves_per_eu(NM <= 9 ? 3 : 1))) void k_moment_stage(Grid G, const double *__restrict__ src,
                                                       double *dst,
                                                       const double *__restrict__ opsT, double dx,
                                                       double dy, double dz, double dt,
                                                       const double *__restrict__ sigT,
                                                       const double *__restrict__ sigS)
{
    constexpr int NMS = NM | 1;  // odd row stride: no bank conflicts reading a row per lane
    extern __shared__ double sMem[];  // moment_lds<NM, KIND>() doubles a wave
    const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
    double *const buf = sMem + wv * moment_lds<NM, KIND>();
    double *const sD = buf + kWave * NMS;  // the Euler factors
    Tile T;
    if (!tile_of(G, blockIdx.x, gridDim.x, blockDim.x, T))
        return;
    // lanes past the run's end work on its last cell and write nothing; waves past it leave
    const TileCell tc = tile_cell(G, T, threadIdx.x);
    const bool have = tc.have;
    if (__ballot(have) == 0)
        return;
    const size_t c = G.idx(T.i + tc.di, tc.j, tc.k);
    const size_t c0 = (size_t)uniform_i64((long long)c);
    // element lane + 64 k of the wave's run: its place in memory, in bytes from the first cell's
    // moments (64 interior cells lie within a few rows or, where the rows are short, planes)
    unsigned rel[NM];
    const int crel = (int)(c - c0);
#pragma unroll
    for (int k = 0; k < NM; ++k) {
        const int e = lane + kWave * k, l = e / NM;
        rel[k] = 8u * (unsigned)(__shfl(crel, l) * NM + (e - l * NM));
    }
    auto el = [](const double *a, unsigned o) { return *(const double *)((const char *)a + o); };
    auto place = [&](int k) {  // the same element in LDS
        const int e = lane + kWave * k, l = e / NM;
        return NM == NMS ? e : l * NMS + (e - l * NM);
    };
    auto run = [&](ptrdiff_t off) { return src + ((ptrdiff_t)c0 + off) * NM; };
    double out[NM];
#pragma unroll(NM <= 4 ? 3 : 1)
    for (int ax = 0; ax < 3; ++ax) {
        const ptrdiff_t s = ax == 0 ? (ptrdiff_t)G.NY * G.NZ : (ax == 1 ? (ptrdiff_t)G.NZ : 1);
        const double h = ax == 0 ? dx : (ax == 1 ? dy : dz);
        const double *O = opsT + (2 * ax) * NM * NM;
        const double *a0 = run(0), *ap1 = run(s), *ap2 = run(2 * s), *am1 = run(-s),
                     *am2 = run(-2 * s);
        double tm[NM], F[NM];
        auto put_tm = [&] {
            wave_lds_sync();
#pragma unroll
            for (int k = 0; k < NM; ++k)
                buf[place(k)] = tm[k];
            wave_lds_sync();
        };
        wave_lds_sync();
#pragma unroll
        for (int k = 0; k < NM; ++k) {
            const double up1 = el(ap1, rel[k]), u0 = el(a0, rel[k]), um1 = el(am1, rel[k]);
            buf[place(k)] = 0.25 * up1 + 0.75 * u0 - 1.25 * um1 + 0.25 * el(am2, rel[k]);
            tm[k] = -0.25 * el(ap2, rel[k]) + 1.25 * up1 - 0.75 * u0 - 0.25 * um1;
        }
        wave_lds_sync();
#pragma unroll
        for (int i = 0; i < NM; ++i)
            F[i] = 0.0;
        if constexpr (NM <= 16) {
            double t[NM];
#pragma unroll
            for (int q = 0; q < NM; ++q)
                t[q] = buf[lane * NMS + q];
            put_tm();
#pragma unroll
            for (int q = 0; q < NM; ++q)
                tm[q] = buf[lane * NMS + q];
            // element e of the stream of both operators' columns: row e % NM, column e / NM
            constexpr int nOp = 2 * NM * NM, nRun = (nOp + kOpRun - 1) / kOpRun;
            OpRun cur = *(const OpRun *)O, nxt = cur;
#pragma unroll
            for (int r = 0; r < nRun; ++r) {
                // scalar loads return in any order, so a wait is for all of them: wait for
                // this run here, before the next one's loads are issued
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("" ::"s"(cur.lo), "s"(cur.hi));
                if (r + 1 < nRun)
                    nxt = *(const OpRun *)(O + (r + 1) * kOpRun);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < kOpRun; ++j) {
                    const int e = r * kOpRun + j, q = e / NM, i = e % NM;
                    if (e < nOp)
                        F[i] += (j < 8 ? cur.lo[j & 7] : cur.hi[j & 7]) *
                                (q < NM ? t[q % NM] : tm[q % NM]);
                }
                cur = nxt;
            }
        } else {  // two runs to a column, columns in a loop
            static_assert(NM <= 16 || NM == 25, "runs of 13 and 12");
            auto apply = [&](const double *Oc) {
                op8 a8 = *(const op8 *)Oc;
                op4 a4 = *(const op4 *)(Oc + 8);
                double a1 = Oc[12], tn = buf[lane * NMS];
#pragma unroll 1
                for (int q = 0; q < NM; ++q) {
                    const double t = tn;
                    __builtin_amdgcn_sched_barrier(0);
                    asm volatile("" ::"s"(a8), "s"(a4), "s"(a1), "v"(t));
                    const op8 b8 = *(const op8 *)(Oc + 13);
                    const op4 b4 = *(const op4 *)(Oc + 21);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = 0; i < 13; ++i)
                        F[i % NM] += (i < 8 ? a8[i & 7] : (i < 12 ? a4[i & 3] : a1)) * t;
                    __builtin_amdgcn_sched_barrier(0);
                    asm volatile("" ::"s"(b8), "s"(b4));
                    Oc += NM;  // past the last column: the next operator's, or the padding
                    a8 = *(const op8 *)Oc;
                    a4 = *(const op4 *)(Oc + 8);
                    a1 = Oc[12];
                    tn = buf[lane * NMS + (q + 1 < NM ? q + 1 : q)];
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = 13; i < 25; ++i)
                        F[i % NM] += (i < 21 ? b8[(i - 13) & 7] : b4[(i - 21) & 3]) * t;
                }
            };
            apply(O);
            put_tm();
            apply(O + NM * NM);
        }
        // flux = xF/dx + yF/dy + zF/dz, accumulated left to right
        const double rh = 1.0 / h;
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const double t = P2 ? F[m] * rh : F[m] / h;
            out[m] = ax == 0 ? t : out[m] + t;
        }
    }
    wave_lds_sync();
    if constexpr (KIND != kMomFlux) {  // the Euler factors of the lane's cell, update.cpp:28-35
        const double st = sigT[c], ss = sigS[c];
        sD[2 * lane] = 1.0 + dt * ss - dt * st;
        sD[2 * lane + 1] = 1.0 - dt * st;
    }
#pragma unroll
    for (int m = 0; m < NM; ++m)
        buf[lane * NMS + m] = out[m];
    wave_lds_sync();
    // the lanes that have a cell are the first of the wave, and so are their elements
    const int nHave = __popcll(__ballot(have)) * NM;
    double *const at = dst + c0 * NM;
#pragma unroll
    for (int k = 0; k < NM; ++k) {
        const int e = lane + kWave * k, l = e / NM;
        double v = buf[place(k)];
        if constexpr (KIND != kMomFlux)
            v = el(run(0), rel[k]) * sD[2 * l + (e - l * NM ? 1 : 0)] - dt * v;
        if constexpr (KIND == kMomStage2)
            v = 0.5 * (v + el(at, rel[k]));
        if (e < nHave)
            *(double *)((char *)at + rel[k]) = v;
    }
}

// -------------------------------------------------------------------- euler
__global__ void k_euler(Grid G, int nm, double *u, const double *__restrict__ flux,
                        const double *__restrict__ sigT, const double *__restrict__ sigS,
                        double dt)
{
    const int64_t ni = (int64_t)G.nx * G.ny * G.nz;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ni)
        return;
    const int k = 2 + (int)(t % G.nz);
    const int j = 2 + (int)((t / G.nz) % G.ny);
    const int i = 2 + (int)(t / ((int64_t)G.nz * G.ny));
    const size_t c = G.idx(i, j, k);
    const double st = sigT[c], ss = sigS[c];
    double *uc = u + c * nm;
    const double *fc = flux + c * nm;
    uc[0] = uc[0] * (1.0 + dt * ss - dt * st) - dt * fc[0];
    for (int m = 1; m < nm; ++m)
        uc[m] = uc[m] * (1.0 - dt * st) - dt * fc[m];
}

// ---------------------------------------------------------------------- rk2
__global__ void k_rk2(Grid G, int nm, double *u, double *uOld, int kind)
{
    const int64_t n = (int64_t)G.nx * G.ny * G.nz * nm;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int m = (int)(t % nm);
        const int64_t cc = t / nm;
        const int k = 2 + (int)(cc % G.nz);
        const int j = 2 + (int)((cc / G.nz) % G.ny);
        const int i = 2 + (int)(cc / ((int64_t)G.nz * G.ny));
        const size_t e = G.idx(i, j, k) * nm + m;
        if (kind == 0)
            uOld[e] = u[e];
        else
            u[e] = 0.5 * (u[e] + uOld[e]);
    }
}

// ------------------------------------------------------------ synthetic batch
__device__ __forceinline__ uint64_t splitmix64(uint64_t x)
{
    uint64_t z = x + 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
__device__ __forceinline__ double uniform01(uint64_t seed, uint64_t idx, uint64_t stream)
{
    uint64_t key = splitmix64(seed ^ (stream * 0xD1B54A32D192ED03ull));
    uint64_t z = splitmix64(key + idx);
    return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}
__device__ __forceinline__ double normal01(uint64_t seed, uint64_t idx, uint64_t stream)
{
    double u1 = uniform01(seed, idx, 2 * stream), u2 = uniform01(seed, idx, 2 * stream + 1);
    return sqrt(-2.0 * log(1.0 - u1)) * cos(2.0 * M_PI * u2);
}

// Initial state over all cells including ghosts (init.cpp:480-506), cell centres at
// a + (i - 2 + 1/2) d with ghosts at their own unwrapped centres (init.cpp:483-485):
//   ic 0: the reference Gaussian, u0 = max(floor, 2 sqrt(pi) G_sigma(x)) with the normalised
//         G (init.cpp:27-34, 493-495);
//   ic 1: pulse rho = max(exp(-|x|^2/(2 sigma^2)), floor) (1 + noise U[-1,1]), u0 = 2 sqrt(pi)
//         rho (counter RNG stream 7 on the cell index);
//   ic 2: the smooth state of init.cpp:497-502.
// sigma_t = sigma_s = crossSection; alpha (if not null) from init.cpp:262-268.
__global__ __launch_bounds__(kTB) void k_init_grid(int nx, int ny, int nz, int nm, double ax,
                                                   double ay, double az, double dx, double dy,
                                                   double dz, int ic, double sigma, double floorv,
                                                   double noise, uint64_t seed, double cross,
                                                   double *u, double *alpha, double *sigmaT,
                                                   double *sigmaS)
{
    const int64_t NX = nx + 4, NY = ny + 4, NZ = nz + 4;
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= NX * NY * NZ)
        return;
    const int k = (int)(c % NZ), j = (int)((c / NZ) % NY), i = (int)(c / (NZ * NY));
    const double x = ax + (i - 2) * dx + dx / 2.0;
    const double y = ay + (j - 2) * dy + dy / 2.0;
    const double z = az + (k - 2) * dz + dz / 2.0;
    sigmaT[c] = cross;
    sigmaS[c] = cross;
    double u0, u123 = 0.0;
    if (ic == 0) {
        const double f1 = 1.0 / (sigma * sqrt(2.0 * M_PI));
        const double g = f1 * f1 * f1 * exp(-(x * x + y * y + z * z) / (2.0 * sigma * sigma));
        u0 = fmax(floorv, g * 2.0 * sqrt(M_PI));
    } else if (ic == 1) {
        double rho = fmax(exp(-(x * x + y * y + z * z) / (2.0 * sigma * sigma)), floorv);
        if (noise != 0.0)
            rho = rho * (1.0 + noise * (2.0 * uniform01(seed, (uint64_t)c, 7) - 1.0));
        u0 = 2.0 * sqrt(M_PI) * rho;
    } else {
        u0 = (2.0 + cos(2 * M_PI * x) * cos(2 * M_PI * y) * cos(2 * M_PI * z)) * 2.0 * sqrt(M_PI);
        u123 = 0.3 * u0;
    }
    u[c * nm] = u0;
    for (int m = 1; m < nm; ++m)
        u[c * nm + m] = (m <= 3) ? u123 : 0.0;
    if (alpha) {
        alpha[c * nm] = sqrt(4.0 * M_PI) * log(u0 / sqrt(4.0 * M_PI));
        for (int m = 1; m < nm; ++m)
            alpha[c * nm + m] = 0.0;
    }
}

template <int NM>
__global__ __launch_bounds__(kTB) void k_make_batch(int64_t n, int nq, const double *__restrict__ M,
                                                     const double *__restrict__ w, uint64_t seed,
                                                     double smin, double smax, double *u,
                                                     double *alpha0, double *alphaStar)
{
    __shared__ double sM[kChunk * NM];
    __shared__ double sWt[kChunk];
    const int64_t c = (int64_t)blockIdx.x * kTB + threadIdx.x;
    const bool have = c < n;
    double as[NM], uc[NM];
    const double s = smin + (smax - smin) * uniform01(seed, (uint64_t)c, 1);
#pragma unroll
    for (int k = 0; k < NM; ++k) {
        as[k] = s * normal01(seed, (uint64_t)c * 64 + k, 2);
        uc[k] = 0.0;
    }
    for (int q0 = 0; q0 < nq; q0 += kChunk) {
        const int nqc = min(kChunk, nq - q0);
        __syncthreads();
        for (int e = threadIdx.x; e < nqc * NM; e += kTB)
            sM[e] = M[(size_t)q0 * NM + e];
        if (threadIdx.x < nqc)
            sWt[threadIdx.x] = w[q0 + threadIdx.x];
        __syncthreads();
        if (have) {
            for (int ql = 0; ql < nqc; ++ql) {
                double e = 0.0;
#pragma unroll
                for (int k = 0; k < NM; ++k)
                    e = e + as[k] * sM[ql * NM + k];
                e = sWt[ql] * exp(e);
#pragma unroll
                for (int k = 0; k < NM; ++k)
                    uc[k] += e * sM[ql * NM + k];
            }
        }
    }
    if (!have)
        return;
#pragma unroll
    for (int k = 0; k < NM; ++k) {
        u[c * NM + k] = uc[k];
        alpha0[c * NM + k] = (k == 0) ? sqrt(4.0 * M_PI) * log(uc[0] / sqrt(4.0 * M_PI)) : 0.0;
        if (alphaStar)
            alphaStar[c * NM + k] = as[k];
    }
}

unsigned blocks_for(int64_t n, int tb = kTB, int64_t cap = 1 << 20)
{
    int64_t b = (n + tb - 1) / tb;
    if (b > cap)
        b = cap;
    if (b < 1)
        b = 1;
    return (unsigned)b;
}

}  // namespace

hipError_t launch_ghost_fill(int nx, int ny, int nz, int nm, double *u, hipStream_t s, double *u2)
{
    Grid G = make_grid(nx, ny, nz);
    int64_t total = ((int64_t)2 * ny * nz + (int64_t)2 * nx * nz + (int64_t)2 * nx * ny) * 2 * nm;
    hipLaunchKernelGGL(k_ghost_fill, dim3(blocks_for(total, 256, 65536)), dim3(256), 0, s, G,
                       nm, u, u2);
    return hipGetLastError();
}

hipError_t launch_ansatz(c3d_ctx_s *ctx, int nx, int ny, int nz, const double *alpha, double *A,
                         int isPn, double dx, double dy, double dz, hipStream_t s)
{
    const double tiny = exact_reciprocals(dx, dy, dz) ? kTinyP2 : kTinyDiv;
    // kind: 1 linear (P_N), 2 deterministic exp (reference-order mode), 0 device exp
    if (!isPn && ctx->precision == C3D_PREC_FP64_REFORDER)
        isPn = 2;
    // k_ansatz's range: magnitudes, or an exponent's middle and half width (a little less: the
    // exponentials round)
    const double lo = log(tiny), hi = log(kTame);
    const double ra = isPn == 1 ? tiny : 0.5 * (lo + hi);
    const double rb = isPn == 1 ? kTame : 0.5 * (hi - lo) - 1e-6;
    const Grid G = make_grid(nx, ny, nz);
    const int64_t ng = (int64_t)G.NX * G.NY * G.NZ;
    const int nq = ctx->t.nq;
    // small grids share out the ordinates too: 8 blocks a CU, at least 16 ordinates each
    const int64_t bx = blocks_for(ng, kTB, INT32_MAX);
    const int64_t want = std::max<int64_t>(1, (int64_t)ctx->numCU * 8 / bx);
    const int split = (int)std::min<int64_t>(want, (nq + 15) / 16);
    const int nqPer = (nq + split - 1) / split;
    dim3 grid((unsigned)bx, (unsigned)split);
    hipLaunchKernelGGL(k_clear_int, dim3(1), dim3(1), 0, s, ctx->d_wild);
#define C3D_ANSATZ(NMV)                                                                        \
    hipLaunchKernelGGL(k_ansatz<NMV>, grid, dim3(kTB), 0, s, G, ng, nq, nqPer, ctx->d_ord, \
                       alpha, A, isPn, ra, rb, ctx->d_wild)
    switch (ctx->t.nm) {
    case 4: C3D_ANSATZ(4); break;
    case 9: C3D_ANSATZ(9); break;
    case 16: C3D_ANSATZ(16); break;
    case 25: C3D_ANSATZ(25); break;
    default: return hipErrorInvalidValue;
    }
#undef C3D_ANSATZ
    return hipGetLastError();
}

hipError_t launch_stencil(c3d_ctx_s *ctx, int nx, int ny, int nz, const double *A, double *flux,
                          double *u, const double *sigmaT, const double *sigmaS, double dt,
                          double dx, double dy, double dz, double theta, int fuseEuler,
                          int zeroGhosts, hipStream_t s)
{
    auto tame = [](double x) { return fabs(x) > 1e-15 && fabs(x) < 1e15; };
    StencilArgs S{make_grid(nx, ny, nz), ctx->t.nq, dx, dy, dz, theta, dt, fuseEuler,
                  1.0 / dx, 1.0 / dy, 1.0 / dz, 0};
    // a block's offsets within its planes are 32 bits of bytes on the fast path
    S.general = !(tame(dx) && tame(dy) && tame(dz) && (theta == 0.0 || tame(theta)) &&
                  ctx->tameOrdinates && (int64_t)S.G.NY * S.G.NZ < (1 << 29));
    const bool p2 = exact_reciprocals(dx, dy, dz);
    const bool th1 = theta == 1.0;
    const int tb = tile_threads(S.G, ctx->numCU);
    dim3 grid(tile_blocks(S.G, tb));
    // four ordinates in flight where there is at most a wave per SIMD
    const bool deep = tb < kTB;
    if (zeroGhosts && !fuseEuler) {
        const int64_t ng = (int64_t)S.G.NX * S.G.NY * S.G.NZ;
        hipLaunchKernelGGL(k_zero_ghost_flux, dim3(blocks_for(ng * ctx->t.nm, 256, 65536)),
                           dim3(256), 0, s, S.G, ctx->t.nm, flux);
    }
#define C3D_STENCIL_V(NMV, P, T, D)                                                           \
    hipLaunchKernelGGL((k_stencil<NMV, P, T, D>), grid, dim3(tb), 0, s, S, A, ctx->d_ord,     \
                       ctx->d_sgn, ctx->d_wild, flux, u, sigmaT, sigmaS)
#define C3D_STENCIL_D(NMV, D)                                                                 \
    if (p2 && th1)                                                                             \
        C3D_STENCIL_V(NMV, true, true, D);                                                     \
    else if (p2)                                                                               \
        C3D_STENCIL_V(NMV, true, false, D);                                                    \
    else if (th1)                                                                              \
        C3D_STENCIL_V(NMV, false, true, D);                                                    \
    else                                                                                       \
        C3D_STENCIL_V(NMV, false, false, D)
#define C3D_STENCIL(NMV)                                                                      \
    if (deep) {                                                                                \
        C3D_STENCIL_D(NMV, 4);                                                                 \
    } else {                                                                                   \
        C3D_STENCIL_D(NMV, 2);                                                                 \
    }
    switch (ctx->t.nm) {
    case 4: C3D_STENCIL(4); break;
    case 9: C3D_STENCIL(9); break;
    case 16: C3D_STENCIL(16); break;
    case 25: C3D_STENCIL(25); break;
    default: return hipErrorInvalidValue;
    }
#undef C3D_STENCIL
#undef C3D_STENCIL_D
#undef C3D_STENCIL_V
    return hipGetLastError();
}

namespace {
template <int KIND>
hipError_t launch_moment_stage(c3d_ctx_s *ctx, int nx, int ny, int nz, const double *src,
                               double *dst, const double *sigmaT, const double *sigmaS, double dt,
                               double dx, double dy, double dz, hipStream_t s)
{
    Grid G = make_grid(nx, ny, nz);
    const bool p2 = exact_reciprocals(dx, dy, dz);
    const int tb = tile_threads(G, ctx->numCU);
    dim3 grid(tile_blocks(G, tb));
#define C3D_MOMENT_V(NMV, P)                                                                   \
    hipLaunchKernelGGL((k_moment_stage<NMV, KIND, P>), grid, dim3(tb),                         \
                       (tb / kWave * moment_lds<NMV, KIND>() * sizeof(double)), s, G, src, dst,\
                       ctx->d_pnOps, dx, dy, dz, dt, sigmaT, sigmaS)
#define C3D_MOMENT(NMV)                                                                        \
    if (p2)                                                                                    \
        C3D_MOMENT_V(NMV, true);                                                               \
    else                                                                                       \
        C3D_MOMENT_V(NMV, false)
    if constexpr (KIND != kMomFlux) {  // k_flux_moment's
        switch (ctx->t.nm) {
        case 4: C3D_MOMENT(4); return hipGetLastError();
        case 9: C3D_MOMENT(9); return hipGetLastError();
        }
    }
    switch (ctx->t.nm) {
    case 16: C3D_MOMENT(16); break;
    case 25: C3D_MOMENT(25); break;
    default: return hipErrorInvalidValue;
    }
#undef C3D_MOMENT
#undef C3D_MOMENT_V
    return hipGetLastError();
}
}  // namespace

hipError_t launch_flux_moment(c3d_ctx_s *ctx, int nx, int ny, int nz, const double *u,
                              double *flux, double dx, double dy, double dz, hipStream_t s)
{
    if (ctx->t.nm > 9)
        return launch_moment_stage<kMomFlux>(ctx, nx, ny, nz, u, flux, nullptr, nullptr, 0.0, dx,
                                             dy, dz, s);
    Grid G = make_grid(nx, ny, nz);
    dim3 grid(tile_blocks(G, kTB));
    if (ctx->t.nm == 4)
        hipLaunchKernelGGL(k_flux_moment<4>, grid, dim3(kTB), 0, s, G, u, flux, ctx->d_pnOps, dx,
                           dy, dz);
    else
        hipLaunchKernelGGL(k_flux_moment<9>, grid, dim3(kTB), 0, s, G, u, flux, ctx->d_pnOps, dx,
                           dy, dz);
    return hipGetLastError();
}

// one SSP-RK2 step of the P_N equations with the moment flux; b: a grid's worth of scratch
hipError_t launch_moment_rk2(c3d_ctx_s *ctx, int nx, int ny, int nz, double *u, double *b,
                             const double *sigmaT, const double *sigmaS, double dt, double dx,
                             double dy, double dz, hipStream_t s)
{
    hipError_t e = launch_ghost_fill(nx, ny, nz, ctx->t.nm, u, s);
    if (e == hipSuccess)
        e = launch_moment_stage<kMomStage1>(ctx, nx, ny, nz, u, b, sigmaT, sigmaS, dt, dx, dy, dz,
                                            s);
    if (e == hipSuccess)  // the step leaves u with the second stage's ghosts
        e = launch_ghost_fill(nx, ny, nz, ctx->t.nm, b, s, u);
    if (e == hipSuccess)
        e = launch_moment_stage<kMomStage2>(ctx, nx, ny, nz, b, u, sigmaT, sigmaS, dt, dx, dy, dz,
                                            s);
    return e;
}

hipError_t launch_euler(int nx, int ny, int nz, int nm, double *u, const double *flux,
                        const double *sigmaT, const double *sigmaS, double dt, hipStream_t s)
{
    Grid G = make_grid(nx, ny, nz);
    const int64_t ni = (int64_t)nx * ny * nz;
    hipLaunchKernelGGL(k_euler, dim3(blocks_for(ni, 256, INT32_MAX)), dim3(256), 0, s, G, nm, u,
                       flux, sigmaT, sigmaS, dt);
    return hipGetLastError();
}

hipError_t launch_rk2(int nx, int ny, int nz, int nm, double *u, double *uOld, int kind,
                      hipStream_t s)
{
    Grid G = make_grid(nx, ny, nz);
    const int64_t n = (int64_t)nx * ny * nz * nm;
    hipLaunchKernelGGL(k_rk2, dim3(blocks_for(n, 256, 1 << 20)), dim3(256), 0, s, G, nm, u, uOld,
                       kind);
    return hipGetLastError();
}

hipError_t launch_init_grid(int nx, int ny, int nz, int nm, const double *a, const double *d,
                            int ic, double sigma, double floorv, double noise, uint64_t seed,
                            double cross, double *u, double *alpha, double *sigmaT,
                            double *sigmaS, hipStream_t s)
{
    const int64_t ng = (int64_t)(nx + 4) * (ny + 4) * (nz + 4);
    hipLaunchKernelGGL(k_init_grid, dim3((unsigned)((ng + kTB - 1) / kTB)), dim3(kTB), 0, s, nx,
                       ny, nz, nm, a[0], a[1], a[2], d[0], d[1], d[2], ic, sigma, floorv, noise,
                       seed, cross, u, alpha, sigmaT, sigmaS);
    return hipGetLastError();
}

hipError_t launch_make_batch(c3d_ctx_s *ctx, int64_t n, uint64_t seed, double smin, double smax,
                             double *u, double *alpha0, double *alphaStar, hipStream_t s)
{
    dim3 grid(blocks_for(n, kTB, INT32_MAX));
    const int nq = ctx->t.nq;
    switch (ctx->t.nm) {
    case 4: hipLaunchKernelGGL(k_make_batch<4>, grid, dim3(kTB), 0, s, n, nq, ctx->d_M, ctx->d_w, seed, smin, smax, u, alpha0, alphaStar); break;
    case 9: hipLaunchKernelGGL(k_make_batch<9>, grid, dim3(kTB), 0, s, n, nq, ctx->d_M, ctx->d_w, seed, smin, smax, u, alpha0, alphaStar); break;
    case 16: hipLaunchKernelGGL(k_make_batch<16>, grid, dim3(kTB), 0, s, n, nq, ctx->d_M, ctx->d_w, seed, smin, smax, u, alpha0, alphaStar); break;
    case 25: hipLaunchKernelGGL(k_make_batch<25>, grid, dim3(kTB), 0, s, n, nq, ctx->d_M, ctx->d_w, seed, smin, smax, u, alpha0, alphaStar); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ------------------------------------------------------------ statistics summary
// Per-block partial sums of the closure's per-cell outcomes, the quantities update.cpp:145-174
// folds: sums and maxima of totalIter and iterGamma, and the count of cells on each ladder
// rung (r within 1e-10 of the rung's value, opt.h:37-38).  Row b of `part` holds block b's
// [n, sumIter, sumGamma, maxIter, maxGamma, rung0..rung4]; the host adds the rows.  No
// atomics: a grid-stride loop, then a tree in LDS.
constexpr int kSumFields = 10;
__global__ __launch_bounds__(kTB) void k_stats_partials(int64_t n,
                                                        const c3d_cell_stats *__restrict__ st,
                                                        long long *part)
{
    __shared__ long long sh[kSumFields][kTB];
    long long v[kSumFields] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const double reg[5] = {0.0, 1e-3, 1e-2, 1e-1, 5e-1};
    for (int64_t c = (int64_t)blockIdx.x * kTB + threadIdx.x; c < n;
         c += (int64_t)gridDim.x * kTB) {
        const c3d_cell_stats s = st[c];
        v[0] += 1;
        v[1] += s.totalIter;
        v[2] += s.iterGamma;
        v[3] = v[3] > s.totalIter ? v[3] : s.totalIter;
        v[4] = v[4] > s.iterGamma ? v[4] : s.iterGamma;
#pragma unroll
        for (int r = 0; r < 5; ++r)
            v[5 + r] += fabs(s.r - reg[r]) < 1e-10 ? 1 : 0;
    }
#pragma unroll
    for (int f = 0; f < kSumFields; ++f)
        sh[f][threadIdx.x] = v[f];
    __syncthreads();
    for (int w = kTB / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
#pragma unroll
            for (int f = 0; f < kSumFields; ++f) {
                const long long a = sh[f][threadIdx.x], b = sh[f][threadIdx.x + w];
                sh[f][threadIdx.x] = (f == 3 || f == 4) ? (a > b ? a : b) : a + b;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < kSumFields)
        part[(size_t)blockIdx.x * kSumFields + threadIdx.x] = sh[threadIdx.x][0];
}

hipError_t launch_stats_partials(int64_t n, const c3d_cell_stats *st, long long *part,
                                 int blocks, hipStream_t s)
{
    hipLaunchKernelGGL(k_stats_partials, dim3(blocks), dim3(kTB), 0, s, n, st, part);
    return hipGetLastError();
}

}  // namespace c3d
