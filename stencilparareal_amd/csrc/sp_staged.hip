// sp_staged.hip -- reference-structured FP64 sweeps for gfx950.
//
// One kernel per reference stencil stage, each evaluating its expression in the
// operation order of the reference stencil functions with floating-point
// contraction disabled (this file is compiled with -ffp-contract=off and every
// kernel repeats `#pragma clang fp contract(off)`), so that on identical inputs
// the results are bit-for-bit those of the reference sweeps:
//   RHS4Stage   src/Convection/Convection.cpp:57-82  (Advection4 ConvectionFunctions.h:66-104,
//                                                      Laplace4 :135-166)
//   RHS2Stage   src/Convection/Convection.cpp:30-55  (Advection2 :4-64, Laplace2 :106-132)
//   EulerStage  src/Convection/Convection.cpp:84-101
//   RKStage     src/Convection/Convection.cpp:103-127
// Periodicity is index arithmetic: a neighbour at i-2 of i = 0 reads i = ni-2,
// the value the reference's halo fill (Periodicity.cpp:100-135) copies there
// for ni >= 2.
//
// Launch shape: 64 x 4 threads per block, one lattice point per thread, grid
// (ceil(ni/64), ceil(nj/4), nk * nslices).  Each wave reads 64 consecutive i
// (512 B), so every row access is one coalesced segment.

#include <cmath>

#include "sp_device.hpp"
#include "sp_internal.hpp"

namespace sp {
namespace {

__device__ __forceinline__ int wrap(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

struct Pt {
    int i, j, k, slice;
    bool ok;
};

__device__ __forceinline__ Pt point(int ni, int nj, int nk)
{
    Pt p;
    p.i = blockIdx.x * 64 + threadIdx.x;
    p.j = blockIdx.y * 4 + threadIdx.y;
    p.k = blockIdx.z % nk;
    p.slice = blockIdx.z / nk;
    p.ok = p.i < ni && p.j < nj;
    return p;
}

__device__ __forceinline__ const double* cptr(const View& v, const Pt& p)
{
    return (const double*)v.p + p.slice * v.slice;
}
__device__ __forceinline__ double* mptr(const View& v, const Pt& p) { return (double*)v.p + p.slice * v.slice; }

__global__ void __launch_bounds__(256) k_rhs4(StagedParams P, View q, View kf, double nu)
{
#pragma clang fp contract(off)
    const Pt p = point(P.ni, P.nj, P.nk);
    if (!p.ok) return;
    const double* Q = cptr(q, p);
    const long long sj = q.sj, sk = q.sk;
    const int i = p.i, j = p.j, k = p.k;
    const int im2 = wrap(i - 2, P.ni), im1 = wrap(i - 1, P.ni), ip1 = wrap(i + 1, P.ni), ip2 = wrap(i + 2, P.ni);
    const int jm2 = wrap(j - 2, P.nj), jm1 = wrap(j - 1, P.nj), jp1 = wrap(j + 1, P.nj), jp2 = wrap(j + 2, P.nj);
    const int km2 = wrap(k - 2, P.nk), km1 = wrap(k - 1, P.nk), kp1 = wrap(k + 1, P.nk), kp2 = wrap(k + 2, P.nk);
    const long long r = j * sj + k * sk;
    const double q0 = Q[r + i];
    const double qim2 = Q[r + im2], qim1 = Q[r + im1], qip1 = Q[r + ip1], qip2 = Q[r + ip2];
    const long long ck = k * sk + i;
    const double qjm2 = Q[ck + jm2 * sj], qjm1 = Q[ck + jm1 * sj], qjp1 = Q[ck + jp1 * sj], qjp2 = Q[ck + jp2 * sj];
    const long long cj = j * sj + i;
    const double qkm2 = Q[cj + km2 * sk], qkm1 = Q[cj + km1 * sk], qkp1 = Q[cj + kp1 * sk], qkp2 = Q[cj + kp2 * sk];
    // Advection4
    const double dq_di = -1. * qim2 + 8. * qim1 - 8. * qip1 + 1. * qip2;
    const double dq_dj = -1. * qjm2 + 8. * qjm1 - 8. * qjp1 + 1. * qjp2;
    const double dq_dk = -1. * qkm2 + 8. * qkm1 - 8. * qkp1 + 1. * qkp2;
    const double tensadv = (P.cx * dq_di + P.cy * dq_dj + P.cz * dq_dk) / (12. * P.dx);
    // Laplace4
    const double d2q_di2 = -1. * qim2 + 16. * qim1 - 30. * q0 + 16. * qip1 - 1. * qip2;
    const double d2q_dj2 = -1. * qjm2 + 16. * qjm1 - 30. * q0 + 16. * qjp1 - 1. * qjp2;
    const double d2q_dk2 = -1. * qkm2 + 16. * qkm1 - 30. * q0 + 16. * qkp1 - 1. * qkp2;
    const double lapl = (d2q_di2 + d2q_dj2 + d2q_dk2) / (12. * P.dx2);
    const double tenslapl = nu * lapl;
    mptr(kf, p)[i + j * kf.sj + k * kf.sk] = tensadv + tenslapl;
}

// What RHS2 divides by; where dx is a power of two (POW2) their reciprocals, whose products are
// the same numbers.
struct Spacing {
    double dx, dx2;  // upwind: dx; central: 2 dx
};

// RHS2 from a point and its six neighbours.  The upwind difference c (q0 - q(-1)) or
// c (q(+1) - q0) is |c| (q0 - q(upwind)): negating both factors changes no bits.
template <bool POW2>
__device__ __forceinline__ double rhs2_value(const StagedParams& P, const Spacing& d, double q0, double qim1,
                                             double qip1, double qjm1, double qjp1, double qkm1, double qkp1,
                                             double nu, int upwind)
{
#pragma clang fp contract(off)
    const auto over = [](double x, double y) { return POW2 ? x * y : x / y; };
    double tensadv;
    if (upwind) {
        const double dq_di = q0 - (P.cx > 0. ? qim1 : qip1);
        const double dq_dj = q0 - (P.cy > 0. ? qjm1 : qjp1);
        const double dq_dk = q0 - (P.cz > 0. ? qkm1 : qkp1);
        tensadv = over(-(fabs(P.cx) * dq_di + fabs(P.cy) * dq_dj + fabs(P.cz) * dq_dk), d.dx);
    } else {
        const double dq_di = +1. * qim1 - 1. * qip1;
        const double dq_dj = +1. * qjm1 - 1. * qjp1;
        const double dq_dk = +1. * qkm1 - 1. * qkp1;
        tensadv = over(P.cx * dq_di + P.cy * dq_dj + P.cz * dq_dk, d.dx);
    }
    const double d2q_di2 = +1. * qim1 - 2. * q0 + 1. * qip1;
    const double d2q_dj2 = +1. * qjm1 - 2. * q0 + 1. * qjp1;
    const double d2q_dk2 = +1. * qkm1 - 2. * q0 + 1. * qkp1;
    const double lapl = over(d2q_di2 + d2q_dj2 + d2q_dk2, d.dx2);
    const double tenslapl = nu * lapl;
    return tensadv + tenslapl;
}

template <bool POW2>
__device__ __forceinline__ double rhs2_point(const StagedParams& P, const Spacing& d, const double* Q, long long sj,
                                             long long sk, int i, int j, int k, double nu, int upwind)
{
    const int im1 = wrap(i - 1, P.ni), ip1 = wrap(i + 1, P.ni);
    const int jm1 = wrap(j - 1, P.nj), jp1 = wrap(j + 1, P.nj);
    const int km1 = wrap(k - 1, P.nk), kp1 = wrap(k + 1, P.nk);
    const long long r = j * sj + k * sk;
    return rhs2_value<POW2>(P, d, Q[r + i], Q[r + im1], Q[r + ip1], Q[i + jm1 * sj + k * sk], Q[i + jp1 * sj + k * sk],
                            Q[i + j * sj + km1 * sk], Q[i + j * sj + kp1 * sk], nu, upwind);
}

__global__ void __launch_bounds__(256) k_rhs2(StagedParams P, Spacing d, View q, View kf, double nu, int upwind)
{
#pragma clang fp contract(off)
    const Pt p = point(P.ni, P.nj, P.nk);
    if (!p.ok) return;
    const double r = rhs2_point<false>(P, d, cptr(q, p), q.sj, q.sk, p.i, p.j, p.k, nu, upwind);
    mptr(kf, p)[p.i + p.j * kf.sj + p.k * kf.sk] = r;
}

// EulerStage: out = q + dt*k.  DoEulerTimestep (Convection.cpp:372-392) as one
// pass: k is the RHS2 value of this point, then the Euler update.
template <bool POW2>
__global__ void __launch_bounds__(256) k_euler_fused(StagedParams P, Spacing d, View qin, View qout, double nu, double dt,
                                                     int upwind)
{
#pragma clang fp contract(off)
    const Pt p = point(P.ni, P.nj, P.nk);
    if (!p.ok) return;
    const double* Q = cptr(qin, p);
    const double k = rhs2_point<POW2>(P, d, Q, qin.sj, qin.sk, p.i, p.j, p.k, nu, upwind);
    const double q0 = Q[p.i + p.j * qin.sj + p.k * qin.sk];
    mptr(qout, p)[p.i + p.j * qout.sj + p.k * qout.sk] = q0 + dt * k;
}

// Two forward Euler steps in one launch.  One step alone moves 16 bytes per point for some 25
// operations and two divisions; here a block loads a 16x16x8 brick with a halo of two cells into
// LDS (38 KB), advances it on the 18x18x10 cells the second step reads, and then on the brick.
// A lane walks a column along k and keeps the values above and below in registers; the first
// step's results wait in registers until every lane has read, then replace the field in LDS.
// Each point is the expression of DoEulerTimestep (Convection.cpp:372-392) in the reference's
// order: the same bits as two launches.  Where dx is a power of two the two divisions are
// products (the same numbers).  Measured per step, before and now: 96^3 9.0 -> 5.6 us, 128^3
// 12.3 -> 6.4, 192^3 34 -> 25, 256^3 79 -> 40, 384^3 318 -> 193; 64^3 and smaller are bound by the
// launches.  Three and four steps per launch were slower from 96^3 on (128^3 8.5 and 8.7 us, 384^3
// 241 and 258): 1.9 and 2.5 times the points' operations.
struct EulerBrick {
    StagedParams P;
    Spacing d;
    View in, out;
    unsigned in_bytes, out_bytes;  // bytes one slice's storage spans from its origin
    int tiles_x, tiles, chunks;
    double nu[2];  // of the two steps
    double dt;
};
constexpr int kEulerNT = 512, kEulerBX = 16, kEulerBZ = 8;

constexpr int kEulerHalo = 2, kEulerW = kEulerBX + 2 * kEulerHalo;

// Step T (0, 1) on the brick and 1 - T cells around it; the second writes to the output field.
template <int T, bool POW2, bool UP>
__device__ __forceinline__ void euler_brick_step(const EulerBrick& a, double* P, __amdgpu_buffer_rsrc_t rout, int x0,
                                                 int y0, int z0)
{
#pragma clang fp contract(off)
    constexpr int W = kEulerW, PL = W * W;
    constexpr int h = 1 - T, C = kEulerBX + 2 * h, COLS = C * C;
    constexpr int ZS = 2 * COLS <= kEulerNT ? 2 : 1;  // lanes per column
    constexpr int N = (kEulerBZ + 2 * h) / ZS;
    static_assert(COLS * ZS <= kEulerNT, "one column part per lane");
    const int tid = threadIdx.x, half = ZS == 2 ? tid / COLS : 0, c = tid - half * COLS;
    const bool live = tid < COLS * ZS;
    const int x = c % C, y = c / C;
    double* const p = P + (kEulerHalo - h + half * N) * PL + (kEulerHalo - h + y) * W + kEulerHalo - h + x;
    double r[N];
    if (live) {
        double below = p[-PL], q0 = p[0];
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const double* const q = p + j * PL;
            const double above = q[PL];
            const double k = rhs2_value<POW2>(a.P, a.d, q0, q[-1], q[1], q[-W], q[W], below, above, a.nu[T], UP);
            r[j] = q0 + a.dt * k;
            below = q0;
            q0 = above;
            __builtin_amdgcn_sched_barrier(0);  // one point's values in flight: 52 registers
        }
    }
    if constexpr (T == 0) {
        __syncthreads();
        if (live) {
#pragma unroll
            for (int j = 0; j < N; ++j) p[j * PL] = r[j];
        }
        __syncthreads();
    } else if (live) {
        const int oskb = (int)a.out.sk * 8;
        // periodic image for partial bricks
        const int o = (near_mod(x0 + x, a.P.ni) + near_mod(y0 + y, a.P.nj) * (int)a.out.sj) * 8;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const int z = z0 + half * N + j;
            if (z < a.P.nk) st_through(rout, o + z * oskb, 0, r[j]);
        }
    }
}

template <bool PAIR, bool POW2, bool UP>
__global__ void __launch_bounds__(kEulerNT, 4) k_euler_brick(EulerBrick a)
{
    constexpr int H = kEulerHalo, W = kEulerW, D = kEulerBZ + 2 * H;
    __shared__ __attribute__((aligned(16))) double P[D * W * W];
    const int bid = xcd_block(blockIdx.x, gridDim.x);
    const int tile = bid % a.tiles, chunk = (bid / a.tiles) % a.chunks, slice = bid / (a.tiles * a.chunks);
    const int x0 = (tile % a.tiles_x) * kEulerBX, y0 = (tile / a.tiles_x) * kEulerBX, z0 = chunk * kEulerBZ;
    const __amdgpu_buffer_rsrc_t rin = make_rsrc((const double*)a.in.p + slice * a.in.slice, a.in_bytes);
    const __amdgpu_buffer_rsrc_t rout = make_rsrc((double*)a.out.p + slice * a.out.slice, a.out_bytes);
    brick_load<PAIR, W, W, D>(P, rin, (int)a.in.sk * 8, (int)a.in.sj, x0 - H, y0 - H, z0 - H, a.P.ni, a.P.nj, a.P.nk,
                              __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), threadIdx.x & 63);
    vm_wait<0>();
    lds_barrier();
    euler_brick_step<0, POW2, UP>(a, P, rout, x0, y0, z0);
    euler_brick_step<1, POW2, UP>(a, P, rout, x0, y0, z0);
}

__global__ void __launch_bounds__(256) k_euler_stage(StagedParams P, View qin, View kf, View qout, double dt)
{
#pragma clang fp contract(off)
    const Pt p = point(P.ni, P.nj, P.nk);
    if (!p.ok) return;
    const double q0 = cptr(qin, p)[p.i + p.j * qin.sj + p.k * qin.sk];
    const double k = cptr(kf, p)[p.i + p.j * kf.sj + p.k * kf.sk];
    const double dt_ = dt;
    mptr(qout, p)[p.i + p.j * qout.sj + p.k * qout.sk] = q0 + dt_ * k;
}

__global__ void __launch_bounds__(256) k_rk_stage(StagedParams P, View qin, View k1, View k2, View k3, View k4,
                                                  View qout, double dt)
{
#pragma clang fp contract(off)
    const Pt p = point(P.ni, P.nj, P.nk);
    if (!p.ok) return;
    const long long o = p.i + p.j * qin.sj + p.k * qin.sk;
    const long long ok = p.i + p.j * k1.sj + p.k * k1.sk;
    const double q0 = cptr(qin, p)[o];
    const double a1 = cptr(k1, p)[ok], a2 = cptr(k2, p)[ok], a3 = cptr(k3, p)[ok], a4 = cptr(k4, p)[ok];
    mptr(qout, p)[p.i + p.j * qout.sj + p.k * qout.sk] = q0 + dt / 6. * (a1 + 2. * a2 + 2. * a3 + a4);
}

// a power of two whose square's reciprocal is one too
bool power_of_two(double x)
{
    int e;
    return std::frexp(x, &e) == 0.5 && e > -400 && e < 400;
}

Spacing spacing(const StagedParams& P, int upwind)
{
    const Spacing d{upwind ? P.dx : 2. * P.dx, P.dx2};
    return power_of_two(P.dx) ? Spacing{1. / d.dx, 1. / d.dx2} : d;
}

dim3 grid_of(const StagedParams& P, int nslices)
{
    return dim3((P.ni + 63) / 64, (P.nj + 3) / 4, P.nk * nslices);
}

}  // namespace

int launch_rhs4(hipStream_t s, const StagedParams& P, View q, View k, double nu)
{
    hipLaunchKernelGGL(k_rhs4, grid_of(P, 1), dim3(64, 4), 0, s, P, q, k, nu);
    SP_HIP(hipGetLastError());
    return SP_OK;
}

int launch_rhs2(hipStream_t s, const StagedParams& P, View q, View k, double nu, int upwind)
{
    const Spacing d{upwind ? P.dx : 2. * P.dx, P.dx2};
    hipLaunchKernelGGL(k_rhs2, grid_of(P, 1), dim3(64, 4), 0, s, P, d, q, k, nu, upwind);
    SP_HIP(hipGetLastError());
    return SP_OK;
}

int launch_euler_stage(hipStream_t s, const StagedParams& P, View qin, View k, View qout, double dt)
{
    hipLaunchKernelGGL(k_euler_stage, grid_of(P, 1), dim3(64, 4), 0, s, P, qin, k, qout, dt);
    SP_HIP(hipGetLastError());
    return SP_OK;
}

int launch_rk_stage(hipStream_t s, const StagedParams& P, View qin, View k1, View k2, View k3, View k4, View qout,
                    double dt)
{
    hipLaunchKernelGGL(k_rk_stage, grid_of(P, 1), dim3(64, 4), 0, s, P, qin, k1, k2, k3, k4, qout, dt);
    SP_HIP(hipGetLastError());
    return SP_OK;
}

int launch_euler_fused(hipStream_t s, const StagedParams& P, View qin, View qout, double nu, double dt, int upwind,
                       int nslices)
{
    if (power_of_two(P.dx))
        hipLaunchKernelGGL(k_euler_fused<true>, grid_of(P, nslices), dim3(64, 4), 0, s, P, spacing(P, upwind), qin, qout, nu, dt, upwind);
    else
        hipLaunchKernelGGL(k_euler_fused<false>, grid_of(P, nslices), dim3(64, 4), 0, s, P, spacing(P, upwind), qin, qout, nu, dt, upwind);
    SP_HIP(hipGetLastError());
    return SP_OK;
}

namespace {

template <bool PAIR, bool POW2>
void euler_brick(hipStream_t s, unsigned blocks, const EulerBrick& a, int upwind)
{
    if (upwind) hipLaunchKernelGGL((k_euler_brick<PAIR, POW2, true>), dim3(blocks), dim3(kEulerNT), 0, s, a);
    else hipLaunchKernelGGL((k_euler_brick<PAIR, POW2, false>), dim3(blocks), dim3(kEulerNT), 0, s, a);
}

// Bytes one slice spans from its first point.
long long span_bytes(const StagedParams& P, const View& v)
{
    return ((P.ni - 1) + (P.nj - 1) * v.sj + (P.nk - 1) * v.sk + 1) * 8;
}

}  // namespace

bool euler_two_steps(const StagedParams& P, View qin, View qout)
{
    // bricks address a field through a buffer resource (2 GiB), and their planes' periodic
    // images reach 9 planes past the field
    return P.nk >= kFusedMinK && span_bytes(P, qin) < (1LL << 31) && span_bytes(P, qout) < (1LL << 31);
}

int launch_euler_two(hipStream_t s, const StagedParams& P, View qin, View qout, const double nu[2], double dt, int upwind,
                     int nslices)
{
    EulerBrick a;
    a.P = P;
    a.d = spacing(P, upwind);
    a.in = qin;
    a.out = qout;
    a.in_bytes = (unsigned)span_bytes(P, qin);
    a.out_bytes = (unsigned)span_bytes(P, qout);
    a.tiles_x = (P.ni + kEulerBX - 1) / kEulerBX;
    a.tiles = a.tiles_x * ((P.nj + kEulerBX - 1) / kEulerBX);
    a.chunks = (P.nk + kEulerBZ - 1) / kEulerBZ;
    a.nu[0] = nu[0];
    a.nu[1] = nu[1];
    a.dt = dt;
    const long long blocks = (long long)a.tiles * a.chunks * nslices;
    SP_CHECK(blocks <= 0x7fffffffLL, SP_ERR_UNSUPPORTED, "Euler steps: too many blocks");
    const auto even = [](long long v) { return (v & 1) == 0; };
    const bool pair = even(P.ni) && even(qin.sj) && even(qin.sk) && even(qin.slice) && ((uintptr_t)qin.p % 16) == 0;
    const bool pow2 = power_of_two(P.dx);
    if (pair && pow2) euler_brick<true, true>(s, (unsigned)blocks, a, upwind);
    else if (pair) euler_brick<true, false>(s, (unsigned)blocks, a, upwind);
    else if (pow2) euler_brick<false, true>(s, (unsigned)blocks, a, upwind);
    else euler_brick<false, false>(s, (unsigned)blocks, a, upwind);
    SP_HIP(hipGetLastError());
    return SP_OK;
}

}  // namespace sp
