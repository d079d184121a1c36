// sp_fused.hip -- one RK4 step of the advection-diffusion operator in one kernel.
//
// What it computes (reference: Convection::DoRK4Timestep, src/Convection/Convection.cpp:318-370,
// stages :57-127).  The right-hand side L q = Advection4(q) + nu*Laplace4(q) is linear and nu is
// fixed for the whole step (Convection.cpp:321), so the four RK4 stages
//   k1 = Lq, k2 = L(q + h/2 k1), k3 = L(q + h/2 k2), k4 = L(q + h k3),
//   q' = q + h/6 (k1 + 2k2 + 2k3 + k4)
// equal the nested form (same polynomial P(hL) = 1 + hL + (hL)^2/2 + (hL)^3/6 + (hL)^4/24):
//   v1 = q + (h/4) L q,  v2 = q + (h/3) L v1,  v3 = q + (h/2) L v2,  q' = q + h L v3.
// Results agree with the reference sweeps to rounding (a few ulp per step); the
// reference-order kernels in sp_staged.hip give the bit-exact path.
//
// How (gfx950, wave64):
//  * A block owns a TX x TY tile of output columns and a chunk of CZ planes in k.  It
//    streams planes k = z0-8 .. z0+CZ+7 of the input once (8 = 4 stages x radius 2).
//  * Stage s reads its input plane from LDS (x-y neighbours) and keeps the k-direction
//    in registers as four running partial sums per column: when plane p arrives it
//    completes point p-2 and starts p+2.  Stage s therefore lags 2 planes behind stage
//    s-1; its output plane goes to the next stage's LDS buffer.
//  * The x-y region a stage computes shrinks by 2 per side per stage (6, 4, 2, 0 halo),
//    so only the ring needed by later stages is recomputed.  Each stage maps its own
//    region flat onto the block's threads, so inactive lanes are only the tail.
//  * The state q needed by each stage's update (v_s = q + ...) is re-read from global
//    memory one plane ahead of its use (an L2 hit: the block loaded it a few planes
//    earlier), keeping the per-column register state at 4 partial sums per stage.
//  * The four running sums of a column are a circular buffer indexed by plane mod 4 and
//    the k loop is unrolled by 4, so advancing a plane moves no registers.
//  * The 13 stencil coefficients and the stage factors are computed on the host and
//    arrive as kernel arguments (scalar registers); global accesses are buffer
//    instructions with the plane offset in a scalar register.
//  * HBM traffic per step: one read and one write of the state (2*sizeof(storage) bytes
//    per lattice update) plus the x-y halo overlap of neighbouring tiles.
//  * The plane for iteration t+1 is loaded into registers while iteration t computes.
// That is the scalar kernel (any sizes and storage types).  The FP64 x-pair and 2x2
// variants further down keep the scheme and change the lane layout (16-byte accesses,
// shared neighbour reads), the way q reaches each stage and the prefetch depth; their
// own comments give the details.

#include <algorithm>
#include <cstring>

#include "sp_device.hpp"
#include "sp_internal.hpp"

namespace sp {

namespace {

// Host-computed coefficients of one step: the 13 star weights of L (offsets -2,-1,+1,+2
// per axis, then the centre) and the stage factors h/4, h/3, h/2, h, in both precisions.
struct Coefs {
    double wd[13];
    double fd[4];
    float wf[13];
    float ff[4];
};

struct FusedArgs {
    View in, out;
    unsigned in_bytes, out_bytes;  // bytes one slice's storage spans from its origin
    int ni, nj, nk;
    int kchunk, chunks;
    int tiles_x, tiles;
    Coefs c;                 // used when cdev == nullptr
    const Coefs* cdev;       // per-slice coefficients (time-dependent nu), or nullptr
};

// A grouped launch: n argument records in device memory and their first block indices.
struct GroupArgs {
    const FusedArgs* __restrict__ args;
    const int* __restrict__ first;
    int n;
};

__device__ __forceinline__ double fmaT(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fmaT(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

template <typename T>
struct StarW {
    T xm2, xm1, xp1, xp2, ym2, ym1, yp1, yp2, zm2, zm1, zp1, zp2, c;
    T f1, f2, f3, f4;
};

template <typename T>
__device__ __forceinline__ StarW<T> load_w(const Coefs& k);
template <>
__device__ __forceinline__ StarW<double> load_w<double>(const Coefs& k)
{
    return StarW<double>{k.wd[0], k.wd[1], k.wd[2], k.wd[3], k.wd[4], k.wd[5], k.wd[6], k.wd[7], k.wd[8],
                         k.wd[9], k.wd[10], k.wd[11], k.wd[12], k.fd[0], k.fd[1], k.fd[2], k.fd[3]};
}
template <>
__device__ __forceinline__ StarW<float> load_w<float>(const Coefs& k)
{
    return StarW<float>{k.wf[0], k.wf[1], k.wf[2], k.wf[3], k.wf[4], k.wf[5], k.wf[6], k.wf[7], k.wf[8],
                        k.wf[9], k.wf[10], k.wf[11], k.wf[12], k.ff[0], k.ff[1], k.ff[2], k.ff[3]};
}

// Stage geometry: stage s (1..4) computes a (TX+2h) x (TY+2h) region, h = 8-2s, from an
// input plane of (TX+2h+4) x (TY+2h+4) held in LDS.
template <int TX, int TY, int S>
struct Geo {
    static constexpr int HO = 8 - 2 * S;
    static constexpr int WO = TX + 2 * HO, HOo = TY + 2 * HO, AO = WO * HOo;
    static constexpr int WI = WO + 4, HI = HOo + 4, AI = WI * HI;
};

// One stage at one plane: consume input plane p (in LDS), emit the completed sum of
// plane p-2 in done[].  The running sums of points p-2 .. p+1 sit in slots (x mod 4)
// of acc; R is the slot of point p.  Every slot m is processed (slots past the region's
// end repeat its last column), so the stream has no per-lane branches.
template <typename T, int TX, int TY, int S, int NT, int M, int R>
__device__ __forceinline__ void stage_step(const T* __restrict__ P, const StarW<T>& w, T (&acc)[M][4], T (&done)[M])
{
    using G = Geo<TX, TY, S>;
    constexpr int WI = G::WI;
    constexpr int sm2 = (R + 2) & 3, sm1 = (R + 3) & 3, s0 = R & 3, sp1 = (R + 1) & 3;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        // LDS centre of this slot's column (recomputed: constant divisors, saves registers)
        const int f = min((int)threadIdx.x + m * NT, G::AO - 1);
        const T* c = P + (f / G::WO + 2) * WI + f % G::WO + 2;
        const T u = c[0];
        const T xm2 = c[-2], xm1 = c[-1], xp1 = c[1], xp2 = c[2];
        const T ym2 = c[-2 * WI], ym1 = c[-WI], yp1 = c[WI], yp2 = c[2 * WI];
        done[m] = fmaT(w.zp2, u, acc[m][sm2]);            // point p-2: its +2 neighbour is p
        acc[m][sm2] = w.zm2 * u;                          // point p+2 starts in the same slot
        acc[m][sm1] = fmaT(w.zp1, u, acc[m][sm1]);        // point p-1
        // point p: centre and x-y neighbours, as two independent chains (x, y)
        T ax = fmaT(w.c, u, acc[m][s0]);
        T ay = w.ym2 * ym2;
        ax = fmaT(w.xm2, xm2, ax);
        ay = fmaT(w.ym1, ym1, ay);
        ax = fmaT(w.xm1, xm1, ax);
        ay = fmaT(w.yp1, yp1, ay);
        ax = fmaT(w.xp1, xp1, ax);
        ay = fmaT(w.yp2, yp2, ay);
        ax = fmaT(w.xp2, xp2, ax);
        acc[m][s0] = ax + ay;
        acc[m][sp1] = fmaT(w.zm1, u, acc[m][sp1]);        // point p+1
        // one slot's neighbour values in flight at a time keeps the register footprint
        // small enough for 16 waves per CU; the other waves hide the LDS latency
        __builtin_amdgcn_sched_barrier(0);
    }
}

template <typename S>
struct Buf;
template <>
struct Buf<double> {
    using T = double;
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    __device__ __forceinline__ static double ld(__amdgpu_buffer_rsrc_t r, int vo, int so)
    {
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, vo, so, 0));
    }
    __device__ __forceinline__ static void st(__amdgpu_buffer_rsrc_t r, int vo, int so, double x)
    {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), r, vo, so, 0);
    }
};
template <>
struct Buf<float> {
    __device__ __forceinline__ static float ld(__amdgpu_buffer_rsrc_t r, int vo, int so)
    {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, vo, so, 0));
    }
    __device__ __forceinline__ static void st(__amdgpu_buffer_rsrc_t r, int vo, int so, float x)
    {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x), r, vo, so, 0);
    }
};
template <>
struct Buf<bf16> {
    __device__ __forceinline__ static float ld(__amdgpu_buffer_rsrc_t r, int vo, int so)
    {
        return bf16_to_f32((uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, vo, so, 0));
    }
    __device__ __forceinline__ static void st(__amdgpu_buffer_rsrc_t r, int vo, int so, float x)
    {
        __builtin_amdgcn_raw_buffer_store_b16((unsigned short)f32_to_bf16(x), r, vo, so, 0);
    }
};

// Per-column constants of one stage: LDS centre index and the byte offset of the column
// in the input field (for the q value of the update).  Slots past the region's end repeat
// its last column.
template <int M>
struct Cols {
    int q[M];
};

template <typename SI, int TX, int TY, int S, int NT, int M>
__device__ __forceinline__ void stage_cols(Cols<M>& cl, int x0, int y0, int ni, int nj, int sj)
{
    using G = Geo<TX, TY, S>;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int f = min((int)threadIdx.x + m * NT, G::AO - 1);
        const int ax = f % G::WO, by = f / G::WO;
        cl.q[m] = (pmod(x0 - G::HO + ax, ni) + pmod(y0 - G::HO + by, nj) * sj) * (int)sizeof(SI);
    }
}

// Loads the q values a stage needs for its update at the plane whose byte offset is zo.
template <typename SI, typename T, int M>
__device__ __forceinline__ void stage_qload(T (&qv)[M], __amdgpu_buffer_rsrc_t r, int zo, const Cols<M>& cl)
{
#pragma unroll
    for (int m = 0; m < M; ++m) qv[m] = (T)Buf<SI>::ld(r, cl.q[m], zo);
}

template <typename SI, typename SO, typename T, int TX, int TY, int NT>
__device__ __forceinline__ void rk4_scalar_body(const FusedArgs& a, const int bid)
{
    using G1 = Geo<TX, TY, 1>;
    using G2 = Geo<TX, TY, 2>;
    using G3 = Geo<TX, TY, 3>;
    using G4 = Geo<TX, TY, 4>;
    constexpr int A0 = G1::AI;  // q plane (stage-1 input) incl. 8-cell halo
    constexpr int M0 = (A0 + NT - 1) / NT;
    constexpr int M1 = (G1::AO + NT - 1) / NT;
    constexpr int M2 = (G2::AO + NT - 1) / NT;
    constexpr int M3 = (G3::AO + NT - 1) / NT;
    constexpr int M4 = (G4::AO + NT - 1) / NT;

    // Every plane buffer is doubled: in iteration t stage s reads what stage s-1 wrote in
    // iteration t-1, so all four stages run between one barrier per plane.
    __shared__ T P0[2][G1::AI];
    __shared__ T P1[2][G2::AI];
    __shared__ T P2[2][G3::AI];
    __shared__ T P3[2][G4::AI];

    const int tid = threadIdx.x;
    const int ni = a.ni, nj = a.nj, nk = a.nk;
    // block -> (tile, k chunk, slice); tiles fastest
    const int tile = bid % a.tiles;
    const int chunk = (bid / a.tiles) % a.chunks;
    const int slice = bid / (a.tiles * a.chunks);
    const int x0 = (tile % a.tiles_x) * TX, y0 = (tile / a.tiles_x) * TY;
    const int z0 = chunk * a.kchunk;
    const int zend = min(z0 + a.kchunk, nk);
    const __amdgpu_buffer_rsrc_t rin = make_rsrc((const SI*)a.in.p + slice * a.in.slice, a.in_bytes);
    const __amdgpu_buffer_rsrc_t rout = make_rsrc((SO*)a.out.p + slice * a.out.slice, a.out_bytes);
    const int iskb = (int)a.in.sk * (int)sizeof(SI), oskb = (int)a.out.sk * (int)sizeof(SO);
    const int isj = (int)a.in.sj, osj = (int)a.out.sj;
    const StarW<T> w = a.cdev ? load_w<T>(a.cdev[slice]) : load_w<T>(a.c);

    // Per-column offsets, fixed for the whole k stream.
    int off0[M0];
#pragma unroll
    for (int m = 0; m < M0; ++m) {
        const int f = min(tid + m * NT, A0 - 1);
        const int ax = f % G1::WI, by = f / G1::WI;
        off0[m] = (pmod(x0 - 8 + ax, ni) + pmod(y0 - 8 + by, nj) * isj) * (int)sizeof(SI);
    }
    Cols<M1> c1;
    Cols<M2> c2;
    Cols<M3> c3;
    Cols<M4> c4;
    stage_cols<SI, TX, TY, 1, NT, M1>(c1, x0, y0, ni, nj, isj);
    stage_cols<SI, TX, TY, 2, NT, M2>(c2, x0, y0, ni, nj, isj);
    stage_cols<SI, TX, TY, 3, NT, M3>(c3, x0, y0, ni, nj, isj);
    stage_cols<SI, TX, TY, 4, NT, M4>(c4, x0, y0, ni, nj, isj);
    int o4[M4];
#pragma unroll
    for (int m = 0; m < M4; ++m) {
        const int fc = min(tid + m * NT, G4::AO - 1);
        const int gx = x0 + fc % G4::WO, gy = y0 + fc / G4::WO;
        // columns of a partial tile past the domain edge are written to their periodic image
        // (where another block writes the same bits)
        o4[m] = (pmod(gx, ni) + pmod(gy, nj) * osj) * (int)sizeof(SO);
    }

    T acc1[M1][4], acc2[M2][4], acc3[M3][4], acc4[M4][4];
    T d1[M1], d2[M2], d3[M3], d4[M4];
    T qv1[M1], qv2[M2], qv3[M3], qv4[M4];  // q for the update, loaded one plane ahead
#pragma unroll
    for (int m = 0; m < M1; ++m) acc1[m][0] = acc1[m][1] = acc1[m][2] = acc1[m][3] = T(0);
#pragma unroll
    for (int m = 0; m < M2; ++m) acc2[m][0] = acc2[m][1] = acc2[m][2] = acc2[m][3] = T(0);
#pragma unroll
    for (int m = 0; m < M3; ++m) acc3[m][0] = acc3[m][1] = acc3[m][2] = acc3[m][3] = T(0);
#pragma unroll
    for (int m = 0; m < M4; ++m) acc4[m][0] = acc4[m][1] = acc4[m][2] = acc4[m][3] = T(0);

    // Iteration t: stage 1 takes q plane t and emits v1 plane t-2; stage 2 takes v1 plane
    // t-3 (written in iteration t-1) and emits v2 plane t-5; stage 3: v2 t-6 -> v3 t-8;
    // stage 4: v3 t-9 -> q' t-11.  Stage s runs while its input planes are valid.
    const int tq0 = z0 - 8, tq1 = zend + 8;  // q planes to stream
    const int tend = zend + 11;
    {
        // q plane tq0 into P0[tq0 & 1]
        const int zo = wrapz(tq0, nk) * iskb;
#pragma unroll
        for (int m = 0; m < M0; ++m) P0[tq0 & 1][min(tid + m * NT, A0 - 1)] = (T)Buf<SI>::ld(rin, off0[m], zo);
        stage_qload<SI, T, M1>(qv1, rin, wrapz(tq0 - 2, nk) * iskb, c1);
        stage_qload<SI, T, M2>(qv2, rin, wrapz(z0 - 8, nk) * iskb, c2);
        stage_qload<SI, T, M3>(qv3, rin, wrapz(z0 - 6, nk) * iskb, c3);
        stage_qload<SI, T, M4>(qv4, rin, wrapz(z0 - 4, nk) * iskb, c4);
    }
    T pre[M0];
    if (tq0 + 1 < tq1) {
        const int zo = wrapz(tq0 + 1, nk) * iskb;
#pragma unroll
        for (int m = 0; m < M0; ++m) pre[m] = (T)Buf<SI>::ld(rin, off0[m], zo);
    }
    __syncthreads();

    // One plane of the stream; R = (t - tq0) mod 4 is a compile-time constant so the slots of
    // the running sums are static register names.  Slot of point x = (x - tq0) mod 4.
    auto plane = [&](auto Rc, int t) {
        constexpr int R = decltype(Rc)::value;
        const int cur = t & 1, prv = cur ^ 1;
        __builtin_amdgcn_sched_barrier(0);  // keep planes apart: bounded live ranges
        // next q plane from registers into the other P0 buffer; start loading the one after
        if (t + 1 < tq1) {
#pragma unroll
            for (int m = 0; m < M0; ++m) P0[prv][min(tid + m * NT, A0 - 1)] = pre[m];
            if (t + 2 < tq1) {
                const int zo = wrapz(t + 2, nk) * iskb;
#pragma unroll
                for (int m = 0; m < M0; ++m) pre[m] = (T)Buf<SI>::ld(rin, off0[m], zo);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // Stage 1: q plane t -> v1 plane t-2.
        if (t < tq1) {
            stage_step<T, TX, TY, 1, NT, M1, R & 3>(P0[cur], w, acc1, d1);
#pragma unroll
            for (int m = 0; m < M1; ++m) P1[cur][min(tid + m * NT, G1::AO - 1)] = fmaT(w.f1, d1[m], qv1[m]);
            stage_qload<SI, T, M1>(qv1, rin, wrapz(t - 1, nk) * iskb, c1);
            __builtin_amdgcn_sched_barrier(0);
        }
        // Stage 2: v1 plane t-3 -> v2 plane t-5.
        if (t >= tq0 + 5 && t < tq1 + 1) {
            stage_step<T, TX, TY, 2, NT, M2, (R + 1) & 3>(P1[prv], w, acc2, d2);
#pragma unroll
            for (int m = 0; m < M2; ++m) P2[cur][min(tid + m * NT, G2::AO - 1)] = fmaT(w.f2, d2[m], qv2[m]);
            stage_qload<SI, T, M2>(qv2, rin, wrapz(t - 4, nk) * iskb, c2);
            __builtin_amdgcn_sched_barrier(0);
        }
        // Stage 3: v2 plane t-6 -> v3 plane t-8.
        if (t >= tq0 + 10 && t < tq1 + 2) {
            stage_step<T, TX, TY, 3, NT, M3, (R + 2) & 3>(P2[prv], w, acc3, d3);
#pragma unroll
            for (int m = 0; m < M3; ++m) P3[cur][min(tid + m * NT, G3::AO - 1)] = fmaT(w.f3, d3[m], qv3[m]);
            stage_qload<SI, T, M3>(qv3, rin, wrapz(t - 7, nk) * iskb, c3);
            __builtin_amdgcn_sched_barrier(0);
        }
        // Stage 4: v3 plane t-9 -> q' plane t-11.
        if (t >= tq0 + 15) {
            stage_step<T, TX, TY, 4, NT, M4, (R + 3) & 3>(P3[prv], w, acc4, d4);
            const int zp = t - 11;
            if (zp >= z0 && zp < zend) {
                const int zo = zp * oskb;
#pragma unroll
                for (int m = 0; m < M4; ++m) Buf<SO>::st(rout, o4[m], zo, fmaT(w.f4, d4[m], qv4[m]));
            }
            stage_qload<SI, T, M4>(qv4, rin, wrapz(t - 10, nk) * iskb, c4);
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };

    // Stage s runs while its input planes are valid.  The loop is unrolled by 4 so that
    // the phase R of every plane is a compile-time constant.
    for (int t = tq0; t < tend; t += 4) {
        plane(std::integral_constant<int, 0>{}, t);
        if (t + 1 < tend) plane(std::integral_constant<int, 1>{}, t + 1);
        if (t + 2 < tend) plane(std::integral_constant<int, 2>{}, t + 2);
        if (t + 3 < tend) plane(std::integral_constant<int, 3>{}, t + 3);
    }
}


// ---- FP64 x-pair variant ----------------------------------------------------------------
// Each lane owns two x-adjacent columns, so every LDS and global access moves 16 bytes
// (ds_read_b128 / buffer_load_dwordx4): per pair and stage, 7 LDS reads give the two centres,
// the four x and eight y neighbours.  Needs even ni and even, 16-byte aligned strides.
typedef double d2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ d2 ld2(__amdgpu_buffer_rsrc_t r, int vo, int so)
{
    return __builtin_bit_cast(d2, __builtin_amdgcn_raw_buffer_load_b128(r, vo, so, 0));
}
__device__ __forceinline__ void st2(__amdgpu_buffer_rsrc_t r, int vo, int so, d2 x)
{
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x), r, vo, so, 0);
}

// Non-temporal variants (cache policy nt): the output plane of a step is not read again in
// that step, and a block's lag-8 reload of q is that plane's last use, so neither needs to
// stay in the XCD's L2 beside the planes the stream will still reuse (the 2x2 kernel's
// counted reads at 64 x 384^3: 3.26x -> 2.73x the state).
__device__ __forceinline__ d2 ld2_last(__amdgpu_buffer_rsrc_t r, int vo, int so)
{
    return __builtin_bit_cast(d2, __builtin_amdgcn_raw_buffer_load_b128(r, vo, so, 2));
}
__device__ __forceinline__ void st2_stream(__amdgpu_buffer_rsrc_t r, int vo, int so, d2 x)
{
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x), r, vo, so, 2);
}
// Two x-adjacent values of compute type T (d2 for FP64), and their global access for
// storage type S: 2 * sizeof(S) bytes per lane (FP64 16, FP32 8, BF16 4), converted to T.
template <typename T>
struct V2 {
    typedef T type __attribute__((ext_vector_type(2)));
};
template <typename S, typename T>
struct PairIO;
template <>
struct PairIO<double, double> {
    __device__ __forceinline__ static d2 ld(__amdgpu_buffer_rsrc_t r, int vo, int so) { return ld2(r, vo, so); }
    __device__ __forceinline__ static void st(__amdgpu_buffer_rsrc_t r, int vo, int so, d2 x) { st2(r, vo, so, x); }
};
template <>
struct PairIO<float, float> {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    __device__ __forceinline__ static f2 ld(__amdgpu_buffer_rsrc_t r, int vo, int so)
    {
        return __builtin_bit_cast(f2, __builtin_amdgcn_raw_buffer_load_b64(r, vo, so, 0));
    }
    __device__ __forceinline__ static void st(__amdgpu_buffer_rsrc_t r, int vo, int so, f2 x)
    {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), r, vo, so, 0);
    }
};
template <>
struct PairIO<double, float> {  // FP64 input of a reduced-precision step: rounded to FP32 on load
    typedef float f2 __attribute__((ext_vector_type(2)));
    __device__ __forceinline__ static f2 ld(__amdgpu_buffer_rsrc_t r, int vo, int so)
    {
        const d2 v = ld2(r, vo, so);
        return f2{(float)v.x, (float)v.y};
    }
};
template <>
struct PairIO<bf16, float> {
    typedef float f2 __attribute__((ext_vector_type(2)));
    __device__ __forceinline__ static f2 ld(__amdgpu_buffer_rsrc_t r, int vo, int so)
    {
        const unsigned v = __builtin_amdgcn_raw_buffer_load_b32(r, vo, so, 0);
        return f2{bf16_to_f32((uint16_t)(v & 0xffffu)), bf16_to_f32((uint16_t)(v >> 16))};
    }
    __device__ __forceinline__ static void st(__amdgpu_buffer_rsrc_t r, int vo, int so, f2 x)
    {
        const unsigned v = (unsigned)f32_to_bf16(x.x) | ((unsigned)f32_to_bf16(x.y) << 16);
        __builtin_amdgcn_raw_buffer_store_b32(v, r, vo, so, 0);
    }
};

// Lane-slot layout of stage S's output pairs (WP pairs x H rows).  Slot g maps to pair
// (ax / 2, by), row-major with VW slots per row.  With VW equal to the input plane's row
// stride in pairs (WI / 2), consecutive slots read consecutive 16-byte LDS chunks across
// row ends too, so no 16-lane group of a ds_read_b128 touches a bank twice; the slots past
// a row's last pair repeat it (same address: a broadcast, and the same value written).
// That layout is used whenever it needs no more passes of NT threads than the dense one
// (VW = WP), whose groups straddling a row end hit two banks twice, unless rows are whole
// 16-lane groups already.
template <int TX, int TY, int S, int NT>
struct PairMap {
    using G = Geo<TX, TY, S>;
    static constexpr int WP = G::WO / 2, H = G::HOo;
    static constexpr int DENSE = WP * H, PADDED = (G::WI / 2) * H;
    static constexpr bool PAD = WP % 16 != 0 && (PADDED + NT - 1) / NT == (DENSE + NT - 1) / NT;
    static constexpr int VW = PAD ? G::WI / 2 : WP;
    static constexpr int SLOTS = VW * H;
    static constexpr int M = (SLOTS + NT - 1) / NT;  // passes
    // pair of slot g: column ax (doubles) and row by of the output region
    __device__ static void at(int g, int& ax, int& by)
    {
        g = min(g, SLOTS - 1);
        by = g / VW;
        ax = 2 * min(g % VW, WP - 1);
    }
    // its centre in the input plane (row stride WIN), and its place in the output plane
    template <int WIN = G::WI>
    __device__ static int centre(int g)
    {
        int ax, by;
        at(g, ax, by);
        return (by + 2) * WIN + ax + 2;
    }
    __device__ static int out(int g)
    {
        int ax, by;
        at(g, ax, by);
        return by * G::WO + ax;
    }
    // slot g is a pair of its own: not past the last slot, not a row's padding slot
    __device__ static bool live(int g) { return g < SLOTS && g % VW < WP; }
};

template <int TX, int TY, int S, int NT, int M, int R, int WI = Geo<TX, TY, S>::WI, typename T>
__device__ __forceinline__ void pair_step(const T* __restrict__ P, const StarW<T>& w, T (&acc)[M][2][4],
                                          T (&done)[M][2], typename V2<T>::type (&cen)[M])
{
    using v2 = typename V2<T>::type;
    constexpr int sm2 = (R + 2) & 3, sm1 = (R + 3) & 3, s0 = R & 3, sp1 = (R + 1) & 3;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const T* c = P + PairMap<TX, TY, S, NT>::template centre<WI>((int)threadIdx.x + m * NT);
        // x group first (centres and x neighbours), then the y group: at most 4 pairs of
        // loaded values are live at a time
        const v2 C = *(const v2*)c, Lx = *(const v2*)(c - 2), Rx = *(const v2*)(c + 2);
        cen[m] = C;
        T ax[2];
        {
            const T u[2] = {C.x, C.y};
            // x neighbours of the two columns: (Lx.x, Lx.y, C.y, Rx.x) and (Lx.y, C.x, Rx.x, Rx.y)
            const T xm2[2] = {Lx.x, Lx.y}, xm1[2] = {Lx.y, C.x}, xp1[2] = {C.y, Rx.x}, xp2[2] = {Rx.x, Rx.y};
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                done[m][e] = fmaT(w.zp2, u[e], acc[m][e][sm2]);
                acc[m][e][sm2] = w.zm2 * u[e];
                acc[m][e][sm1] = fmaT(w.zp1, u[e], acc[m][e][sm1]);
                acc[m][e][sp1] = fmaT(w.zm1, u[e], acc[m][e][sp1]);
                T a = fmaT(w.c, u[e], acc[m][e][s0]);
                a = fmaT(w.xm2, xm2[e], a);
                a = fmaT(w.xm1, xm1[e], a);
                a = fmaT(w.xp1, xp1[e], a);
                ax[e] = fmaT(w.xp2, xp2[e], a);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        {
            const v2 Ym2 = *(const v2*)(c - 2 * WI), Ym1 = *(const v2*)(c - WI);
            const v2 Yp1 = *(const v2*)(c + WI), Yp2 = *(const v2*)(c + 2 * WI);
            const T ym2[2] = {Ym2.x, Ym2.y}, ym1[2] = {Ym1.x, Ym1.y}, yp1[2] = {Yp1.x, Yp1.y},
                    yp2[2] = {Yp2.x, Yp2.y};
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                T a = w.ym2 * ym2[e];
                a = fmaT(w.ym1, ym1[e], a);
                a = fmaT(w.yp1, yp1[e], a);
                a = fmaT(w.yp2, yp2[e], a);
                acc[m][e][s0] = ax[e] + a;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Byte offsets (element size ES) of stage S's output pairs in a field (periodic images).
template <int TX, int TY, int S, int NT, int M, int ES = 8>
__device__ __forceinline__ void pair_offsets(int (&q)[M], int x0, int y0, int ni, int nj, int sj)
{
    using G = Geo<TX, TY, S>;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        int ax, by;
        PairMap<TX, TY, S, NT>::at((int)threadIdx.x + m * NT, ax, by);
        q[m] = (pmod(x0 - G::HO + ax, ni) + pmod(y0 - G::HO + by, nj) * sj) * ES;
    }
}

template <typename SI, int M, typename T>
__device__ __forceinline__ void pair_qload(T (&qv)[M], __amdgpu_buffer_rsrc_t r, int zo, const int (&q)[M])
{
#pragma unroll
    for (int m = 0; m < M; ++m) qv[m] = PairIO<SI, decltype(qv[m].x + 0)>::ld(r, q[m], zo);
}

// Index of pair g of stage S's output region inside a plane of region stage S+d
// (d = 0: the same region; d = 1: the next, smaller one, or `dump` when the pair lies in
// the halo that the next stage does not compute).
template <int TX, int TY, int S, int NT, int M>
__device__ __forceinline__ void pair_qidx(int (&same)[M], int (&next)[M])
{
    using G = Geo<TX, TY, S>;
    constexpr int WN = G::WO - 4, AN = WN * (G::HOo - 4);
#pragma unroll
    for (int m = 0; m < M; ++m) {
        int ax, by;
        PairMap<TX, TY, S, NT>::at((int)threadIdx.x + m * NT, ax, by);
        same[m] = by * G::WO + ax;
        const bool in = ax >= 2 && ax < G::WO - 2 && by >= 2 && by < G::HOo - 2;
        next[m] = in ? (by - 2) * WN + ax - 2 : AN;  // AN: a dump pair past the plane
    }
}

// RK4 step, two x-adjacent columns per lane: FP64 (SI = SO = T = double), or FP32 arithmetic
// over FP32 / BF16 storage (T = float; SI = double for a step from an FP64 input).  The
// arithmetic is the scalar kernel's for the same types, so both give the same bits.  The
// stage updates v_s = q + f_s L v_{s-1}
// need q at each stage's output plane, which lags the q plane being loaded by 2, 5, 8 and
// 11 planes.  Reloading it from global memory at those lags keeps a 12-plane window per
// block live in L2, more than an XCD's L2 holds for its resident blocks.  Instead:
//   stage 1 keeps the centre values of the q planes it reads from LDS (2-deep register
//     ring), stage 2 reloads q at lag 5 (a window the L2 holds), and writes it into an
//     LDS plane Q3 beside its output; stage 3 reads q from Q3 with its input plane, keeps
//     it 2 planes in registers and forwards it through Q4 to stage 4 the same way.
template <typename SI, typename SO, typename T, int TX, int TY, int NT>
__device__ __forceinline__ void rk4_pair_body(const FusedArgs& a, const int bid)
{
    using v2 = typename V2<T>::type;
    constexpr int ESI = sizeof(SI), ESO = sizeof(SO);
    using G1 = Geo<TX, TY, 1>;
    using G2 = Geo<TX, TY, 2>;
    using G3 = Geo<TX, TY, 3>;
    using G4 = Geo<TX, TY, 4>;
    constexpr int A0P = G1::AI / 2;  // pairs of the q plane incl. its 8-cell halo
    constexpr int M0 = (A0P + NT - 1) / NT;
    using PM1 = PairMap<TX, TY, 1, NT>;
    using PM2 = PairMap<TX, TY, 2, NT>;
    using PM3 = PairMap<TX, TY, 3, NT>;
    using PM4 = PairMap<TX, TY, 4, NT>;
    constexpr int M1 = PM1::M, M2 = PM2::M, M3 = PM3::M, M4 = PM4::M;

    __shared__ __attribute__((aligned(16))) T P0[2][G1::AI];
    __shared__ __attribute__((aligned(16))) T P1[2][G2::AI];
    __shared__ __attribute__((aligned(16))) T P2[2][G3::AI];
    __shared__ __attribute__((aligned(16))) T P3[2][G4::AI];
    __shared__ __attribute__((aligned(16))) T Q3[2][G3::AO + 2];  // q on stage 3's region
    __shared__ __attribute__((aligned(16))) T Q4[2][G4::AO + 2];  // q on stage 4's region

    const int tid = threadIdx.x;
    const int ni = a.ni, nj = a.nj, nk = a.nk;
    const int tile = bid % a.tiles;
    const int chunk = (bid / a.tiles) % a.chunks;
    const int slice = bid / (a.tiles * a.chunks);
    const int x0 = (tile % a.tiles_x) * TX, y0 = (tile / a.tiles_x) * TY;
    const int z0 = chunk * a.kchunk;
    const int zend = min(z0 + a.kchunk, nk);
    const __amdgpu_buffer_rsrc_t rin = make_rsrc((const SI*)a.in.p + slice * a.in.slice, a.in_bytes);
    const __amdgpu_buffer_rsrc_t rout = make_rsrc((SO*)a.out.p + slice * a.out.slice, a.out_bytes);
    const int iskb = (int)a.in.sk * ESI, oskb = (int)a.out.sk * ESO;
    const int isj = (int)a.in.sj, osj = (int)a.out.sj;
    const StarW<T> w = a.cdev ? load_w<T>(a.cdev[slice]) : load_w<T>(a.c);

    int off0[M0];
#pragma unroll
    for (int m = 0; m < M0; ++m) {
        const int g = min(tid + m * NT, A0P - 1);
        const int ax = 2 * (g % (G1::WI / 2)), by = g / (G1::WI / 2);
        off0[m] = (pmod(x0 - 8 + ax, ni) + pmod(y0 - 8 + by, nj) * isj) * ESI;
    }
    int q2[M2], o4[M4];
    pair_offsets<TX, TY, 2, NT, M2, ESI>(q2, x0, y0, ni, nj, isj);
#pragma unroll
    for (int m = 0; m < M4; ++m) {
        int ax, by;
        PM4::at(tid + m * NT, ax, by);
        o4[m] = (pmod(x0 + ax, ni) + pmod(y0 + by, nj) * osj) * ESO;  // periodic image for partial tiles
    }
    int s2[M2], w3[M2], r3x[M3], w4[M3], r4x[M4], n4[M4];
    // slots past a stage's last pair and the padding slots of padded rows repeat a pair:
    // they write nothing (several lanes writing one LDS address serialise).  The 32x32
    // tile has no registers left for the masks and writes the repeats.
    constexpr bool MASK = TX * TY <= 512;
    bool lv1[M1], lv2[M2], lv3[M3], lv4[M4];
    if constexpr (MASK) {
#pragma unroll
        for (int m = 0; m < M1; ++m) lv1[m] = PM1::live(tid + m * NT);
#pragma unroll
        for (int m = 0; m < M2; ++m) lv2[m] = PM2::live(tid + m * NT);
#pragma unroll
        for (int m = 0; m < M3; ++m) lv3[m] = PM3::live(tid + m * NT);
#pragma unroll
        for (int m = 0; m < M4; ++m) lv4[m] = PM4::live(tid + m * NT);
    }
    const auto wr0 = [&](int m) { return !MASK || m < M0 - 1 || tid + m * NT < A0P; };  // loader tail
    pair_qidx<TX, TY, 2, NT, M2>(s2, w3);
    pair_qidx<TX, TY, 3, NT, M3>(r3x, w4);
    pair_qidx<TX, TY, 4, NT, M4>(r4x, n4);

    T acc1[M1][2][4], acc2[M2][2][4], acc3[M3][2][4], acc4[M4][2][4];
    T d1[M1][2], d2v[M2][2], d3[M3][2], d4[M4][2];
    v2 qv2[M2];
    v2 c1[M1], c2[M2], c3[M3], c4[M4];                   // centres read this plane
    // q one and two planes back, in two-slot rings indexed by the plane's parity (R & 1 in
    // the unrolled loop): slot B holds the value stored two planes ago
    v2 r1[2][M1], r3[2][M3], r4[2][M4];
#pragma unroll
    for (int m = 0; m < M1; ++m) {
        r1[0][m] = r1[1][m] = v2{T(0), T(0)};
        for (int e = 0; e < 2; ++e) acc1[m][e][0] = acc1[m][e][1] = acc1[m][e][2] = acc1[m][e][3] = T(0);
    }
#pragma unroll
    for (int m = 0; m < M2; ++m)
        for (int e = 0; e < 2; ++e) acc2[m][e][0] = acc2[m][e][1] = acc2[m][e][2] = acc2[m][e][3] = T(0);
#pragma unroll
    for (int m = 0; m < M3; ++m) {
        r3[0][m] = r3[1][m] = v2{T(0), T(0)};
        for (int e = 0; e < 2; ++e) acc3[m][e][0] = acc3[m][e][1] = acc3[m][e][2] = acc3[m][e][3] = T(0);
    }
#pragma unroll
    for (int m = 0; m < M4; ++m) {
        r4[0][m] = r4[1][m] = v2{T(0), T(0)};
        for (int e = 0; e < 2; ++e) acc4[m][e][0] = acc4[m][e][1] = acc4[m][e][2] = acc4[m][e][3] = T(0);
    }

    // Same skewed schedule as k_rk4_fused: iteration t, stage 1: q t -> v1 t-2; stage 2:
    // v1 t-3 -> v2 t-5; stage 3: v2 t-6 -> v3 t-8; stage 4: v3 t-9 -> q' t-11.  Outputs
    // of a stage's first iterations are incomplete and never consumed by a later stage's
    // complete outputs (each stage starts when its first complete input plane exists).
    const int tq0 = z0 - 8, tq1 = zend + 8;
    const int tend = zend + 11;
    {
        const int zo = wrapz(tq0, nk) * iskb;
#pragma unroll
        for (int m = 0; m < M0; ++m)
            if (wr0(m)) *(v2*)&P0[tq0 & 1][2 * min(tid + m * NT, A0P - 1)] = PairIO<SI, T>::ld(rin, off0[m], zo);
        pair_qload<SI>(qv2, rin, wrapz(z0 - 8, nk) * iskb, q2);
    }
    v2 pre[M0];
    if (tq0 + 1 < tq1) {
        const int zo = wrapz(tq0 + 1, nk) * iskb;
#pragma unroll
        for (int m = 0; m < M0; ++m) pre[m] = PairIO<SI, T>::ld(rin, off0[m], zo);
    }
    __syncthreads();

    auto plane = [&](auto Rc, int t) {
        constexpr int R = decltype(Rc)::value;
        constexpr int B = R & 1;  // ring slot of this plane's parity
        const int cur = t & 1, prv = cur ^ 1;
        __builtin_amdgcn_sched_barrier(0);  // keep planes apart: bounded live ranges
        if (t + 1 < tq1) {
#pragma unroll
            for (int m = 0; m < M0; ++m)
                if (wr0(m)) *(v2*)&P0[prv][2 * min(tid + m * NT, A0P - 1)] = pre[m];
            if (t + 2 < tq1) {
                const int zo = wrapz(t + 2, nk) * iskb;
#pragma unroll
                for (int m = 0; m < M0; ++m) pre[m] = PairIO<SI, T>::ld(rin, off0[m], zo);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (t < tq1) {
            // centres of plane t are q(t); r1[B] = q(t-2) is the update's q
            pair_step<TX, TY, 1, NT, M1, R & 3>(P0[cur], w, acc1, d1, c1);
#pragma unroll
            for (int m = 0; m < M1; ++m) {
                if (!MASK || lv1[m])
                    *(v2*)&P1[cur][PM1::out(tid + m * NT)] =
                        v2{fmaT(w.f1, d1[m][0], r1[B][m].x), fmaT(w.f1, d1[m][1], r1[B][m].y)};
                r1[B][m] = c1[m];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (t >= tq0 + 5 && t < tq1 + 1) {
            pair_step<TX, TY, 2, NT, M2, (R + 1) & 3>(P1[prv], w, acc2, d2v, c2);
#pragma unroll
            for (int m = 0; m < M2; ++m) {
                if (!MASK || lv2[m]) {
                    *(v2*)&P2[cur][PM2::out(tid + m * NT)] =
                        v2{fmaT(w.f2, d2v[m][0], qv2[m].x), fmaT(w.f2, d2v[m][1], qv2[m].y)};
                    *(v2*)&Q3[cur][w3[m]] = qv2[m];  // q(t-5) for stage 3
                }
            }
            pair_qload<SI>(qv2, rin, wrapz(t - 4, nk) * iskb, q2);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (t >= tq0 + 10 && t < tq1 + 2) {
            pair_step<TX, TY, 3, NT, M3, (R + 2) & 3>(P2[prv], w, acc3, d3, c3);
#pragma unroll
            for (int m = 0; m < M3; ++m) {
                const v2 qn = *(const v2*)&Q3[prv][r3x[m]];  // q(t-6), written by stage 2 last plane
                if (!MASK || lv3[m]) {
                    *(v2*)&P3[cur][PM3::out(tid + m * NT)] =
                        v2{fmaT(w.f3, d3[m][0], r3[B][m].x), fmaT(w.f3, d3[m][1], r3[B][m].y)};
                    *(v2*)&Q4[cur][w4[m]] = r3[B][m];  // q(t-8) for stage 4
                }
                r3[B][m] = qn;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (t >= tq0 + 15) {
            pair_step<TX, TY, 4, NT, M4, (R + 3) & 3>(P3[prv], w, acc4, d4, c4);
            const int zp = t - 11;
            if (zp >= z0 && zp < zend) {
                const int zo = zp * oskb;
#pragma unroll
                for (int m = 0; m < M4; ++m)
                    if (!MASK || lv4[m])
                        PairIO<SO, T>::st(rout, o4[m], zo,
                                          v2{fmaT(w.f4, d4[m][0], r4[B][m].x), fmaT(w.f4, d4[m][1], r4[B][m].y)});
            }
#pragma unroll
            for (int m = 0; m < M4; ++m) r4[B][m] = *(const v2*)&Q4[prv][r4x[m]];  // q(t-9)
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };

    // Stage s runs while its input planes are valid.  The loop is unrolled by 4 so that
    // the phase R of every plane is a compile-time constant.
    for (int t = tq0; t < tend; t += 4) {
        plane(std::integral_constant<int, 0>{}, t);
        if (t + 1 < tend) plane(std::integral_constant<int, 1>{}, t + 1);
        if (t + 2 < tend) plane(std::integral_constant<int, 2>{}, t + 2);
        if (t + 3 < tend) plane(std::integral_constant<int, 3>{}, t + 3);
    }
}

// Waits for every outstanding vector-memory access of this wave (s_waitcnt vmcnt(0), the
// other counters left alone).  The compiler's own waits treat loads and stores as completing
// out of order, so with a store pending every use of a loaded register waits for all loads
// issued so far, the prefetches included; one explicit wait where all the data a stretch of
// planes consumes is known to have been requested lets the loads issued after it stay in flight.
__device__ __forceinline__ void vm_wait_all() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// ---- FP64 RK4 step in two launches of a two-stage kernel ----------------------------------
// The four-stage stream fills its pipeline with 19 planes per block.  A slice small enough to
// stay in the last-level cache (one 128^3 slice: 16.8 MB) is chunked in k to give every CU
// a block, and then a block streams 35 planes for 16 outputs, its stage-1 region 2.4x its
// tile.  Split in two launches, each block streams kchunk + 9 planes over the regions of
// stages 3 and 4 (tile + 4, tile):
//   launch A: u = q,  v_a = q + f1 L u,  out = q + f2 L v_a   (= v2, into a work field)
//   launch B: u = v2, v_a = q + f3 L u,  out = q + f4 L v_a   (= q')
// The work field adds one write and two reads of a field per step, cheap while the fields
// stay cached.  Each stage is pair_step with the same operands in the same order as in the
// four-stage kernel, so q' equals that kernel's bit for bit.
// Schedule, iteration t: stage a reads u plane t and emits v_a(t-2) into LDS; stage b reads
// v_a(t-3) and emits out(t-5).  q for the updates: in launch A stage a takes it from the
// centres it read two planes before; otherwise it is loaded from the q field.
struct HalfArgs {
    FusedArgs a;       // a.in: u; a.out: the output
    View q;            // the update base (launch A: the same field as a.in)
    unsigned q_bytes;  // bytes one slice of q spans from its origin
    int bricks;        // brick kernel: bricks of all slices, (2^32 - 1) over each divisor
    unsigned inv_tiles, inv_chunks, inv_tiles_x;
};

template <int TX, int TY, int NT, bool FIRST>
__device__ __forceinline__ void rk4_half_pair_body(const HalfArgs& h, const int bid)
{
    const FusedArgs& a = h.a;
    using G3 = Geo<TX, TY, 3>;
    constexpr int A0P = G3::AI / 2;  // pairs of the u plane incl. its 4-cell halo
    constexpr int M0 = (A0P + NT - 1) / NT;
    using PMa = PairMap<TX, TY, 3, NT>;
    using PMb = PairMap<TX, TY, 4, NT>;
    constexpr int Ma = PMa::M, Mb = PMb::M;

    __shared__ __attribute__((aligned(16))) double P0[2][G3::AI];
    __shared__ __attribute__((aligned(16))) double Pa[2][Geo<TX, TY, 4>::AI];

    const int tid = threadIdx.x;
    const int ni = a.ni, nj = a.nj, nk = a.nk;
    const int tile = bid % a.tiles;
    const int chunk = (bid / a.tiles) % a.chunks;
    const int slice = bid / (a.tiles * a.chunks);
    const int x0 = (tile % a.tiles_x) * TX, y0 = (tile / a.tiles_x) * TY;
    const int z0 = chunk * a.kchunk;
    const int zend = min(z0 + a.kchunk, nk);
    const __amdgpu_buffer_rsrc_t rin = make_rsrc((const double*)a.in.p + slice * a.in.slice, a.in_bytes);
    const __amdgpu_buffer_rsrc_t rq = make_rsrc((const double*)h.q.p + slice * h.q.slice, h.q_bytes);
    const __amdgpu_buffer_rsrc_t rout = make_rsrc((double*)a.out.p + slice * a.out.slice, a.out_bytes);
    const int iskb = (int)a.in.sk * 8, qskb = (int)h.q.sk * 8, oskb = (int)a.out.sk * 8;
    const int isj = (int)a.in.sj, qsj = (int)h.q.sj, osj = (int)a.out.sj;
    const StarW<double> w = a.cdev ? load_w<double>(a.cdev[slice]) : load_w<double>(a.c);
    const double fa = FIRST ? w.f1 : w.f3, fb = FIRST ? w.f2 : w.f4;

    int off0[M0];
#pragma unroll
    for (int m = 0; m < M0; ++m) {
        const int g = min(tid + m * NT, A0P - 1);
        const int ax = 2 * (g % (G3::WI / 2)), by = g / (G3::WI / 2);
        off0[m] = (pmod(x0 - 4 + ax, ni) + pmod(y0 - 4 + by, nj) * isj) * 8;
    }
    int qa[Ma], qb[Mb], ob[Mb];
    if constexpr (!FIRST) pair_offsets<TX, TY, 3, NT, Ma>(qa, x0, y0, ni, nj, qsj);
    pair_offsets<TX, TY, 4, NT, Mb>(qb, x0, y0, ni, nj, qsj);
#pragma unroll
    for (int m = 0; m < Mb; ++m) {
        int ax, by;
        PMb::at(tid + m * NT, ax, by);
        ob[m] = (pmod(x0 + ax, ni) + pmod(y0 + by, nj) * osj) * 8;  // periodic image for partial tiles
    }
    constexpr bool MASK = TX * TY <= 512;
    bool lva[Ma], lvb[Mb];
    if constexpr (MASK) {
#pragma unroll
        for (int m = 0; m < Ma; ++m) lva[m] = PMa::live(tid + m * NT);
#pragma unroll
        for (int m = 0; m < Mb; ++m) lvb[m] = PMb::live(tid + m * NT);
    }
    const auto wr0 = [&](int m) { return !MASK || m < M0 - 1 || tid + m * NT < A0P; };

    double acca[Ma][2][4], accb[Mb][2][4];
    double da[Ma][2], db[Mb][2];
    d2 ca[Ma], cb[Mb];
    // Global loads are issued four planes before use, in rings of four slots indexed by
    // (plane - tq0) & 3, and waited for once every four planes (vm_wait_all at phase 0):
    // everything a plane consumes was loaded before that wait, so no other wait stalls.
    d2 ra[2][Ma];     // launch A: q one and two planes back (ring by plane parity)
    d2 pre[4][M0];    // u planes t+1 .. t+4
    d2 qva[4][Ma];    // launch B: q planes t-2 .. t+1 for stage a
    d2 qvb[4][Mb];    // q planes t-5 .. t-2 for stage b
#pragma unroll
    for (int m = 0; m < Ma; ++m) {
        ra[0][m] = ra[1][m] = d2{0., 0.};
        for (int e = 0; e < 2; ++e) acca[m][e][0] = acca[m][e][1] = acca[m][e][2] = acca[m][e][3] = 0.;
    }
#pragma unroll
    for (int m = 0; m < Mb; ++m)
        for (int e = 0; e < 2; ++e) accb[m][e][0] = accb[m][e][1] = accb[m][e][2] = accb[m][e][3] = 0.;

    const int tq0 = z0 - 4, tq1 = zend + 4;  // u planes read: tq0 .. tq1 - 1
    const int tend = zend + 5;
    {
        const int zo = wrapz(tq0, nk) * iskb;
#pragma unroll
        for (int m = 0; m < M0; ++m)
            if (wr0(m)) *(d2*)&P0[tq0 & 1][2 * min(tid + m * NT, A0P - 1)] = ld2(rin, off0[m], zo);
#pragma unroll
        for (int j = 1; j <= 4; ++j) {
            const int zj = wrapz(tq0 + j, nk) * iskb;  // planes past tq1 - 1 are read and not used
#pragma unroll
            for (int m = 0; m < M0; ++m) pre[j & 3][m] = ld2(rin, off0[m], zj);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if constexpr (!FIRST) {
                const int za = wrapz(tq0 - 2 + j, nk) * qskb;
#pragma unroll
                for (int m = 0; m < Ma; ++m) qva[(j + 2) & 3][m] = ld2(rq, qa[m], za);
            }
            const int zb = wrapz(tq0 + j, nk) * qskb;  // first used at tq0 + 5
#pragma unroll
            for (int m = 0; m < Mb; ++m) qvb[j][m] = ld2(rq, qb[m], zb);
        }
    }
    __syncthreads();

    auto plane = [&](auto Rc, int t) {
        constexpr int R = decltype(Rc)::value;
        constexpr int B = R & 1;
        constexpr int S1 = (R + 1) & 3, SA = (R + 2) & 3, SB = (R + 3) & 3;  // slots of planes t+1, t-2, t-5
        const int cur = t & 1, prv = cur ^ 1;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (R == 0) vm_wait_all();
        if (t + 1 < tq1) {
#pragma unroll
            for (int m = 0; m < M0; ++m)
                if (wr0(m)) *(d2*)&P0[prv][2 * min(tid + m * NT, A0P - 1)] = pre[S1][m];
            if (t + 5 < tq1) {
                const int zo = wrapz(t + 5, nk) * iskb;
#pragma unroll
                for (int m = 0; m < M0; ++m) pre[S1][m] = ld2(rin, off0[m], zo);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (t < tq1) {
            pair_step<TX, TY, 3, NT, Ma, R & 3>(P0[cur], w, acca, da, ca);
#pragma unroll
            for (int m = 0; m < Ma; ++m) {
                const d2 q = FIRST ? ra[B][m] : qva[SA][m];
                if (!MASK || lva[m])
                    *(d2*)&Pa[cur][PMa::out(tid + m * NT)] = d2{fmaT(fa, da[m][0], q.x), fmaT(fa, da[m][1], q.y)};
                if constexpr (FIRST) ra[B][m] = ca[m];
            }
            if constexpr (!FIRST) {
                const int zo = wrapz(t + 2, nk) * qskb;
#pragma unroll
                for (int m = 0; m < Ma; ++m) qva[SA][m] = ld2(rq, qa[m], zo);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (t >= tq0 + 5) {
            pair_step<TX, TY, 4, NT, Mb, (R + 1) & 3>(Pa[prv], w, accb, db, cb);
            const int zp = t - 5;
            if (zp >= z0 && zp < zend) {
                const int zo = zp * oskb;
#pragma unroll
                for (int m = 0; m < Mb; ++m)
                    if (!MASK || lvb[m])
                        st2(rout, ob[m], zo,
                            d2{fmaT(fb, db[m][0], qvb[SB][m].x), fmaT(fb, db[m][1], qvb[SB][m].y)});
            }
            const int zo = wrapz(t - 1, nk) * qskb;
#pragma unroll
            for (int m = 0; m < Mb; ++m) qvb[SB][m] = ld2(rq, qb[m], zo);
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };

    for (int t = tq0; t < tend; t += 4) {
        plane(std::integral_constant<int, 0>{}, t);
        if (t + 1 < tend) plane(std::integral_constant<int, 1>{}, t + 1);
        if (t + 2 < tend) plane(std::integral_constant<int, 2>{}, t + 2);
        if (t + 3 < tend) plane(std::integral_constant<int, 3>{}, t + 3);
    }
}

// ---- FP64 2x2 variant (32x32 tiles, 12 waves) --------------------------------------------
// A lane owns one 2x2 block of columns (an x pair in two consecutive rows) in every stage it
// takes part in, and the four stages are divided between the waves:
//   waves 0-5, 7   stages 1 and 2      waves 8-11   stages 3 and 4
//   wave 6         stage 1 on its outermost ring and stage 3 on its ring
// Regions in blocks: stage 4 is the tile's 16x16 blocks; the star reaches one block (two
// cells) per stage along one axis only, so stage 3 needs those and the 64 blocks beside them
// (no corners), stage 2 68 more, stage 1 72 more: 460, 388, 320, 256 blocks.  The order
//   0-255 the tile, 256-319, 320-383, 384-447 the sides of rings 1-3, 448-459 the diagonals
//   (four of stage 2 first)
// gives every wave two stage steps per plane and every SIMD (waves w, w+4, w+8) six, against
// 7 for square regions with all stages in every wave.
// A lane's own values pass from stage to stage in registers: the centres of stages 2 and 4,
// and q at lags 2 and 4 (stages 1, 2; read once from LDS) and 7 and 10 (stages 3, 4; loaded
// once from global memory into a ring of four).  Of the sums, only the planes that have x and
// y terms still to come or z terms missing are kept; the first two z terms are taken from the
// centres when a plane's turn comes.  So 162 registers hold two stages, three waves per SIMD.
// What a plane costs (counted in the assembly): 120 VALU instructions per wave, all FP64, and
// per CU 218 ds_read_b128, 40 ds_write_b128 and 37 wave-wide global accesses.  Measured alone
// those are about 1600 cycles of VALU per SIMD, 1150 + 560 of LDS and 600 of the memory path;
// a plane takes about 2750, and the clock drops from 2.4 to 2.0-2.15 GHz under it, so the step
// is bound by VALU, LDS and power together, not by HBM.
// Reads are issued a part ahead of the arithmetic that uses them, and stage 1's x and y
// neighbours before the plane's barrier: the q planes sit in four buffers used in turn, so no
// one writes what those reads still fetch.  The q plane goes from global memory straight into
// LDS (buffer loads to LDS, 19 of one kilobyte each), two planes ahead; the buffer of a plane
// is fixed at compile time by its phase, so that no read waits for a load into another.
// Bank conflicts: see quad_lane; the strides W1 to W3 (4 mod 8) put the two rows of a write
// pass on different chunks.  Against the kernel this one replaced (8 waves, each with all four
// stages in 228 registers; 412 VALU instructions per SIMD and 304 reads per plane), on one box:
// 16 x 128^3 246 -> 199 us, 16 x 384^3 6320 -> 5150 us per step.  Measured and dropped: loads
// three planes ahead, the loads or the stores later in the plane, wave priorities by role (no
// change); reads in the order of consecutive lanes (+2 %); scheduling left to the compiler
// (+3 %); plain instead of non-temporal stores (+6 %).
struct QuadCfg {
    static constexpr int TX = 32, TY = 32;
    static constexpr int NT = 512;        // the tile descriptor's thread count (sp_prop_set_tile)
    static constexpr int WAVES = 12;      // the launch's waves
    static constexpr int W0 = 50, W1 = 44, W2 = 44, W3 = 36;  // strides of the planes q, v1, v2, v3
    static constexpr int H0 = 48, H1 = 44, H2 = 40, H3 = 36;  // their rows
    static constexpr int LOADS = (W0 / 2 * H0 + 63) / 64;     // wave loads of a q plane
};
static_assert(QuadCfg::W1 % 8 == 4 && QuadCfg::W2 % 8 == 4 && QuadCfg::W3 % 8 == 4,
              "two rows of a write pass on different chunks");
static_assert(QuadCfg::LOADS > 16 && QuadCfg::LOADS <= 19, "two loads by waves 0-7 and a third by waves 0-2");

// Lane l's place in the order above, within its wave.  The LDS serves a ds_read_b128 in four
// passes of 16 lanes, but not of 16 consecutive ones: lanes 0-3, 12-15, 20-23, 24-27 share a
// pass, then 4-7, 8-11, 16-19, 28-31, and the same in the upper half (measured: rows of 16
// consecutive lanes take 8.3 cycles per wave at strides of 50 chunks, this order 5.2 at any
// stride).  The places make every pass one group of 16 blocks.
__device__ __forceinline__ int quad_lane(int l) { return (l & 32) + ((0x73261540 >> (l & 28)) & 7) * 4 + (l & 3); }

// Block q of the order above, relative to the tile's first block.
__device__ __forceinline__ void quad_block(int q, int& bx, int& by)
{
    if (q < 256) {
        bx = q & 15;
        by = q >> 4;
    } else if (q < 448) {
        const int d = (q - 192) >> 6, g = ((q & 63) >> 4), i = q & 15;  // ring 1..3; above, below, two halves beside
        if (g < 2) {
            bx = i;
            by = g ? 15 + d : -d;
        } else {
            bx = i < 8 ? -d : 15 + d;
            by = 8 * (g - 2) + (i & 7);
        }
    } else {
        const int i = min(q - 448, 11);  // lanes past the last block repeat it (and write nothing)
        if (i < 4) {
            bx = i & 1 ? 16 : -1;
            by = i & 2 ? 16 : -1;
        } else {
            const int j = i - 4, far = j & 1;  // one of (-2, -1), (-1, -2) mirrored to each corner
            const int ax = far ? 1 : 2, ay = far ? 2 : 1;
            bx = j & 2 ? 15 + ax : -ax;
            by = j & 4 ? 15 + ay : -ay;
        }
    }
}

// One stage on a 2x2 block, in parts, so that the reads of one part are in flight during the
// arithmetic of another.  a: the running sums of one plane's four points, point 2 f + e in row f,
// column e; c: the block's first centre in an LDS plane (row stride W); u: a plane's centres.
// A point's terms come in the order z-2, z-1, centre, x, y, z+1, z+2.

__device__ __forceinline__ void quad_fence() { __builtin_amdgcn_sched_barrier(0); }
// Holds the arithmetic on a there: without it the compiler moves reads past arithmetic, which
// carries no order of its own, and the values in flight no longer fit the registers.
__device__ __forceinline__ void quad_hold(double (&a)[4])
{
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]));
    __builtin_amdgcn_sched_barrier(0);
}
// starts the sums of plane p with the centres of planes p-2 and p-1
__device__ __forceinline__ void quad_start(double (&a)[4], const StarW<double>& w, const d2 (&um2)[2],
                                           const d2 (&um1)[2])
{
#pragma unroll
    for (int f = 0; f < 2; ++f) {
        a[2 * f] = fmaT(w.zm1, um1[f].x, w.zm2 * um2[f].x);
        a[2 * f + 1] = fmaT(w.zm1, um1[f].y, w.zm2 * um2[f].y);
    }
}
template <int W>
__device__ __forceinline__ void quad_read_c(const double* __restrict__ c, d2 (&u)[2])
{
    u[0] = *(const d2*)c;
    u[1] = *(const d2*)(c + W);
}
// centre and x neighbours (the pairs beside the block's two rows)
template <int W>
__device__ __forceinline__ void quad_read_x(const double* __restrict__ c, d2 (&x)[4])
{
#pragma unroll
    for (int f = 0; f < 2; ++f) {
        x[2 * f] = *(const d2*)(c + f * W - 2);
        x[2 * f + 1] = *(const d2*)(c + f * W + 2);
    }
}
template <bool HOLD = true>
__device__ __forceinline__ void quad_x(double (&a)[4], const StarW<double>& w, const d2 (&u)[2], const d2 (&x)[4])
{
#pragma unroll
    for (int f = 0; f < 2; ++f) {
        const d2 C = u[f], Lx = x[2 * f], Rx = x[2 * f + 1];
        const double c[2] = {C.x, C.y};
        const double xm2[2] = {Lx.x, Lx.y}, xm1[2] = {Lx.y, C.x}, xp1[2] = {C.y, Rx.x}, xp2[2] = {Rx.x, Rx.y};
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            double s = fmaT(w.c, c[e], a[2 * f + e]);
            s = fmaT(w.xm2, xm2[e], s);
            s = fmaT(w.xm1, xm1[e], s);
            s = fmaT(w.xp1, xp1[e], s);
            a[2 * f + e] = fmaT(w.xp2, xp2[e], s);
        }
    }
    if constexpr (HOLD) quad_hold(a);
}
// y neighbours: rows y-2, y-1, y+2, y+3 (the block's own rows are the centres)
template <int W>
__device__ __forceinline__ void quad_read_y(const double* __restrict__ c, d2 (&y)[4])
{
    y[0] = *(const d2*)(c - 2 * W);
    y[1] = *(const d2*)(c - W);
    y[2] = *(const d2*)(c + 2 * W);
    y[3] = *(const d2*)(c + 3 * W);
}
template <bool HOLD = true>
__device__ __forceinline__ void quad_y(double (&a)[4], const StarW<double>& w, const d2 (&u)[2], const d2 (&y)[4])
{
    const double r[6][2] = {{y[0].x, y[0].y}, {y[1].x, y[1].y}, {u[0].x, u[0].y},
                            {u[1].x, u[1].y}, {y[2].x, y[2].y}, {y[3].x, y[3].y}};
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            // row y+f: neighbours at rows (y+f) -2, -1, +1, +2 = r[f], r[f+1], r[f+3], r[f+4]
            double s = w.ym2 * r[f][e];
            s = fmaT(w.ym1, r[f + 1][e], s);
            s = fmaT(w.yp1, r[f + 3][e], s);
            s = fmaT(w.yp2, r[f + 4][e], s);
            a[2 * f + e] += s;
        }
    if constexpr (HOLD) quad_hold(a);
}
// adds the centres of plane p+1
template <bool HOLD = true>
__device__ __forceinline__ void quad_next(double (&a)[4], const StarW<double>& w, const d2 (&u)[2])
{
#pragma unroll
    for (int f = 0; f < 2; ++f) {
        a[2 * f] = fmaT(w.zp1, u[f].x, a[2 * f]);
        a[2 * f + 1] = fmaT(w.zp1, u[f].y, a[2 * f + 1]);
    }
    if constexpr (HOLD) quad_hold(a);
}
// adds the centres of plane p+2 and gives the stage's result q + f * sum
__device__ __forceinline__ void quad_done(d2 (&v)[2], double f, const double (&a)[4], const StarW<double>& w,
                                          const d2 (&u)[2], const d2 (&q)[2])
{
#pragma unroll
    for (int r = 0; r < 2; ++r)
        v[r] = d2{fmaT(f, fmaT(w.zp2, u[r].x, a[2 * r]), q[r].x), fmaT(f, fmaT(w.zp2, u[r].y, a[2 * r + 1]), q[r].y)};
}

template <int W>
__device__ __forceinline__ void quad_write(double* c, const d2 (&v)[2])
{
    *(d2*)c = v[0];
    *(d2*)(c + W) = v[1];
}

template <int N>
__device__ __forceinline__ void quad_zero(double (&acc)[N][4])
{
#pragma unroll
    for (int j = 0; j < N; ++j) acc[j][0] = acc[j][1] = acc[j][2] = acc[j][3] = 0.;
}

__device__ __forceinline__ void rk4_quad_body(const FusedArgs& a, const int bid)
{
    using Q = QuadCfg;
    constexpr int W0 = Q::W0, W1 = Q::W1, W2 = Q::W2, W3 = Q::W3;
    // one array per buffer: reads of one never alias the loads into another
    __shared__ __attribute__((aligned(16))) double P0a[Q::H0 * W0];
    __shared__ __attribute__((aligned(16))) double P0b[Q::H0 * W0];
    __shared__ __attribute__((aligned(16))) double P0c[Q::H0 * W0];
    __shared__ __attribute__((aligned(16))) double P0d[Q::H0 * W0];
    __shared__ __attribute__((aligned(16))) double P1[2][Q::H1 * W1];
    __shared__ __attribute__((aligned(16))) double P2[2][Q::H2 * W2];
    __shared__ __attribute__((aligned(16))) double P3[2][Q::H3 * W3];
    const auto P0 = [&](auto Rc) -> double* {
        constexpr int R = decltype(Rc)::value & 3;
        if constexpr (R == 0) return P0a;
        else if constexpr (R == 1) return P0b;
        else if constexpr (R == 2) return P0c;
        else return P0d;
    };

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int v = quad_lane(lane);
    const int ni = a.ni, nj = a.nj, nk = a.nk;
    const int tile = bid % a.tiles;
    const int chunk = (bid / a.tiles) % a.chunks;
    const int slice = bid / (a.tiles * a.chunks);
    const int x0 = (tile % a.tiles_x) * Q::TX, y0 = (tile / a.tiles_x) * Q::TY;
    const int z0 = chunk * a.kchunk;
    const int zend = min(z0 + a.kchunk, nk);
    const __amdgpu_buffer_rsrc_t rin = make_rsrc((const double*)a.in.p + slice * a.in.slice, a.in_bytes);
    const __amdgpu_buffer_rsrc_t rout = make_rsrc((double*)a.out.p + slice * a.out.slice, a.out_bytes);
    const int iskb = (int)a.in.sk * 8, oskb = (int)a.out.sk * 8;
    const int isj = (int)a.in.sj, osj = (int)a.out.sj;
    const StarW<double> w = a.cdev ? load_w<double>(a.cdev[slice]) : load_w<double>(a.c);

    // Iteration t: stage 1's z sums take q(t) and complete v1(t-2), its x and y sums q(t-1),
    // whose neighbours were read at the end of iteration t-1; stage 2's z sums take v1(t-2) at
    // once and complete v2(t-4), its x and y sums v1(t-3), written in iteration t-1; stage 3
    // takes v2(t-5) and completes v3(t-7); stage 4 takes v3(t-8) and completes q'(t-10).  Every
    // stage runs in every iteration: its first outputs are incomplete and no complete output
    // reads them.
    const int tq0 = z0 - 8, tend = zend + 10;

    // Loads of a q plane: load m of wave w fills slots 512 m + 64 w .. + 63 of 16 bytes; slot g
    // is column pair g % 25 of row g / 25 (the 25th pair is padding).
    int off0[3];
    const auto load_offsets = [&] {
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const int g = min(m * 512 + wave * 64 + lane, W0 / 2 * Q::H0 - 1);
            const int col = g % (W0 / 2), row = g / (W0 / 2);
            off0[m] = (pmod(x0 - 8 + 2 * col, ni) + pmod(y0 - 8 + row, nj) * isj) * 8;
        }
    };
    const bool third = wave < Q::LOADS - 16, tail = 1024 + wave * 64 + lane < W0 / 2 * Q::H0;
    const auto load_q = [&](double* P, int p) {  // q plane p
        const int zo = wrapz(p, nk) * iskb;
        ld2_to_lds(rin, P + 2 * (wave * 64), off0[0], zo);
        ld2_to_lds(rin, P + 2 * (512 + wave * 64), off0[1], zo);
        if (third) {
            if (tail) ld2_to_lds(rin, P + 2 * (1024 + wave * 64), off0[2], zo);
        }
    };
    // before the barrier of a plane: this wave's loads of the previous plane have landed, the
    // ones of this plane may be in flight
    const auto wait_q = [&] {
        if (third) vm_wait<3>();
        else vm_wait<2>();
    };
    using std::integral_constant;
    // Whole groups of four planes, so that a plane's phase is known at compile time and the
    // loop has no exits inside; the planes past tend store nothing.
    const auto stream = [&](auto&& plane) {
        lds_barrier();
        for (int t = tq0; t < tend; t += 4) {
            plane(integral_constant<int, 0>{}, t);
            plane(integral_constant<int, 1>{}, t + 1);
            plane(integral_constant<int, 2>{}, t + 2);
            plane(integral_constant<int, 3>{}, t + 3);
        }
    };

    if (wave < 6 || wave == 7) {
        // ---- stages 1 and 2
        const int q = wave < 6 ? wave * 64 + v : 448 + v;
        int bx, by;
        quad_block(q, bx, by);
        const int i0 = (2 * by + 8) * W0 + 2 * bx + 8;
        const int i1 = (2 * by + 6) * W1 + 2 * bx + 6;
        const int i2 = (2 * by + 4) * W2 + 2 * bx + 4;
        // wave 7: lanes without a block in a stage write nothing
        const bool live1 = q < 460, live2 = q < 452;
        load_offsets();
        // running sums by plane phase: stage 1's of two planes, stage 2's of three
        double a1[4][4], a2[4][4];
        d2 uc[2], qr[4][2];  // v1 of this block; q at lags 1-4 by plane phase
        d2 x[4], y[4];
        quad_zero(a1);
        quad_zero(a2);
#pragma unroll
        for (int f = 0; f < 2; ++f) uc[f] = qr[0][f] = qr[1][f] = qr[2][f] = qr[3][f] = d2{0., 0.};
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = y[i] = d2{0., 0.};
        load_q(P0a, tq0);
        load_q(P0b, tq0 + 1);
        vm_wait<0>();
        stream([&](auto Rc, int t) {
            constexpr int R = decltype(Rc)::value, cur = R & 1, prv = cur ^ 1;
            constexpr int R1 = (R + 3) & 3, R2 = (R + 2) & 3, R3 = (R + 1) & 3;  // phases of planes t-1, t-2, t-3
            load_q(P0(integral_constant<int, R + 2>{}), t + 2);
            const double *const c0 = P0(Rc) + i0, *const c1 = &P1[prv][i1];
            d2 qc[2], un[2], v2[2];
            quad_read_c<W0>(c0, qc);
            quad_start(a1[R1], w, qr[R3], qr[R2]);
            quad_x(a1[R1], w, qr[R1], x);
            quad_read_x<W1>(c1, x);
            quad_fence();
            quad_y(a1[R1], w, qr[R1], y);
            quad_read_y<W1>(c1, y);
            quad_fence();
            quad_x(a2[R3], w, uc, x);
            quad_y(a2[R3], w, uc, y);
            quad_done(un, w.f1, a1[R2], w, qc, qr[R2]);
            if (live1) quad_write<W1>(&P1[cur][i1], un);
            quad_fence();
            quad_done(v2, w.f2, a2[R], w, un, qr[R]);
            if (live2) quad_write<W2>(&P2[cur][i2], v2);
            quad_fence();
            quad_read_x<W0>(c0, x);
            quad_read_y<W0>(c0, y);
            quad_fence();
            quad_next(a1[R1], w, qc);
            quad_next(a2[R3], w, un);
            quad_start(a2[R1], w, uc, un);
            quad_hold(a2[R1]);
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                uc[f] = un[f];
                qr[R][f] = qc[f];
            }
            wait_q();
            lds_barrier<8>();
        });
        vm_wait<0>();  // no load into LDS outlives the block
    } else if (wave == 6) {
        // ---- stage 1 on ring 3, stage 3 on ring 1
        int bx, by, cx, cy;
        quad_block(384 + v, bx, by);
        quad_block(256 + v, cx, cy);
        const int i0 = (2 * by + 8) * W0 + 2 * bx + 8;
        const int i1 = (2 * by + 6) * W1 + 2 * bx + 6;
        const int i2 = (2 * cy + 4) * W2 + 2 * cx + 4;
        const int i3 = (2 * cy + 2) * W3 + 2 * cx + 2;
        int q3[2];
#pragma unroll
        for (int f = 0; f < 2; ++f) q3[f] = (pmod(x0 + 2 * cx, ni) + pmod(y0 + 2 * cy + f, nj) * isj) * 8;
        load_offsets();
        double a1[4][4], a3[4][4];
        d2 qr[4][2], vp[2], qe[2], qo[2];  // q at lags 1-4 by plane phase, v2 of the last plane, q at lags 7 and 6
        d2 x[4], y[4];
        quad_zero(a1);
        quad_zero(a3);
        vp[0] = vp[1] = qe[0] = qe[1] = qo[0] = qo[1] = d2{0., 0.};
#pragma unroll
        for (int f = 0; f < 2; ++f) qr[0][f] = qr[1][f] = qr[2][f] = qr[3][f] = d2{0., 0.};
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = y[i] = d2{0., 0.};
        load_q(P0a, tq0);
        load_q(P0b, tq0 + 1);
        vm_wait<0>();
        stream([&](auto Rc, int t) {
            constexpr int R = decltype(Rc)::value, cur = R & 1, prv = cur ^ 1;
            constexpr int R1 = (R + 3) & 3, R2 = (R + 2) & 3, R3 = (R + 1) & 3;
            load_q(P0(integral_constant<int, R + 2>{}), t + 2);
            const double *const c0 = P0(Rc) + i0, *const c2 = &P2[prv][i2];
            d2(&qv)[2] = R & 1 ? qo : qe;  // q(t-7)
            d2 qc[2], vc[2], v1[2], v3[2];
            quad_read_c<W0>(c0, qc);
            quad_read_c<W2>(c2, vc);
            quad_start(a1[R1], w, qr[R3], qr[R2]);
            quad_x(a1[R1], w, qr[R1], x);
            quad_read_x<W2>(c2, x);
            quad_fence();
            quad_y(a1[R1], w, qr[R1], y);
            quad_read_y<W2>(c2, y);
            quad_fence();
            quad_done(v1, w.f1, a1[R2], w, qc, qr[R2]);
            quad_write<W1>(&P1[cur][i1], v1);
            quad_fence();
            // plane t-5: its phase is R1, t-6's R2, t-7's R3
            quad_done(v3, w.f3, a3[R3], w, vc, qv);
            quad_write<W3>(&P3[cur][i3], v3);
            quad_fence();
            {
                const int zo = wrapz(t - 5, nk) * iskb;  // q(t-5): stage 3's q two planes on
#pragma unroll
                for (int f = 0; f < 2; ++f) qv[f] = ld2(rin, q3[f], zo);
            }
            quad_next(a3[R2], w, vc);
            quad_x(a3[R1], w, vc, x);
            quad_y(a3[R1], w, vc, y);
            quad_read_x<W0>(c0, x);
            quad_read_y<W0>(c0, y);
            quad_fence();
            quad_next(a1[R1], w, qc);
            quad_start(a3[R], w, vp, vc);
            quad_hold(a3[R]);
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                vp[f] = vc[f];
                qr[R][f] = qc[f];
            }
            vm_wait<6>();  // two loads of a q plane and two of q since the last plane's
            lds_barrier<8>();
        });
        vm_wait<0>();
    } else {
        // ---- stages 3 and 4
        int bx, by;
        quad_block((wave - 8) * 64 + v, bx, by);
        const int i2 = (2 * by + 4) * W2 + 2 * bx + 4;
        const int i3 = (2 * by + 2) * W3 + 2 * bx + 2;
        int q3[2], o4[2];
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            const int gx = pmod(x0 + 2 * bx, ni), gy = pmod(y0 + 2 * by + f, nj);  // periodic image for partial tiles
            q3[f] = (gx + gy * isj) * 8;
            o4[f] = (gx + gy * osj) * 8;
        }
        double a3[4][4], a4[4][4];
        d2 yc[2], yp[2], vp[2], qr[4][2];  // v3 of this block and the plane before, v2 before; q at lags 7-10
        quad_zero(a3);
        quad_zero(a4);
#pragma unroll
        for (int f = 0; f < 2; ++f) yc[f] = yp[f] = vp[f] = qr[0][f] = qr[1][f] = qr[2][f] = qr[3][f] = d2{0., 0.};
        stream([&](auto Rc, int t) {
            constexpr int R = decltype(Rc)::value, cur = R & 1, prv = cur ^ 1;
            constexpr int R1 = (R + 3) & 3, R2 = (R + 2) & 3, R3 = (R + 1) & 3;
            const double *const c2 = &P2[prv][i2], *const c3 = &P3[prv][i3];
            d2 vc[2], x[4], y[4], qn[2];
            quad_read_x<W3>(c3, x);
            quad_read_y<W3>(c3, y);
            quad_fence();
            // stage 4 at plane t-8 (phase R; t-9's R1, t-10's R2): the stores outside z0 to zend
            // go past the field's end and are dropped (issued all the same, so that waits count
            // loads and stores exactly)
            const bool st = t >= tq0 + 18 && t < tend;
            const int zo = st ? (t - 10) * oskb : 0;
            quad_done(qn, w.f4, a4[R2], w, yc, qr[R2]);
#pragma unroll
            for (int f = 0; f < 2; ++f) st2_stream(rout, st ? o4[f] : (int)0x80000000, zo, qn[f]);
            {
                const int zq = wrapz(t - 6, nk) * iskb;  // q(t-6): stage 3's q at the next plane
#pragma unroll
                for (int f = 0; f < 2; ++f) qr[R2][f] = ld2_last(rin, q3[f], zq);
            }
            quad_fence();
            quad_next(a4[R1], w, yc);
            quad_x(a4[R], w, yc, x);
            quad_read_c<W2>(c2, vc);
            quad_read_x<W2>(c2, x);
            quad_fence();
            quad_y(a4[R], w, yc, y);
            quad_read_y<W2>(c2, y);
            quad_fence();
            quad_start(a4[R3], w, yp, yc);
            quad_hold(a4[R3]);
#pragma unroll
            for (int f = 0; f < 2; ++f) yp[f] = yc[f];
            // stage 3 at plane t-5 (phase R1; t-6's R2, t-7's R3)
            quad_done(yc, w.f3, a3[R3], w, vc, qr[R3]);
            quad_write<W3>(&P3[cur][i3], yc);
            quad_fence();
            quad_next(a3[R2], w, vc);
            quad_x(a3[R1], w, vc, x);
            quad_y(a3[R1], w, vc, y);
            quad_start(a3[R], w, vp, vc);
            quad_hold(a3[R]);
#pragma unroll
            for (int f = 0; f < 2; ++f) vp[f] = vc[f];
            lds_barrier();
        });
    }
}

// ---- FP64 step of small fields: bricks, two launches of two stages ---------------------------
// A small field has too few tiles to fill the chip, and a chunk's walk along k is bound by one
// plane's latency (0.5-1.2 us) times its planes, most of which fill the pipeline.  Here nothing
// walks: a block loads the whole input of a 16x16x8 brick of results at once (24x24x16 cells,
// 74 KB of LDS), computes one stage on the cells that the next one reads (the brick's 64 2x2
// columns over 12 planes and the 32 columns around it over 8: two planes per lane of eight
// waves), puts the result over the input in LDS and computes the next stage.  A block takes
// several bricks in turn where there are more than CUs: two more waves load the next one into a
// second buffer meanwhile.  Four stages take two launches through the split step's work field:
//   launch A: u = q,  v_a = q + f1 L u,  out = q + f2 L v_a   (= v2)
//   launch B: u = v2, v_a = q + f3 L u,  out = q + f4 L v_a   (= q')
// with the other kernels' operations in the same order (the same bits).  Any sizes, strides and
// alignment: PAIR loads and stores 16 bytes, otherwise each cell's two words are loaded by
// lanes of their own.  Eight columns per row and a row pair of 24 chunks of 16 bytes (8 mod 16)
// put consecutive lanes on consecutive chunks across rows: no bank conflicts.
// Bound by latency up to 256 bricks (64^3 13.0 us a step), then by no one part alone: 128^3, 1024
// bricks, took 32.4 us, without its loads 32.6, without its stores 27 (30.5 since these go
// through), without the two stages 28, without all of them 18.  One brick per block on six waves,
// loads not overlapped: 64^3 13.9 us, 128^3 42.0, 127^3 52.4 against 40.4, 8 x 64^3 40.3 against 29.5.
struct BrickCfg {
    static constexpr int BX = 16, BY = 16, BZ = 8, NT = 384;  // NT: the descriptor's only
    static constexpr int W = 24, H = 24, D = 16, PLANE = W * H, CELLS = D * PLANE;  // the input's cells in LDS
    static constexpr int WAVES = 8, THREADS = (WAVES + 2) * 64;                     // the last two load
};

// The base values q of a lane's 2x2 block in N planes, from global memory.
template <bool PAIR>
struct BrickCols {
    int o[2][PAIR ? 1 : 2];  // byte offsets of the block's rows (and columns, if not PAIR)
    __device__ __forceinline__ void set(int x, int y, int ni, int nj, int sj)
    {
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int e = 0; e < (PAIR ? 1 : 2); ++e) o[f][e] = (near_mod(x + e, ni) + near_mod(y + f, nj) * sj) * 8;
    }
    __device__ __forceinline__ d2 ld(__amdgpu_buffer_rsrc_t r, int f, int zo) const
    {
        if constexpr (PAIR) return ld2(r, o[f][0], zo);
        else return d2{Buf<double>::ld(r, o[f][0], zo), Buf<double>::ld(r, o[f][1], zo)};
    }
    // zo of the lane's own
    __device__ __forceinline__ d2 ld_lane(__amdgpu_buffer_rsrc_t r, int f, int zo) const
    {
        if constexpr (PAIR) return ld2(r, o[f][0] + zo, 0);
        else return d2{Buf<double>::ld(r, o[f][0] + zo, 0), Buf<double>::ld(r, o[f][1] + zo, 0)};
    }
    __device__ __forceinline__ void st(__amdgpu_buffer_rsrc_t r, int f, int zo, d2 v) const
    {
        if constexpr (PAIR) {
            st_through(r, o[f][0], zo, v);
        } else {
            Buf<double>::st(r, o[f][0], zo, v.x);  // halves of lines: 10 % slower stored through
            Buf<double>::st(r, o[f][1], zo, v.y);
        }
    }
};

// One stage of a block's column at N consecutive planes; c: its first centre two planes below.
template <int N>
__device__ __forceinline__ void brick_stage(d2 (&v)[N][2], const double* __restrict__ c, const StarW<double>& w,
                                            double f, const d2 (*q)[2])
{
    using B = BrickCfg;
    d2 u[N + 4][2];
#pragma unroll
    for (int k = 0; k < N + 4; ++k) quad_read_c<B::W>(c + k * B::PLANE, u[k]);
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const double* p = c + (j + 2) * B::PLANE;
        d2 x[4], y[4];
        double a[4];
        quad_read_x<B::W>(p, x);
        quad_read_y<B::W>(p, y);
        quad_start(a, w, u[j], u[j + 1]);
        quad_x<false>(a, w, u[j + 2], x);
        quad_y<false>(a, w, u[j + 2], y);
        quad_next<false>(a, w, u[j + 3]);
        quad_done(v[j], f, a, w, u[j + 4], q ? q[j] : u[j + 2]);
    }
}

// A brick's input, with periodic images, straight into LDS in the order of its cells: two planes
// are nine whole wave loads of 16-byte slots (part 4 is half of each plane) or, where rows are
// not 16-byte aligned pairs, a plane 18 of single words.  What bounds this is the instructions
// around a load: masked loads and a general wrap of each plane's index took 50 of them, and 3000
// cycles for a brick; the byte offset of a plane steps with three.
template <bool PAIR>
struct BrickLoads {
    static constexpr int W = BrickCfg::W, PLANE = BrickCfg::PLANE, N = PAIR ? 9 : 18;
    static_assert(2 * PLANE / 2 == 9 * 64 && PLANE * 2 == 18 * 64, "whole wave loads");
    // part t's cell: byte offset in its plane
    static __device__ __forceinline__ int offset(int t, int lane, int sj, int x, int y, int ni, int nj)
    {
        const int e = PAIR ? (2 * (t * 64 + lane)) % PLANE : t * 32 + (lane >> 1);
        return (near_mod(x + e % W, ni) + near_mod(y + e / W, nj) * sj) * 8 + (PAIR ? 0 : (lane & 1) * 4);
    }
    // part t of the plane pair at dst, planes at byte offsets z0 and z1
    static __device__ __forceinline__ void load(double* dst, int t, int off, __amdgpu_buffer_rsrc_t r, int z0, int z1,
                                                int lane)
    {
        if constexpr (PAIR) {
            if (t == 4) ld2_to_lds(r, dst + t * 128, off + (lane < 32 ? z0 : z1), 0);
            else ld2_to_lds(r, dst + t * 128, off, t < 4 ? z0 : z1);
        } else {
            ldw_to_lds(r, dst + t * 32, off, z0);
            ldw_to_lds(r, dst + PLANE + t * 32, off, z1);
        }
    }
};

template <bool FIRST, bool PAIR>
__device__ __forceinline__ void rk4_brick_body(const HalfArgs& h)
{
    using B = BrickCfg;
    const FusedArgs& a = h.a;
    __shared__ __attribute__((aligned(16))) double P[2 * B::CELLS];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ni = a.ni, nj = a.nj, nk = a.nk;
    const int iskb = (int)a.in.sk * 8, isj = (int)a.in.sj, qskb = (int)h.q.sk * 8, oskb = (int)a.out.sk * 8;

    // this block's bricks: every step-th of its XCD's contiguous range
    const int xcd = blockIdx.x % 8, extra = h.bricks % 8;
    const int step = ((int)gridDim.x + 7 - xcd) / 8;
    const int first = xcd * (h.bricks / 8) + min(xcd, extra), last = first + h.bricks / 8 + (xcd < extra ? 1 : 0);
    int b = first + (int)blockIdx.x / 8;
    if (b >= last) return;

    int slice, x0, y0, z0;
    const auto divide = [](int n, int d, unsigned inv, int& rest) {  // inv: (2^32 - 1) / d
        int v = (int)__umulhi((unsigned)n, inv);
        rest = n - v * d;
        if (rest >= d) ++v, rest -= d;
        return v;
    };
    const auto place = [&](int n) {
        int tile, chunk, tx;
        slice = divide(divide(n, a.tiles, h.inv_tiles, tile), a.chunks, h.inv_chunks, chunk);
        y0 = divide(tile, a.tiles_x, h.inv_tiles_x, tx) * B::BY;
        x0 = tx * B::BX;
        z0 = chunk * B::BZ;
    };
    const auto input = [&]() { return make_rsrc((const double*)a.in.p + slice * a.in.slice, a.in_bytes); };
    place(b);
    using L = BrickLoads<PAIR>;
    const unsigned span = (unsigned)nk * iskb;
    {
        const __amdgpu_buffer_rsrc_t r = input();
        unsigned z = wrapz(z0 - 4, nk) * iskb;
        if constexpr (PAIR) {
            // a part per wave
            if (wave < L::N) {
                const int off = L::offset(wave, lane, isj, x0 - 4, y0 - 4, ni, nj);
                z = wave * 64 + lane < B::PLANE / 2 ? z : plane_step(z, iskb, span);
#pragma unroll
                for (int u = 0; u < B::D / 2; ++u) {
                    ld2_to_lds(r, P + 2 * u * B::PLANE + wave * 128, off + z, 0);
                    z = plane_step(z, 2 * iskb, span);
                }
            }
        } else if (wave < L::N / 2) {
            const int off0 = L::offset(2 * wave, lane, isj, x0 - 4, y0 - 4, ni, nj);
            const int off1 = L::offset(2 * wave + 1, lane, isj, x0 - 4, y0 - 4, ni, nj);
#pragma unroll
            for (int p = 0; p < B::D; ++p) {
                ldw_to_lds(r, P + p * B::PLANE + wave * 64, off0, z);
                ldw_to_lds(r, P + p * B::PLANE + wave * 64 + 32, off1, z);
                z = plane_step(z, iskb, span);
            }
        }
        vm_wait<0>();
    }

    if (wave >= B::WAVES) {
        // the next brick's plane pairs into the other buffer, alternating between the two waves
        double* dst = P + B::CELLS;
        for (;;) {
            const bool more = b + step < last;
            if (more) place(b + step);
            const __amdgpu_buffer_rsrc_t r = input();
            int off[L::N];
#pragma unroll
            for (int t = 0; t < L::N; ++t) off[t] = L::offset(t, lane, isj, x0 - 4, y0 - 4, ni, nj);
            unsigned z = wrapz(z0 - 4 + 2 * (wave - B::WAVES), nk) * iskb;
            double* d = dst + 2 * (wave - B::WAVES) * B::PLANE;
            const auto pairs = [&](int n) {
                if (more)
                    for (int u = 0; u < n; ++u) {
                        const unsigned z1 = plane_step(z, iskb, span);
#pragma unroll
                        for (int t = 0; t < L::N; ++t) L::load(d, t, off[t], r, z, z1, lane);
                        z = plane_step(z, 4 * iskb, span);
                        d += 4 * B::PLANE;
                    }
            };
            vm_wait<0>();  // the brick that is computed now
            lds_barrier();
            pairs(3);
            lds_barrier();
            pairs(1);
            lds_barrier();
            if (!more) break;
            b += step;
            dst = P + (dst == P ? B::CELLS : 0);
        }
        return;
    }

    const StarW<double> w0 = load_w<double>(a.c);
    // first stage: planes za and za + 1 of twelve of the column (bx, by); the last two waves take
    // the columns around the brick
    const int ring = lane & 31;
    int bx = lane & 7, by = lane >> 3, za = 2 * wave;
    if (wave >= 6) {
        bx = ring < 16 ? ring & 7 : ring < 24 ? -1 : 8;
        by = ring < 8 ? -1 : ring < 16 ? 8 : ring & 7;
        za = 2 + 4 * (wave - 6) + 2 * (lane >> 5);
    }
    double* ca = P + za * B::PLANE + (2 * by + 4) * B::W + 2 * bx + 4;
    // second stage: a plane per wave
    const int zb = wave, cx = 2 * (lane & 7), cy = 2 * (lane >> 3);
    const double* cb = P + (zb + 2) * B::PLANE + (cy + 4) * B::W + cx + 4;

    d2 qa[2][2], qb[1][2];
    const auto bases = [&]() {  // launch A reads them from the input in LDS
        if constexpr (!FIRST) {
            const __amdgpu_buffer_rsrc_t r = make_rsrc((const double*)h.q.p + slice * h.q.slice, h.q_bytes);
            BrickCols<PAIR> col;
            col.set(x0 + 2 * bx, y0 + 2 * by, ni, nj, (int)h.q.sj);
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int f = 0; f < 2; ++f) qa[j][f] = col.ld_lane(r, f, wrapz(z0 - 2 + za + j, nk) * qskb);
            col.set(x0 + cx, y0 + cy, ni, nj, (int)h.q.sj);
#pragma unroll
            for (int f = 0; f < 2; ++f) qb[0][f] = col.ld(r, f, wrapz(z0 + zb, nk) * qskb);
        }
    };
    bases();
    int next = B::CELLS;
    for (;;) {
        lds_barrier();
        const StarW<double> w = a.cdev ? load_w<double>(a.cdev[slice]) : w0;
        d2 va[2][2];
        if constexpr (FIRST) {
            brick_stage<2>(va, ca, w, w.f1, nullptr);
            quad_read_c<B::W>(cb + 2 * B::PLANE, qb[0]);
        } else {
            brick_stage<2>(va, ca, w, w.f3, qa);
        }
        lds_barrier();
#pragma unroll
        for (int j = 0; j < 2; ++j) quad_write<B::W>(ca + (j + 2) * B::PLANE, va[j]);
        lds_barrier();
        d2 vb[1][2];
        brick_stage<1>(vb, cb, w, FIRST ? w.f2 : w.f4, qb);
        if (z0 + zb < nk) {
            const __amdgpu_buffer_rsrc_t r = make_rsrc((double*)a.out.p + slice * a.out.slice, a.out_bytes);
            BrickCols<PAIR> col;
            col.set(x0 + cx, y0 + cy, ni, nj, (int)a.out.sj);  // periodic image for partial bricks
#pragma unroll
            for (int f = 0; f < 2; ++f) col.st(r, f, (z0 + zb) * oskb, vb[0][f]);
        }
        if (b + step >= last) break;
        b += step;
        place(b);
        bases();
        ca += next;
        cb += next;
        next = -next;
    }
}

// One launch over one batch of slices.
template <typename SI, typename SO, typename T, int TX, int TY, int NT>
__global__ void __launch_bounds__(NT) k_rk4_fused(FusedArgs a)
{
    rk4_scalar_body<SI, SO, T, TX, TY, NT>(a, xcd_block(blockIdx.x, gridDim.x));
}

template <typename SI, typename SO, typename T, int TX, int TY, int NT>
__global__ void __launch_bounds__(NT) k_rk4_fused_pair(FusedArgs a)
{
    rk4_pair_body<SI, SO, T, TX, TY, NT>(a, xcd_block(blockIdx.x, gridDim.x));
}

__global__ void __launch_bounds__(QuadCfg::WAVES * 64) k_rk4_fused_quad(FusedArgs a)
{
    rk4_quad_body(a, xcd_block(blockIdx.x, gridDim.x));
}

template <int TX, int TY, int NT, bool FIRST>
__global__ void __launch_bounds__(NT) k_rk4_half_pair(HalfArgs h)
{
    rk4_half_pair_body<TX, TY, NT, FIRST>(h, xcd_block(blockIdx.x, gridDim.x));
}

template <bool FIRST, bool PAIR>
__global__ void __launch_bounds__(BrickCfg::THREADS) k_rk4_brick(HalfArgs h)
{
    rk4_brick_body<FIRST, PAIR>(h);
}

// One launch over several independent batches (problems of different sizes, steps and
// coefficients): entry e owns blocks [first[e], first[e+1]); a block finds its entry by a
// scalar scan (entries are few) and runs the same body on that entry's arguments.
__device__ __forceinline__ int group_entry(const GroupArgs& g, int bid)
{
    int e = 0;
    while (e + 1 < g.n && g.first[e + 1] <= bid) ++e;
    return e;
}

// The records are read through the constant address space: with a block-uniform index
// the loads are scalar, so the arguments live in scalar registers as kernel arguments do.
typedef __attribute__((address_space(4))) const FusedArgs ConstArgs;

template <typename SI, typename SO, typename T, int TX, int TY, int NT>
__global__ void __launch_bounds__(NT) k_rk4_fused_grouped(GroupArgs g)
{
    const int bid = xcd_block(blockIdx.x, gridDim.x);
    const int e = group_entry(g, bid);
    ConstArgs* rec = (ConstArgs*)g.args + e;
    rk4_scalar_body<SI, SO, T, TX, TY, NT>(*(const FusedArgs*)rec, bid - g.first[e]);
}

template <typename SI, typename SO, typename T, int TX, int TY, int NT>
__global__ void __launch_bounds__(NT) k_rk4_fused_pair_grouped(GroupArgs g)
{
    const int bid = xcd_block(blockIdx.x, gridDim.x);
    const int e = group_entry(g, bid);
    ConstArgs* rec = (ConstArgs*)g.args + e;
    rk4_pair_body<SI, SO, T, TX, TY, NT>(*(const FusedArgs*)rec, bid - g.first[e]);
}

__global__ void __launch_bounds__(QuadCfg::WAVES * 64) k_rk4_fused_quad_grouped(GroupArgs g)
{
    const int bid = xcd_block(blockIdx.x, gridDim.x);
    const int e = group_entry(g, bid);
    ConstArgs* rec = (ConstArgs*)g.args + e;
    rk4_quad_body(*(const FusedArgs*)rec, bid - g.first[e]);
}

}  // namespace

Coefs make_coefs(double nu, double cx, double cy, double cz, double dx, double h)
{
    const Coef13 k = make_coef13(nu, cx, cy, cz, dx);
    Coefs c;
    const double w[13] = {k.x[0], k.x[1], k.x[2], k.x[3], k.y[0], k.y[1], k.y[2],
                          k.y[3], k.z[0], k.z[1], k.z[2], k.z[3], k.c};
    const double f[4] = {0.25 * h, h / 3., 0.5 * h, h};
    for (int i = 0; i < 13; ++i) {
        c.wd[i] = w[i];
        c.wf[i] = (float)w[i];
    }
    for (int i = 0; i < 4; ++i) {
        c.fd[i] = f[i];
        c.ff[i] = (float)f[i];
    }
    return c;
}

size_t coefs_size() { return sizeof(Coefs); }

void fill_coefs(void* dst, double nu, double cx, double cy, double cz, double dx, double h)
{
    *(Coefs*)dst = make_coefs(nu, cx, cy, cz, dx, h);
}

namespace {

// The split variant's brick shape (its k chunk is the brick's).
bool is_brick(const FusedTile& t)
{
    return t.variant == SP_KERNEL_SPLIT && t.tx == BrickCfg::BX && t.ty == BrickCfg::BY && t.nt == BrickCfg::NT;
}

int fill_args(FusedArgs& a, const FusedStep& st, const FusedTile& tile, View in, View out, int isz, int osz)
{
    a.in = in;
    a.out = out;
    const long long span_in = (st.ni - 1) + (st.nj - 1) * in.sj + (st.nk - 1) * in.sk + 1;
    const long long span_out = (st.ni - 1) + (st.nj - 1) * out.sj + (st.nk - 1) * out.sk + 1;
    const long long bi = span_in * isz, bo = span_out * osz;
    if (bi >= (1LL << 31) || bo >= (1LL << 31))
        return fail(SP_ERR_UNSUPPORTED, "fused RK4: one field must span less than 2 GiB");
    a.in_bytes = (unsigned)bi;
    a.out_bytes = (unsigned)bo;
    a.ni = st.ni;
    a.nj = st.nj;
    a.nk = st.nk;
    a.kchunk = is_brick(tile) ? BrickCfg::BZ : tile.kchunk > 0 ? min(tile.kchunk, st.nk) : st.nk;
    a.tiles_x = (st.ni + tile.tx - 1) / tile.tx;
    const int tiles_y = (st.nj + tile.ty - 1) / tile.ty;
    a.tiles = a.tiles_x * tiles_y;
    a.chunks = (st.nk + a.kchunk - 1) / a.kchunk;
    a.c = make_coefs(st.nu, st.cx, st.cy, st.cz, st.dx, st.dt);
    a.cdev = (const Coefs*)st.coef_dev;
    const long long nblocks = (long long)a.tiles * a.chunks * st.nslices;
    if (nblocks > 0x7fffffffLL) return fail(SP_ERR_UNSUPPORTED, "fused RK4: too many blocks");
    return SP_OK;
}

unsigned nblocks_of(const FusedArgs& a, int nslices) { return (unsigned)((long long)a.tiles * a.chunks * nslices); }

template <typename SI, typename SO, typename T>
int launch_typed(hipStream_t s, const FusedStep& st, const FusedTile& tile, View in, View out)
{
    FusedArgs a;
    SP_TRY(fill_args(a, st, tile, in, out, (int)sizeof(SI), (int)sizeof(SO)));
    const dim3 grid(nblocks_of(a, st.nslices));
#define SP_FUSED_CASE(TX_, TY_, NT_)                                                             \
    if (tile.tx == TX_ && tile.ty == TY_ && tile.nt == NT_) {                                    \
        hipLaunchKernelGGL((k_rk4_fused<SI, SO, T, TX_, TY_, NT_>), grid, dim3(NT_), 0, s, a);   \
        SP_HIP(hipGetLastError());                                                               \
        return SP_OK;                                                                            \
    }
    SP_FUSED_CASE(32, 32, 1024)
    SP_FUSED_CASE(32, 24, 1024)
    SP_FUSED_CASE(24, 24, 1024)
    SP_FUSED_CASE(32, 16, 512)
    SP_FUSED_CASE(16, 16, 256)
#undef SP_FUSED_CASE
    return fail(SP_ERR_UNSUPPORTED, "fused RK4: unsupported tile shape");
}

template <typename SI, typename SO, typename T>
int launch_pair(hipStream_t s, const FusedStep& st, const FusedTile& tile, View in, View out)
{
    FusedArgs a;
    SP_TRY(fill_args(a, st, tile, in, out, (int)sizeof(SI), (int)sizeof(SO)));
    const dim3 grid(nblocks_of(a, st.nslices));
#define SP_PAIR_CASE(TX_, TY_, NT_)                                                                  \
    if (tile.tx == TX_ && tile.ty == TY_ && tile.nt == NT_) {                                        \
        hipLaunchKernelGGL((k_rk4_fused_pair<SI, SO, T, TX_, TY_, NT_>), grid, dim3(NT_), 0, s, a); \
        SP_HIP(hipGetLastError());                                                                   \
        return SP_OK;                                                                                \
    }
    SP_PAIR_CASE(32, 32, 512)
    SP_PAIR_CASE(32, 16, 512)
    SP_PAIR_CASE(16, 16, 256)
#undef SP_PAIR_CASE
    return fail(SP_ERR_UNSUPPORTED, "fused RK4 (pair): unsupported tile shape");
}

int launch_quad(hipStream_t s, const FusedStep& st, const FusedTile& tile, View in, View out)
{
    SP_CHECK(tile.tx == QuadCfg::TX && tile.ty == QuadCfg::TY && tile.nt == QuadCfg::NT, SP_ERR_UNSUPPORTED,
             "fused RK4 (2x2): unsupported tile shape");
    FusedArgs a;
    SP_TRY(fill_args(a, st, tile, in, out, 8, 8));
    hipLaunchKernelGGL(k_rk4_fused_quad, dim3(nblocks_of(a, st.nslices)), dim3(QuadCfg::WAVES * 64), 0, s, a);
    SP_HIP(hipGetLastError());
    return SP_OK;
}

// Pair access (two elements per lane) needs even x extent, even strides and origins aligned
// to two elements of each field's storage type (FP64: 16 bytes).
bool pair_ok(const FusedStep& st, View in, View out, int isz = 8, int osz = 8)
{
    const auto even = [](long long v) { return (v & 1) == 0; };
    return even(st.ni) && even(in.sj) && even(in.sk) && even(out.sj) && even(out.sk) && even(in.slice) &&
           even(out.slice) && ((uintptr_t)in.p % (2 * isz)) == 0 && ((uintptr_t)out.p % (2 * osz)) == 0;
}

// Launch A (in -> work: v2) and launch B (work, in -> out: q').  Requires st.work.
int launch_split(hipStream_t s, const FusedStep& st, const FusedTile& tile, View in, View out)
{
    SP_CHECK(st.work && st.work_bytes >= split_work_bytes(st.ni, st.nj, st.nk, st.nslices), SP_ERR_INVALID,
             "fused RK4 (split): no work field for this batch");
    View wv;
    wv.p = st.work;
    wv.sj = st.ni;
    wv.sk = (long long)st.ni * st.nj;
    wv.slice = wv.sk * st.nk;
    HalfArgs A, B;
    SP_TRY(fill_args(A.a, st, tile, in, wv, 8, 8));
    A.q = in;
    A.q_bytes = A.a.in_bytes;
    SP_TRY(fill_args(B.a, st, tile, wv, out, 8, 8));
    B.q = in;
    B.q_bytes = A.a.in_bytes;
    dim3 grid(nblocks_of(A.a, st.nslices));
    if (is_brick(tile)) {
        for (HalfArgs* h : {&A, &B}) {
            h->bricks = (int)grid.x;
            h->inv_tiles = 0xffffffffu / h->a.tiles;
            h->inv_chunks = 0xffffffffu / h->a.chunks;
            h->inv_tiles_x = 0xffffffffu / h->a.tiles_x;
        }
        grid.x = std::min(grid.x, 256u);  // two buffers fill a CU's LDS: one block per CU
        const dim3 block(BrickCfg::THREADS);
        // each launch by its own fields' alignment (the work field's rows are ni long)
        const bool even = (st.ni & 1) == 0;
        if (even && pair_ok(st, in, wv)) hipLaunchKernelGGL((k_rk4_brick<true, true>), grid, block, 0, s, A);
        else hipLaunchKernelGGL((k_rk4_brick<true, false>), grid, block, 0, s, A);
        SP_HIP(hipGetLastError());
        if (even && pair_ok(st, in, wv) && pair_ok(st, wv, out))
            hipLaunchKernelGGL((k_rk4_brick<false, true>), grid, block, 0, s, B);
        else hipLaunchKernelGGL((k_rk4_brick<false, false>), grid, block, 0, s, B);
        SP_HIP(hipGetLastError());
        return SP_OK;
    }
#define SP_SPLIT_CASE(TX_, TY_, NT_)                                                           \
    if (tile.tx == TX_ && tile.ty == TY_ && tile.nt == NT_) {                                  \
        hipLaunchKernelGGL((k_rk4_half_pair<TX_, TY_, NT_, true>), grid, dim3(NT_), 0, s, A);  \
        SP_HIP(hipGetLastError());                                                             \
        hipLaunchKernelGGL((k_rk4_half_pair<TX_, TY_, NT_, false>), grid, dim3(NT_), 0, s, B); \
        SP_HIP(hipGetLastError());                                                             \
        return SP_OK;                                                                          \
    }
    SP_SPLIT_CASE(32, 32, 512)
    SP_SPLIT_CASE(32, 16, 512)
    SP_SPLIT_CASE(32, 16, 256)
    SP_SPLIT_CASE(16, 16, 256)
#undef SP_SPLIT_CASE
    return fail(SP_ERR_UNSUPPORTED, "fused RK4 (split): unsupported tile shape");
}

template <typename SI, typename SO, typename T>
int launch_grouped_pair(hipStream_t s, const FusedTile& tile, GroupArgs g, long long nblocks)
{
    const dim3 grid((unsigned)nblocks);
#define SP_PAIR_CASE(TX_, TY_, NT_)                                                                            \
    if (tile.tx == TX_ && tile.ty == TY_ && tile.nt == NT_) {                                                  \
        hipLaunchKernelGGL((k_rk4_fused_pair_grouped<SI, SO, T, TX_, TY_, NT_>), grid, dim3(NT_), 0, s, g); \
        SP_HIP(hipGetLastError());                                                                             \
        return SP_OK;                                                                                          \
    }
    SP_PAIR_CASE(32, 32, 512)
    SP_PAIR_CASE(32, 16, 512)
    SP_PAIR_CASE(16, 16, 256)
#undef SP_PAIR_CASE
    return fail(SP_ERR_UNSUPPORTED, "grouped fused RK4 (pair): unsupported tile shape");
}

template <typename SI, typename SO, typename T>
int launch_grouped_typed(hipStream_t s, const FusedTile& tile, GroupArgs g, long long nblocks)
{
    const dim3 grid((unsigned)nblocks);
#define SP_FUSED_CASE(TX_, TY_, NT_)                                                                     \
    if (tile.tx == TX_ && tile.ty == TY_ && tile.nt == NT_) {                                            \
        hipLaunchKernelGGL((k_rk4_fused_grouped<SI, SO, T, TX_, TY_, NT_>), grid, dim3(NT_), 0, s, g);   \
        SP_HIP(hipGetLastError());                                                                       \
        return SP_OK;                                                                                    \
    }
    SP_FUSED_CASE(32, 32, 1024)
    SP_FUSED_CASE(32, 24, 1024)
    SP_FUSED_CASE(24, 24, 1024)
    SP_FUSED_CASE(32, 16, 512)
    SP_FUSED_CASE(16, 16, 256)
#undef SP_FUSED_CASE
    return fail(SP_ERR_UNSUPPORTED, "grouped fused RK4: unsupported tile shape");
}

}  // namespace

size_t fused_record_size() { return sizeof(FusedArgs); }

int fused_record_fill(void* rec, const FusedStep& st, const FusedTile& tile, int in_dtype, View in, int out_dtype,
                      View out, long long* nblocks)
{
    SP_CHECK(st.nk >= kFusedMinK, SP_ERR_UNSUPPORTED, "grouped fused RK4: ksize below the fused kernel's minimum");
    FusedArgs a;
    SP_TRY(fill_args(a, st, tile, in, out, dtype_size(in_dtype), dtype_size(out_dtype)));
    std::memcpy(rec, &a, sizeof(a));
    *nblocks = (long long)nblocks_of(a, st.nslices);
    return SP_OK;
}

bool fused_record_pair_ok(const FusedStep& st, View in, View out, int in_dtype, int out_dtype)
{
    return pair_ok(st, in, out, dtype_size(in_dtype), dtype_size(out_dtype));
}

int launch_rk4_grouped(hipStream_t s, const FusedTile& tile, int in_dtype, int out_dtype, const void* records,
                       const int* first, int n, long long nblocks)
{
    SP_CHECK(n >= 1 && nblocks >= 1 && nblocks <= 0x7fffffffLL, SP_ERR_INVALID, "grouped fused RK4: empty or too large");
    const GroupArgs g{(const FusedArgs*)records, first, n};
    if (tile.variant == SP_KERNEL_QUAD) {
        SP_CHECK(in_dtype == SP_F64 && out_dtype == SP_F64, SP_ERR_UNSUPPORTED, "grouped 2x2 kernel is FP64 only");
        SP_CHECK(tile.tx == QuadCfg::TX && tile.ty == QuadCfg::TY && tile.nt == QuadCfg::NT, SP_ERR_UNSUPPORTED,
                 "grouped fused RK4 (2x2): unsupported tile shape");
        hipLaunchKernelGGL(k_rk4_fused_quad_grouped, dim3((unsigned)nblocks), dim3(QuadCfg::WAVES * 64), 0, s, g);
        SP_HIP(hipGetLastError());
        return SP_OK;
    }
    if (tile.variant == SP_KERNEL_PAIR) {
        if (in_dtype == SP_F64 && out_dtype == SP_F64) return launch_grouped_pair<double, double, double>(s, tile, g, nblocks);
        if (in_dtype == SP_F64 && out_dtype == SP_F32) return launch_grouped_pair<double, float, float>(s, tile, g, nblocks);
        if (in_dtype == SP_F32 && out_dtype == SP_F32) return launch_grouped_pair<float, float, float>(s, tile, g, nblocks);
        if (in_dtype == SP_F64 && out_dtype == SP_BF16) return launch_grouped_pair<double, bf16, float>(s, tile, g, nblocks);
        if (in_dtype == SP_BF16 && out_dtype == SP_BF16) return launch_grouped_pair<bf16, bf16, float>(s, tile, g, nblocks);
        return fail(SP_ERR_UNSUPPORTED, "grouped fused RK4 (pair): unsupported dtype pair");
    }
    if (in_dtype == SP_F64 && out_dtype == SP_F64) return launch_grouped_typed<double, double, double>(s, tile, g, nblocks);
    if (in_dtype == SP_F64 && out_dtype == SP_F32) return launch_grouped_typed<double, float, float>(s, tile, g, nblocks);
    if (in_dtype == SP_F32 && out_dtype == SP_F32) return launch_grouped_typed<float, float, float>(s, tile, g, nblocks);
    if (in_dtype == SP_F64 && out_dtype == SP_BF16) return launch_grouped_typed<double, bf16, float>(s, tile, g, nblocks);
    if (in_dtype == SP_BF16 && out_dtype == SP_BF16) return launch_grouped_typed<bf16, bf16, float>(s, tile, g, nblocks);
    return fail(SP_ERR_UNSUPPORTED, "grouped fused RK4: unsupported dtype pair");
}

bool fused_tile_brick(const FusedTile& t) { return is_brick(t); }

bool fused_tile_supported(const FusedTile& t, int /*compute_f64*/)
{
    static const int scalar[][3] = {{32, 32, 1024}, {32, 24, 1024}, {24, 24, 1024}, {32, 16, 512}, {16, 16, 256}};
    static const int pair[][3] = {{32, 32, 512}, {32, 16, 512}, {16, 16, 256}};
    static const int split[][3] = {{32, 32, 512}, {32, 16, 512}, {32, 16, 256}, {16, 16, 256}, {16, 16, 384}};
    if (t.variant == SP_KERNEL_QUAD) return t.tx == QuadCfg::TX && t.ty == QuadCfg::TY && t.nt == QuadCfg::NT;
    if (t.variant == SP_KERNEL_SPLIT) {
        for (const auto& sh : split)
            if (t.tx == sh[0] && t.ty == sh[1] && t.nt == sh[2]) return true;
        return false;
    }
    if (t.variant == SP_KERNEL_PAIR) {
        for (const auto& sh : pair)
            if (t.tx == sh[0] && t.ty == sh[1] && t.nt == sh[2]) return true;
        return false;
    }
    for (const auto& sh : scalar)
        if (t.tx == sh[0] && t.ty == sh[1] && t.nt == sh[2]) return true;
    return false;
}

namespace {

long long tiles_of(int ni, int nj, int nslices, int tx, int ty)
{
    return (long long)((ni + tx - 1) / tx) * ((nj + ty - 1) / ty) * nslices;
}

// A streaming kernel's time in us: each block walks its k chunk and `fill` planes more, in groups
// of `group`.  A plane of a round of 256 blocks (one per CU) takes `first`, and `more` for every
// round where several blocks share a CU.
struct WalkCost {
    int fill, group;
    double first, more;
};
constexpr WalkCost kQuadWalk{18, 4, 1.3, 1.3};

// The k chunk for which the blocks of these tiles finish first, and that time.
int best_kchunk(long long tiles, int nk, const WalkCost& c, double* us)
{
    int best = nk;
    *us = 1e30;
    for (int chunks = 1; chunks <= nk / 8 || chunks == 1; ++chunks) {
        const int kc = (nk + chunks - 1) / chunks;
        const long long rounds = (tiles * ((nk + kc - 1) / kc) + 255) / 256;
        const double t = std::max(c.first, c.more * rounds) * ((kc + c.fill + c.group - 1) / c.group * c.group);
        if (t < *us) {
            *us = t;
            best = kc;
        }
    }
    return best;
}

}  // namespace

FusedTile default_tile(int ni, int nj, int nk, int nslices, int compute_f64, bool one_launch, bool aligned)
{
    const bool pairs = aligned && !(ni & 1);  // rows of aligned x pairs
    // FP64: the 2x2 kernel with the k chunk that finishes first, or bricks (two launches) while
    // those are few.  Measured on MI355X in us per step:
    //   2x2: 1.25-1.4 per plane and round of 256 blocks (1 x 256^3 in 64-plane chunks 120, 4 x
    //   128^3 in 32-plane chunks 73, 16 x 128^3 210, 1 x 384^3 in 128-plane chunks 389); the
    //   whole-k and 64-plane chunks chosen before: 1 x 256^3 250, 4 x 128^3 155, 1 x 384^3 437.
    //   bricks: 7.5 and 5.7 per round of 256 (1 x 64^3 13.0 against 35 for the 2x2 kernel; 432
    //   bricks, 1 x 96^3: 19 against 35; 1024, 1 x 128^3: 30.5 against 35.3; 1728, 4 x 96^3: 46
    //   against 41).
    // Odd x extents and strides cannot take the 2x2 kernel's 16-byte accesses: bricks, 8.1 per
    // round, while they are faster than the scalar kernel (127^3 40 against 56, 161^3 84 against
    // 145, 201^3 141 against 271; 255^3, 8192 bricks, 284 against 287, and 256^3 in rows of 257
    // 267 for the scalar kernel).
    const long long bricks = tiles_of(ni, nj, nslices, 16, 16) * ((nk + 7) / 8);
    if (compute_f64 && !one_launch) {
        const FusedTile brick{16, 16, 384, 8, SP_KERNEL_SPLIT};
        if (!pairs) {
            if (bricks < 8192) return brick;
        } else {
            double us;
            const int kc = best_kchunk(tiles_of(ni, nj, nslices, 32, 32), nk, kQuadWalk, &us);
            if (7.5 + 5.7 * ((bricks + 255) / 256) < us) return brick;
            return FusedTile{32, 32, 512, kc >= nk ? 0 : kc, SP_KERNEL_QUAD};
        }
    }
    // FP32 / BF16 storage: the x-pair kernel in the tile and k chunk that finish first.  Measured in
    // FP32, us per plane (BF16 5-20 % more): 32x32 1.46 per round, 32x16 1.05 alone and 0.78 per
    // round of two and more, 16x16 0.88 and 0.60.  1 x 64^3 16x16 in 8-plane chunks 23.6 us (34.5
    // for 32x16 in 16), 1 x 256^3 32x32 in 64 122 (154 for 32x16 in 128), 1 x 384^3 32x32 in 77-80
    // 420 (479 in 64; BF16 526 against 598, its best, 32x16 in 64, 499).
    if (!compute_f64 && !one_launch && pairs) {
        static constexpr struct {
            int tx, ty, nt;
            WalkCost cost;
        } shapes[] = {{32, 32, 512, {19, 1, 1.46, 1.46}},
                      {32, 16, 512, {19, 1, 1.05, 0.78}},
                      {16, 16, 256, {19, 1, 0.88, 0.60}}};
        FusedTile t{};
        double least = 1e30;
        for (const auto& sh : shapes) {
            double us;
            const int kc = best_kchunk(tiles_of(ni, nj, nslices, sh.tx, sh.ty), nk, sh.cost, &us);
            if (us < least) t = FusedTile{sh.tx, sh.ty, sh.nt, kc >= nk ? 0 : kc, SP_KERNEL_PAIR}, least = us;
        }
        return t;
    }
    // One launch per step (which other problems may share), and odd extents past the bricks: the
    // scalar kernel in reduced precision and where accesses are not aligned.
    const long long want = 256;  // one block per CU
    FusedTile t{32, 32, 512, 0, compute_f64 ? SP_KERNEL_QUAD : SP_KERNEL_PAIR};
    long long blocks = tiles_of(ni, nj, nslices, t.tx, t.ty);
    if (blocks < want && blocks * (nk / 64) >= 3 * want) {
        t.kchunk = 64;
        return t;
    }
    if (blocks < want) {
        t.ty = 16;
        t.variant = SP_KERNEL_PAIR;
        blocks = tiles_of(ni, nj, nslices, t.tx, t.ty);
    }
    int chunks = (int)((want + blocks - 1) / blocks);
    if (chunks < 1) chunks = 1;
    int kc = (nk + chunks - 1) / chunks;
    if (kc < 16) kc = 16;
    t.kchunk = kc >= nk ? 0 : kc;
    return t;
}

void fused_candidates(int ni, int nj, int nk, int nslices, int compute_f64, std::vector<FusedTile>& out)
{
    static const int scalar[][3] = {{32, 32, 1024}, {32, 24, 1024}, {24, 24, 1024}, {32, 16, 512}, {16, 16, 256}};
    static const int pair[][3] = {{32, 32, 512}, {32, 16, 512}, {16, 16, 256}};
    static const int split[][3] = {{32, 32, 512}, {32, 16, 512}, {32, 16, 256}, {16, 16, 256}, {16, 16, 384}};
    std::vector<FusedTile> shapes;
    if (!compute_f64 && ni % 2 == 0)
        for (const auto& sh : pair) shapes.push_back(FusedTile{sh[0], sh[1], sh[2], 0, SP_KERNEL_PAIR});
    if (compute_f64 && ni % 2 == 0) {
        shapes.push_back(FusedTile{QuadCfg::TX, QuadCfg::TY, QuadCfg::NT, 0, SP_KERNEL_QUAD});
        for (const auto& sh : pair) shapes.push_back(FusedTile{sh[0], sh[1], sh[2], 0, SP_KERNEL_PAIR});
        // the split steps move a third field: candidates while a field of the batch stays
        // within 64 MiB (the last-level cache holds the three)
        if (split_work_bytes(ni, nj, nk, nslices) <= (64u << 20))
            for (const auto& sh : split) shapes.push_back(FusedTile{sh[0], sh[1], sh[2], 0, SP_KERNEL_SPLIT});
    } else if (compute_f64 && split_work_bytes(ni, nj, nk, nslices) <= (64u << 20))
        shapes.push_back(FusedTile{BrickCfg::BX, BrickCfg::BY, BrickCfg::NT, 0, SP_KERNEL_SPLIT});
    for (const auto& sh : scalar) shapes.push_back(FusedTile{sh[0], sh[1], sh[2], 0, SP_KERNEL_SCALAR});
    out.clear();
    for (const FusedTile& t : shapes) {
        if (is_brick(t)) {
            out.push_back(FusedTile{t.tx, t.ty, t.nt, BrickCfg::BZ, t.variant});
            continue;
        }
        const long long blocks = tiles_of(ni, nj, nslices, t.tx, t.ty);
        // k chunks: the whole extent, and shorter ones (>= 16 planes, >= 8 for the 2x2 and split
        // kernels) only while the tiles alone give fewer than 4 blocks per CU
        const int cmin = t.variant == SP_KERNEL_SPLIT || t.variant == SP_KERNEL_QUAD ? 8 : 16;
        std::vector<int> kcs{0};
        double us;
        const int best = t.variant == SP_KERNEL_QUAD ? best_kchunk(blocks, nk, kQuadWalk, &us) : 0;
        if (blocks < 1024)
            for (int c : {nk / 2, nk / 4, nk / 8, 64, 32, 16, 8})
                if (c >= cmin && c < nk && std::find(kcs.begin(), kcs.end(), c) == kcs.end()) kcs.push_back(c);
        if (best > 0 && best < nk && std::find(kcs.begin(), kcs.end(), best) == kcs.end()) kcs.push_back(best);
        for (int c : kcs) {
            FusedTile x = t;
            x.kchunk = c;
            out.push_back(x);
        }
    }
}

int launch_rk4_fused(hipStream_t s, const FusedStep& st, const FusedTile& tile_in, int in_dtype, View in,
                     int out_dtype, View out)
{
    FusedTile tile = tile_in;
    const bool f64 = in_dtype == SP_F64 && out_dtype == SP_F64;
    if (st.nk < kFusedMinK)
        return fail(SP_ERR_UNSUPPORTED, "fused RK4: ksize " + std::to_string(st.nk) + " < " +
                                            std::to_string(kFusedMinK) + " (use the staged path)");
    if (f64 && tile.variant == SP_KERNEL_QUAD && pair_ok(st, in, out)) return launch_quad(s, st, tile, in, out);
    if (f64 && tile.variant == SP_KERNEL_PAIR && pair_ok(st, in, out))
        return launch_pair<double, double, double>(s, st, tile, in, out);
    if (!f64 && tile.variant == SP_KERNEL_PAIR &&
        pair_ok(st, in, out, (int)dtype_size(in_dtype), (int)dtype_size(out_dtype))) {
        if (in_dtype == SP_F64 && out_dtype == SP_F32) return launch_pair<double, float, float>(s, st, tile, in, out);
        if (in_dtype == SP_F32 && out_dtype == SP_F32) return launch_pair<float, float, float>(s, st, tile, in, out);
        if (in_dtype == SP_F64 && out_dtype == SP_BF16) return launch_pair<double, bf16, float>(s, st, tile, in, out);
        if (in_dtype == SP_BF16 && out_dtype == SP_BF16) return launch_pair<bf16, bf16, float>(s, st, tile, in, out);
    }
    if (f64 && tile.variant == SP_KERNEL_SPLIT && (is_brick(tile) || pair_ok(st, in, out)))
        return launch_split(s, st, tile, in, out);
    if (tile.variant == SP_KERNEL_PAIR || tile.variant == SP_KERNEL_QUAD || tile.variant == SP_KERNEL_SPLIT) {
        // odd sizes, unaligned views or reduced-precision storage: the scalar kernel with
        // its fastest FP64 shape and the caller's k chunk
        tile.tx = 32;
        tile.ty = 16;
        tile.nt = 512;
        tile.variant = SP_KERNEL_SCALAR;
    }
    if (f64) return launch_typed<double, double, double>(s, st, tile, in, out);
    if (in_dtype == SP_F64 && out_dtype == SP_F32) return launch_typed<double, float, float>(s, st, tile, in, out);
    if (in_dtype == SP_F32 && out_dtype == SP_F32) return launch_typed<float, float, float>(s, st, tile, in, out);
    if (in_dtype == SP_F64 && out_dtype == SP_BF16) return launch_typed<double, bf16, float>(s, st, tile, in, out);
    if (in_dtype == SP_BF16 && out_dtype == SP_BF16) return launch_typed<bf16, bf16, float>(s, st, tile, in, out);
    if (in_dtype == SP_F32 && out_dtype == SP_F64) return launch_typed<float, double, float>(s, st, tile, in, out);
    if (in_dtype == SP_BF16 && out_dtype == SP_F64) return launch_typed<bf16, double, float>(s, st, tile, in, out);
    if (in_dtype == SP_BF16 && out_dtype == SP_F32) return launch_typed<bf16, float, float>(s, st, tile, in, out);
    if (in_dtype == SP_F32 && out_dtype == SP_BF16) return launch_typed<float, bf16, float>(s, st, tile, in, out);
    return fail(SP_ERR_UNSUPPORTED, "fused RK4: unsupported dtype pair");
}

}  // namespace sp
