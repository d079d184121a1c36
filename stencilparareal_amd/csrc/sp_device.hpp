// sp_device.hpp -- device helpers shared by the kernels: periodic indices, buffer-resource
// access, loads into LDS and their waits, the XCD-aware block order.
#pragma once

#include <hip/hip_runtime.h>

namespace sp {
namespace {

__device__ __forceinline__ int pmod(int a, int n)
{
    int r = a % n;
    return r < 0 ? r + n : r;
}

// a in [-n, 2n) where n >= 24 (block-uniform), any a otherwise: two selects instead of a division
__device__ __forceinline__ int near_mod(int a, int n)
{
    if (n < 24) return pmod(a, n);
    a += a < 0 ? n : 0;
    return a - (a >= n ? n : 0);
}

// z, a plane's byte offset below span (all planes'), d <= span further on
__device__ __forceinline__ unsigned plane_step(unsigned z, unsigned d, unsigned span)
{
    return min(z + d, z + d - span);  // the second is huge unless the first is past the end
}

// Plane index p in [-3n, 4n) wrapped into [0, n) without branches (scalar selects).  The
// stream touches planes z0-18 .. zend+16, inside that range for n >= 8; the host sends
// smaller k extents to the reference-order path.
__device__ __forceinline__ int wrapz(int p, int n)
{
    p += p < 0 ? n : 0;
    p += p < 0 ? n : 0;
    p += p < 0 ? n : 0;
    p -= p >= n ? n : 0;
    p -= p >= n ? n : 0;
    p -= p >= n ? n : 0;
    return p;
}

// Buffer-resource access: one SGPR descriptor per field, 32-bit per-lane byte offsets
// and the plane offset in an SGPR, so the k stream needs no 64-bit address arithmetic.
// Out-of-range offsets read 0 / drop the store instead of faulting.
#define SP_RSRC_DWORD3 0x00020000  // gfx9 family raw buffer (as composable_kernel uses)

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, unsigned bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, SP_RSRC_DWORD3);
}

// Blocks are handed to the 8 XCDs round-robin (block b runs on XCD b % 8).  Renumber so
// that each XCD receives a contiguous range of tiles: neighbouring tiles, which read each
// other's halo columns, then share one L2.  (The first n % 8 XCDs get one block more.)
__device__ __forceinline__ int xcd_block(int b, int n)
{
    const int x = b % 8, r = n % 8;
    return x * (n / 8) + min(x, r) + b / 8;
}

// 16 bytes (or one word) per lane from global memory straight into LDS: lane l of the wave
// writes lds + 16 l (+ 4 l) bytes (lds: the wave's base, the same for every lane).
__device__ __forceinline__ void ld2_to_lds(__amdgpu_buffer_rsrc_t r, double* lds, int vo, int so)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, vo, so, 0, 0);
}
__device__ __forceinline__ void ldw_to_lds(__amdgpu_buffer_rsrc_t r, double* lds, int vo, int so)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 4, vo, so, 0, 0);
}

// Stores through to device scope (cache policy sc1) at once: what a short launch leaves dirty in
// the L2s is written back at its end, after all work, before the next one starts.  A step by
// bricks, before and with it: 96^3 21.2 and 19.0 us, 128^3 32.3 and 30.4, 8 x 64^3 32.1 and 29.5;
// a forward Euler step of 128^3 7.4 and 6.4.  No gain where blocks stream (the 2x2 and pair
// kernels).
template <typename V>
__device__ __forceinline__ void st_through(__amdgpu_buffer_rsrc_t r, int vo, int so, V x)
{
    typedef unsigned u32xn __attribute__((ext_vector_type(sizeof(V) / 4)));
    if constexpr (sizeof(V) == 16) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32xn, x), r, vo, so, 16);
    else __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32xn, x), r, vo, so, 16);
}

// Waits until at most N of this wave's vector-memory accesses are outstanding (they complete
// in the order of issue).
template <int N>
__device__ __forceinline__ void vm_wait() { __builtin_amdgcn_s_waitcnt(0x0F70 | N); }

// Workgroup barrier for LDS data: this wave's LDS accesses are complete before it, but for the
// last N issued (reads of planes that nobody writes next), and none moves across it.  Unlike
// __syncthreads it leaves loads into LDS in flight (vm_wait before it for those that another wave
// reads next).
template <int N = 0>
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_s_waitcnt(0xC07F | N << 8);  // lgkmcnt(N)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_sched_barrier(0);
}

// Loads a brick of D planes of H rows of W doubles (W even, at most 640 cells per plane) from
// (x, y, z) on (x and y at most 24 cells outside the field), with periodic images, into P in the
// order of its cells, straight into LDS: a plane's 16-byte slots by the lanes of waves 0 to 4, or
// (not PAIR: rows that are not 16-byte aligned pairs) four words per lane.  The caller waits for
// the loads (vm_wait, barrier).
template <bool PAIR, int W, int H, int D>
__device__ __forceinline__ void brick_load(double* P, __amdgpu_buffer_rsrc_t r, int skb, int sj, int x, int y, int z,
                                           int ni, int nj, int nk, int wave, int lane)
{
    static_assert(W % 2 == 0 && W * H <= 640, "five waves' slots hold a plane");
    if (wave >= 5) return;
    const unsigned span = (unsigned)nk * skb, zo = wrapz(z, nk) * skb;
    // one mask for all planes of a lane's cell: masks and scalar work around each load would
    // cost more than the load
#pragma unroll
    for (int m = 0; m < (PAIR ? 1 : 4); ++m) {
        const int e = PAIR ? 2 * (wave * 64 + lane) : wave * 128 + m * 32 + (lane >> 1);  // cell of the plane
        if (e < W * H) {
            const int off = (near_mod(x + e % W, ni) + near_mod(y + e / W, nj) * sj) * 8 + (PAIR ? 0 : (lane & 1) * 4);
            double* const dst = P + wave * 128 + m * 32;
            unsigned o = zo;
#pragma unroll
            for (int p = 0; p < D; ++p, o = plane_step(o, skb, span)) {
                if constexpr (PAIR) ld2_to_lds(r, dst + p * W * H, off, o);
                else ldw_to_lds(r, dst + p * W * H, off, o);
            }
        }
    }
}

}  // namespace
}  // namespace sp
