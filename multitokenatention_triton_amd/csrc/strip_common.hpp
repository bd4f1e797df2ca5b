// Helpers shared by the kernels that stage strips of a score plane in LDS with asynchronous copies and read them from
// inline assembly (conv2d_causal.hip, conv_mix16.hip).
#pragma once

#include "common.hpp"

#include <type_traits>
#include <utility>

namespace {
using namespace mta;

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// Returns its argument, opaquely: what is derived from the result cannot be hoisted out of the (rarely taken) block
// that computes it, so it does not occupy registers in the main loop.
__device__ __forceinline__ int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

typedef __attribute__((address_space(3))) void lds_void_t;
typedef const __attribute__((address_space(1))) void glb_void_t;

// LDS is read and written through these, not through C++ accesses: the compiler cannot tell an access to one half of
// the double buffer from the asynchronous copy in flight into the other half and would wait for the copy first (the copy
// would then never overlap the matrix products).  LDS operations of a wavefront complete in order; lds_wait() waits for
// all of them and ties the loaded values to that point.
__device__ __forceinline__ u32x4 lds_load16(unsigned addr)
{
    u32x4 v;
    asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(addr) : "memory");
    return v;
}
// read and wait in one statement: the value is defined when the statement ends (for values that live across code the
// compiler arranges freely)
__device__ __forceinline__ u32x4 lds_load16_sync(unsigned addr)
{
    u32x4 v;
    asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(addr) : "memory");
    return v;
}
// four such reads (1 KB apart, from byte offset `off`: a compile-time constant below 62464) and the wait, one statement
__device__ __forceinline__ void lds_load4x16_sync(unsigned addr, int off, u32x4 &a, u32x4 &b, u32x4 &c, u32x4 &d)
{
    asm volatile("ds_read_b128 %0, %4 offset:%5\n\t"
                 "ds_read_b128 %1, %4 offset:%6\n\t"
                 "ds_read_b128 %2, %4 offset:%7\n\t"
                 "ds_read_b128 %3, %4 offset:%8\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(a), "=&v"(b), "=&v"(c), "=&v"(d)
                 : "v"(addr), "n"(off), "n"(off + 1024), "n"(off + 2048), "n"(off + 3072)
                 : "memory");
}
// the same with a compile-time byte offset in the instruction (no address arithmetic per access)
// (`off` must fold to a constant below 65536: it goes into the instruction's offset field)
__device__ __forceinline__ u32x4 lds_load16_at(unsigned addr, int off)
{
    u32x4 v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(off) : "memory");
    return v;
}
__device__ __forceinline__ unsigned lds_load_u16(unsigned addr)
{
    unsigned v;
    asm volatile("ds_read_u16 %0, %1" : "=v"(v) : "v"(addr) : "memory");
    return v;
}
__device__ __forceinline__ void lds_store8_at(unsigned addr, int off, unsigned lo, unsigned hi)
{
    const u32x2 v = {lo, hi};
    asm volatile("ds_write_b64 %0, %1 offset:%2" : : "v"(addr), "v"(v), "n"(off) : "memory");
}
__device__ __forceinline__ void lds_store16(unsigned addr, u32x4 v)
{
    asm volatile("ds_write_b128 %0, %1" : : "v"(addr), "v"(v) : "memory");
}
// the transpose read: of 16 lanes, lane l at 8 bytes (16-bit elements 4 (l % 4) ..) of row l / 4; it gets element l of the four rows
__device__ __forceinline__ u32x2 lds_load_tr8_at(unsigned addr, int off)
{
    u32x2 v;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(off) : "memory");
    return v;
}
__device__ __forceinline__ void lds_wait() { asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory"); }
__device__ __forceinline__ void lds_wait(u32x4 &a) { asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a) : : "memory"); }
// workgroup barrier without the memory fence __syncthreads() carries (which would wait for the copy in flight)
__device__ __forceinline__ void wg_barrier() { asm volatile("s_barrier" : : : "memory"); }

template <int N> __device__ __forceinline__ void copies_wait() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }
template <int N> __device__ __forceinline__ void lds_wait_upto(u32x2 &a, u32x2 &b) { asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(a), "+v"(b) : "n"(N) : "memory"); }
// what is asked for behind this is asked for after what is ahead of it: the waits count
__device__ __forceinline__ void in_order()
{
    asm volatile("" : : : "memory");
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ unsigned lds_at(const void *p) { return (unsigned)(uintptr_t)(lds_void_t *)p; }

// 16 bytes a lane from a buffer of `bytes` bytes, at `at` (past its end: zeros), to LDS.  From a buffer, not from an address: copies
// from addresses make the compiler wait for everything in flight ahead of any use of a loaded register, these it counts.
__device__ __forceinline__ void copy_to_lds(const void *from, int bytes, void *to, int at)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(from), 0, bytes, 0x00027000), (lds_void_t *)to, 16, at, 0, 0, 0);
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>), in order
template <int... I, typename F> __device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F &&f)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F> __device__ __forceinline__ void static_for(F &&f)
{
    static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

// The (batch, head) and the rank of workgroup wg's block in a grid of heads x blocks whose blocks get shorter with their rank (rows
// under the causal rule): all heads' longest blocks first, so that the short ones fill the end of the grid.  Workgroup ids are
// dealt to the 8 XCDs round-robin; where the heads divide evenly an XCD keeps its own, whose operands then stay in its L2.
// cus > 0: the grid is resident at once, a round of `cus` workgroups per XCD after the other - every second round comes in
// reverse, so that a CU gets a long block and a short one.  False beyond the grid.
__device__ __forceinline__ bool longest_first(unsigned wg, int heads, int blocks, int cus, int &bh, int &rank)
{
    const bool own = heads % 8 == 0;
    const int n = (own ? heads / 8 : heads) * blocks, round = own ? cus : 8 * cus;
    // At most one workgroup per CU: the order does not matter, and an XCD takes a run of neighbouring blocks.  Rows that are no whole
    // lines share one with the next: dealt over the XCDs such rows cost the kernels around this one 2 us (forward of B1 H4 S1571 D64
    // bf16, 6x11 / 3x3: 56.2 against 53.7 us).
    if (!own && cus > 0 && n <= 8 * cus) {
        const int per = (n + 7) / 8, at = (int)(wg & 7) * per + (int)(wg >> 3);
        if (at >= n || (int)(wg >> 3) >= per) return false;
        bh = at / blocks;
        rank = at % blocks;
        return true;
    }
    int pos = own ? (int)(wg >> 3) : (int)wg;
    if (pos >= n) return false;
    if (round > 0 && (pos / round & 1)) {
        const int first = pos / round * round, end = first + round < n ? first + round : n;
        pos = first + (end - 1 - pos);
    }
    const int h = own ? heads / 8 : heads;
    rank = pos / h;
    bh = own ? (int)(wg & 7) * h + pos % h : pos % h;
    return true;
}
__device__ __forceinline__ bool longest_first(int heads, int blocks, int cus, int &bh, int &rank)
{
    return longest_first(blockIdx.x, heads, blocks, cus, bh, rank);
}

}  // namespace
