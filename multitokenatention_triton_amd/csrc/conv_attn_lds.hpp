// What the fused conv-attention kernel (conv_attn_mfma.hpp) and the scores kernel (conv_scores_mfma.hpp) share: LDS accesses issued from
// assembly, loops over compile-time indexes.
#pragma once

#include <type_traits>
#include <utility>

#include "conv_attn.hpp"
#include "mfma.hpp"

namespace {
using namespace mta;

typedef __attribute__((address_space(3))) void lds_void_t;
typedef const __attribute__((address_space(1))) void glb_void_t;
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));

constexpr int F_BK = 64;   // keys per iteration

// LDS accesses issued from assembly: the compiler neither reorders them nor waits for the asynchronous copy in flight
// ahead of them (it cannot tell a read of the score tile from the copy's target), and the wait points are placed by
// hand.  LDS operations of a wavefront complete in order, so "at most n operations outstanding" names the oldest ones
// as complete; a loaded value is tied to the wait that covers it through an in/out operand.
__device__ __forceinline__ unsigned lds_addr(const void *p) { return (unsigned)(uintptr_t)(lds_void_t *)p; }
__device__ __forceinline__ u32x4_t lds_read16_at(unsigned addr, int off)
{
    u32x4_t v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(off) : "memory");
    return v;
}
__device__ __forceinline__ void lds_write16_at(unsigned addr, int off, u32x4_t v)
{
    asm volatile("ds_write_b128 %0, %1 offset:%2" : : "v"(addr), "v"(v), "n"(off) : "memory");
}
template <int N> __device__ __forceinline__ void lds_wait_upto(u32x4_t &v)
{
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(v) : "n"(N) : "memory");
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
// The score phase of either kernel writes the scores of 16-key blocks cb-1 and cb (cb odd, both row blocks: two writes) right
// after step (cb+1)*KS + LAG - 1 of its score phase; the last pair after the loop.  Number of those writes issued at the
// end of a step in [lo, hi).
constexpr int score_writes_between(int lo, int hi, int KS, int NCB, int LAG, int writes)
{
    int c = 0;
    for (int cb = 1; cb + 1 < NCB; cb += 2) {
        const int s = (cb + 1) * KS + LAG - 1;
        if (s >= lo && s < hi) c += writes;
    }
    return c;
}

// Inside a rarely taken, wavefront-uniform `if`: keeps it a branch.  Without it the compiler turns the masks of the
// diagonal key blocks into selects that every key block executes (a third of the attention kernel's vector
// instructions).
#define MTA_KEEP_BRANCH() asm volatile("" ::: "memory")

// Returns its argument, opaquely: what is derived from the result cannot be hoisted out of the block that computes it.
__device__ __forceinline__ int opaque_lane(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}
}  // namespace
