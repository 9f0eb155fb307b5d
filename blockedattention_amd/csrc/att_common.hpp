// What the one-pass attention (attention.hip) and its backward (attention_backward.hip) share: counted LDS operand
// reads, the rows of the per-query arrays.
#pragma once
#include <type_traits>
#include <utility>

#include "row_pieces.hpp"

namespace ba {

constexpr int kAttKeys = 64;                          // keys (backward: or queries) staged in LDS at a time

// Rows past a segment's last one that a kernel asks for, at most: the pipelines request two blocks ahead, where rows that
// do not exist read as zeros by their byte offset, which must not wrap.  Dimensions and areas of a plan's segments are below
// 2^30 (the scheduler refuses others) and head dimensions at most 128: every such segment fits.
constexpr int kAttAhead = 3 * kAttKeys;
__host__ __device__ constexpr bool att_offsets_fit(int64_t rows, int K) { return (rows + kAttAhead) * K < (int64_t(1) << 31); }
static_assert(att_offsets_fit((1 << 30) - 1, 1) && att_offsets_fit(((1 << 30) - 1) / 128, 128));
static_assert(!att_offsets_fit((int64_t(1) << 31) - kAttAhead, 1) && !att_offsets_fit((1 << 24) - kAttAhead, 128));

// LDS operand reads as inline assembly, so that kAttRing of them are in flight under the matrix instructions
// (left to itself the compiler, short of registers, issues each read right before its use and every matrix
// instruction waits a full LDS round trip).  The compiler does not count these reads: lds_wait<n> waits until at
// most n of them are outstanding and hands the register on, so the use cannot move above the wait.  Counting is
// conservative when other LDS or scalar loads are in flight: the counter is then higher, the wait longer.
template <int OFF> __device__ __forceinline__ void lds_read128(u32x4 &dst, uint32_t addr) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF) : "memory");
}
template <int N> __device__ __forceinline__ void lds_wait(u32x4 &x) {
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(x) : "n"(N) : "memory");
}
// Reads that turn out not to be needed arrive before their registers are free for something else.  One statement that names
// them all and hands none on: of one for each the compiler copied the registers before the first wait.
__device__ __forceinline__ void lds_drain(const u32x4 (&x)[4]) {
    asm volatile("s_waitcnt lgkmcnt(0)" : : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]) : "memory");
}
// The same for the transposing read: four elements of one column from each of two groups of rows NEXT bytes apart.
template <int OFF, int NEXT> __device__ __forceinline__ void lds_read_tr(u32x2 &lo, u32x2 &hi, uint32_t addr) {
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo) : "v"(addr), "n"(OFF) : "memory");
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi) : "v"(addr), "n"(OFF + NEXT) : "memory");
}
template <int N> __device__ __forceinline__ void lds_wait_tr(u32x2 &lo, u32x2 &hi) {
    asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(lo), "+v"(hi) : "n"(N) : "memory");
}
template <typename F, int... I> __device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F> __device__ __forceinline__ void static_for(F &&f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}
__device__ __forceinline__ uint32_t lds_offset(const void *p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)p;
}

// The operands that a wavefront keeps for a whole loop have arrived before the loop: without a use in front of it the
// compiler waits for their loads at their first use inside, in every iteration, and there the wait is for the loads of
// the next block, issued a moment before.
template <int A, int B> __device__ __forceinline__ void arrived(u32x4 (&x)[A][B]) {
#pragma unroll
    for (int i = 0; i < A; ++i)
#pragma unroll
        for (int k = 0; k < B; ++k) asm volatile("" : "+v"(x[i][k]));
}

// Barrier that waits for this wavefront's LDS traffic only (the loads of the next block stay in flight).
__device__ __forceinline__ void att_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// a * b + c for a, b below 2^24: one instruction
__device__ __forceinline__ uint32_t mad24(uint32_t a, uint32_t b, uint32_t c) { return __umul24(a, b) + c; }

// Where the rows of a segment lie in a per-query array of the backward pass: ceil(Dm1 / min_K) floats per head, row r
// of segment g at ceil(off1 / min_K) + r.  Segments do not overlap there because none has fewer than min_K elements a
// row (segments without keys, which min_K does not count, have no entry).  The arrays are sized from the host's summary:
// a kernel gets its min_K with the launch and touches them only if the plan has the same.
__host__ __device__ inline int64_t att_rows_per_head(int min_K, int64_t Dm1) {
    const int64_t k = min_K > 1 ? min_K : 1;
    return (Dm1 + k - 1) / k;
}
__device__ __forceinline__ int64_t att_row_base(int min_K, int64_t Dm1, int64_t h, int64_t off1) {
    return h * att_rows_per_head(min_K, Dm1) + att_rows_per_head(min_K, off1);
}

}  // namespace ba
