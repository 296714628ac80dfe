// Rows of 64 channels that move between memory and LDS as whole lines, eight lanes to a row, and are used as matrix fragments.
// (A load in the order of a fragment, four lanes on four rows, is four lookups of a compute unit's vector cache per four lanes:
// 28 ns for a wavefront's 16 bytes per lane instead of 9, and 28 instead of 20 to store.)
#pragma once
#include "frag.hpp"

namespace wkv {

// 16-byte pieces of rows of 64 channels.  A fragment read takes piece 4pr + g of 16 rows: eight pieces of two rows lie in
// different banks, so the pieces of a pair of rows are permuted by the pair's number.
__device__ __forceinline__ int piece_slot(int row, int piece) { return 8 * row + (piece ^ ((row >> 1) & 7)); }
// the bytes at a 32-bit offset from a wavefront-uniform address: no 64-bit address per load
__device__ __forceinline__ const bf16x8& piece_at(const __bf16* base, unsigned bytes) {
    return *reinterpret_cast<const bf16x8*>(reinterpret_cast<const char*>(base) + bytes);
}
__device__ __forceinline__ bf16x8& piece_at(__bf16* base, unsigned bytes) {
    return *reinterpret_cast<bf16x8*>(reinterpret_cast<char*>(base) + bytes);
}
// 16 bytes there through the L2 (see store_through in frag.hpp), as a store that the compiler counts: behind one that it does not see it would wait
// for what was requested before it to be written as well.  base: the same for a wavefront; bytes: up to 2^32 - 32, as
// far as piece_at reaches (a descriptor holds at most 2^32 - 1 bytes).
template <class V>
__device__ __forceinline__ void store_through_at(void* base, unsigned bytes, V v) {
    static_assert(sizeof(V) == 16, "one access");
    typedef unsigned words __attribute__((ext_vector_type(4)));
    constexpr int DEVICE_SCOPE = 16, FOUR_GIB = -1;
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(words, v), __builtin_amdgcn_make_buffer_rsrc(base, 0, FOUR_GIB, 0x00020000), bytes, 0, DEVICE_SCOPE);
}
// LDS instructions of one wavefront run in their order: what its lanes have written, the others of them may read
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ bf16x4 half_of(const bf16x8 v, int hlf) {
    return hlf ? __builtin_shufflevector(v, v, 4, 5, 6, 7) : __builtin_shufflevector(v, v, 0, 1, 2, 3);
}
__device__ __forceinline__ bf16x8 join(const bf16x4 lo, const bf16x4 hi) { return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7); }

}  // namespace wkv
