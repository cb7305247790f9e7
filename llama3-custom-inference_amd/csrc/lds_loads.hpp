// Loads from global memory straight into LDS that the compiler does not see, the waits for them, and the bare
// workgroup barrier: what a ring of stages needs whose newer loads stay in flight across a barrier.
#pragma once

#include "attn_mfma_core.hpp"

namespace l3 {

typedef uint32_t srd_t __attribute__((ext_vector_type(4)));   // a buffer resource: base, no range limit, raw

__device__ __forceinline__ srd_t make_srd(const void* base) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    srd_t r;
    r.x = uint32_t(wave_uniform(int(uint32_t(a))));
    r.y = uint32_t(wave_uniform(int(uint32_t(a >> 32) & 0xffffu)));
    r.z = 0xffffffffu;
    r.w = 0x00020000u;
    return r;
}

__device__ __forceinline__ uint32_t lds_address(const void* p) {
    return uint32_t(reinterpret_cast<uintptr_t>(L3_LDS_PTR(const unsigned char, p)));
}

// 16 bytes per lane from base + lane_off + uniform_off to LDS address lds + lane * 16 (lds is wave-uniform).
// The compiler does not see the load (it would wait for every one of them before it reads LDS at the head of a
// loop): whoever reads that LDS waits for it with wait_loads().
template <bool STREAM>
__device__ __forceinline__ void load_to_lds(const srd_t& base, uint32_t lds, uint32_t lane_off, int uniform_off) {
    if constexpr (STREAM) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
                     ::"s"(lds), "v"(lane_off), "s"(base), "s"(uniform_off) : "memory");
    } else {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     ::"s"(lds), "v"(lane_off), "s"(base), "s"(uniform_off) : "memory");
    }
}

// Until at most NEWER of this wavefront's vector memory operations are outstanding.
template <int NEWER>
__device__ __forceinline__ void wait_loads() {
    static_assert(NEWER < 64, "six bits");
    __builtin_amdgcn_s_waitcnt((NEWER & 15) | ((NEWER >> 4) << 14) | 0x0F70);
}
// The bare barrier, for wavefronts that read no LDS.
__device__ __forceinline__ void barrier() { asm volatile("s_barrier" ::: "memory"); }
// For wavefronts that do: behind it a stage may be loaded over, so what they have asked of LDS has to have arrived.  (The
// compiler waits where the values are used, and may move that use behind a barrier; it costs nothing where it did not.)
__device__ __forceinline__ void barrier_after_lds() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

}  // namespace l3
