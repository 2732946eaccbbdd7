// Buffer-to-LDS copies ordered by hand (the many-token GEMM kernels).
#pragma once

#include "common.h"

namespace rsllm_hip {

// A raw-buffer resource in scalar registers (base, size in bytes).
typedef uint32_t bl_rsrc __attribute__((ext_vector_type(4)));
__device__ __forceinline__ bl_rsrc bl_make_rsrc(const void *p, uint32_t bytes) {
    const uint64_t a = (uint64_t)(size_t)p;
    return bl_rsrc{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
                   (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32) & 0xFFFF),
                   (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}
// LDS byte address of a pointer into the workgroup's LDS.
__device__ __forceinline__ uint32_t bl_lds(const void *p) {
    return (uint32_t)(size_t)(const __attribute__((address_space(3))) void *)p;
}
// 16 bytes per lane from the buffer to LDS: lane i's bytes at voff + soff go to lds
// + 16 i (lds uniform); a lane whose bytes lie past the resource moves zeros
// without an access. Written by hand, so the compiler adds no wait for it
// before LDS reads (with the builtin it waits for every copy in flight):
// bl_barrier orders each copy against its readers. M0 is restored; the
// memory clobber keeps LDS accesses on their side.
__device__ __forceinline__ void bl_dma16(const bl_rsrc &r, uint32_t voff, uint32_t soff, uint32_t lds) {
    const uint32_t ls = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds);
    const uint32_t so = (uint32_t)__builtin_amdgcn_readfirstlane((int)soff);
    uint32_t saved;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\t"
                 "buffer_load_dwordx4 %1, %2, %4 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(saved)
                 : "v"(voff), "s"(r), "s"(ls), "s"(so)
                 : "memory");
}
// All but this wavefront's N newest copies have landed and its LDS accesses
// are done, then everyone's.
template <int N> __device__ __forceinline__ void bl_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

}  // namespace rsllm_hip
