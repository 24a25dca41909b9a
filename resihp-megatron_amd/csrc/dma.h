// Direct HBM -> LDS loads: the buffer view and the 1 KB wave load the GEMM and
// routing kernels stage their operands with.  The loads are inline assembly,
// so each kernel waits for them itself (s_waitcnt vmcnt).
#pragma once

#include "rhp_common.h"

namespace rhp {
namespace {

typedef int i32x4_t __attribute__((ext_vector_type(4)));

struct Rsrc {
    i32x4_t d;
};
__device__ __forceinline__ Rsrc make_dma_rsrc(const void* base, int64_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    Rsrc r;
    r.d[0] = __builtin_amdgcn_readfirstlane(static_cast<int>(a));
    r.d[1] = __builtin_amdgcn_readfirstlane(static_cast<int>(a >> 32));
    r.d[2] = __builtin_amdgcn_readfirstlane(static_cast<int>(bytes > 0x7ffffff0 ? 0x7ffffff0 : bytes));
    r.d[3] = 0x00020000;
    return r;
}
// 16 bytes per lane from the buffer at voff + soff into LDS at lds + 16 * lane.
__device__ __forceinline__ void dma16(const Rsrc& r, uint32_t voff, uint32_t soff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %3\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
                 :
                 : "v"(voff), "s"(r.d), "s"(__builtin_amdgcn_readfirstlane(soff)),
                   "s"(__builtin_amdgcn_readfirstlane(lds))
                 : "memory");
}

}  // namespace
}  // namespace rhp
