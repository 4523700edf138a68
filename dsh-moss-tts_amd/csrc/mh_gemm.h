// mh_gemm.h -- what the two matrix-core GEMMs (gemm_mfma.hip, gemm_tile.hip) share.
#pragma once

#include "mh_ops.h"

namespace mh {

typedef float floatx4 __attribute__((ext_vector_type(4)));

// x = hi + lo: hi rounds toward zero (v_cvt_pkrtz, two values per
// instruction), so x - hi is exact in fp32; lo keeps the next ~10 bits.
__device__ __forceinline__ void split_hi_lo(const float (&x)[8], half8 &hi, half8 &lo) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const auto h = __builtin_amdgcn_cvt_pkrtz(x[2 * i], x[2 * i + 1]);
        const auto l = __builtin_amdgcn_cvt_pkrtz(x[2 * i] - (float)h[0], x[2 * i + 1] - (float)h[1]);
        hi[2 * i] = (_Float16)h[0];
        hi[2 * i + 1] = (_Float16)h[1];
        lo[2 * i] = (_Float16)l[0];
        lo[2 * i + 1] = (_Float16)l[1];
    }
}

// Operands through buffer resources: the lane's byte offset at its first block is one
// VGPR per operand; the block within a chunk is the instruction's immediate offset and
// the chunk base and column subtile an SGPR offset, so a load costs no address
// arithmetic.  A load past a resource's last byte returns 0 instead of faulting, so
// every load is unconditional (blocks past the last one, or rows past M, are read and
// never used).
typedef __amdgpu_buffer_rsrc_t rsrc_t;
constexpr int kRsrcWord3 = 0x00020000;  // gfx9 raw buffer word 3 (32-bit data format)

__device__ __forceinline__ rsrc_t make_rsrc(const void *p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, kRsrcWord3);
}

// gemm_tile.hip: 64 x 64 tiles for many rows; tile_gemm_fits says whether it takes the call
bool tile_gemm_fits(const GemmArgs &g, Epilogue epi);
hipError_t launch_gemm_tile(const GemmArgs &g, Epilogue epi, KvType kv, hipStream_t s);

}  // namespace mh
