// Device helpers of the LDS-tiled kernels: panel layout and range-checked operand access.

#pragma once

#include <hip/hip_runtime.h>

namespace ctg {

typedef unsigned int uint2_t __attribute__((ext_vector_type(2)));
typedef double double2_t __attribute__((ext_vector_type(2)));

constexpr int TK = 16;                       // k-panel
// A panel in LDS lies in fragment order: entry (16 sub + i, 4 step + q) of a 64 x 16 panel at
// step T_STEP + (sub / 2) T_PAIR + q T_Q + 2 i + sub % 2, so that one 16-byte read gives a lane its entries
// of two sub-tiles. The paddings (T_Q 34 for 32, T_STEP 280 for 272) are for the writes of both operand
// layouts; bank conflicts still take a fifth of a busy CU's cycles.
constexpr int T_Q = 34, T_PAIR = 4 * T_Q, T_STEP = 2 * T_PAIR + 8, TPANEL = (TK / 4) * T_STEP;
// an offset past the end of every operand (their extents stay below 2^30 bytes): a load there returns
// zero and a store is dropped
constexpr int TILE_OOB = (int)0x80000000;

__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

// an operand of the current panel: address and bytes left from there, uniform over the workgroup. The
// descriptor is put together where it is used, from values that the compiler knows to be uniform (a
// descriptor carried round the loop ends up in vector registers, and every load in a loop over its
// distinct values). Loads past the end return zero, dword by dword.
struct TileOperand
{
	uint64_t p;
	int32_t bytes;
	__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc() const
	{
		const uint64_t q = (uint64_t)(uint32_t)uni((int)(uint32_t)p) | ((uint64_t)(uint32_t)uni((int)(uint32_t)(p >> 32)) << 32);
		return __builtin_amdgcn_make_buffer_rsrc((void*)(uintptr_t)q, 0, uni(bytes), 0x00027000);
	}
	__device__ __forceinline__ void advance(int step) { p += (uint64_t)step; bytes -= step; }
};

__device__ __forceinline__ double2_t buf_load2(__amdgpu_buffer_rsrc_t r, int voff)
{
	return __builtin_bit_cast(double2_t, __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0));
}

}  // namespace ctg
