/* blocks.hpp -- 4x4 blocks and their rows in the storage precisions of matrices and
 * preconditioner factors (FP64, FP32, bfloat16); arithmetic is FP64 throughout.
 */
#ifndef FVX_BLOCKS_HPP
#define FVX_BLOCKS_HPP

#include "fvx_internal.hpp"
#include "wave.hpp"

namespace fvx {

template <class VT> __device__ __forceinline__ void load_row(const VT* p, double* v);
template <> __device__ __forceinline__ void load_row<double>(const double* p, double* v)
{
	const double2 a = reinterpret_cast<const double2*>(p)[0];
	const double2 b = reinterpret_cast<const double2*>(p)[1];
	v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
}
template <> __device__ __forceinline__ void load_row<float>(const float* p, double* v)
{
	const float4 a = *reinterpret_cast<const float4*>(p);
	v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
/// bfloat16 rows: 4 x 2 bytes (8-byte aligned: rows start at multiples of 4 values)
__device__ __forceinline__ double bf16_value(unsigned int h)
{
	return (double)__uint_as_float(h << 16);
}
template <> __device__ __forceinline__ void load_row<bf16>(const bf16* p, double* v)
{
	const uint2 w = *reinterpret_cast<const uint2*>(p);
	v[0] = bf16_value(w.x & 0xffffu); v[1] = bf16_value(w.x >> 16);
	v[2] = bf16_value(w.y & 0xffffu); v[3] = bf16_value(w.y >> 16);
}
/// FP64 -> FP32 (rounded) -> bfloat16, rounded to nearest even; NaN stays NaN
__device__ __forceinline__ unsigned int bf16_bits(double x)
{
	const unsigned int u = __float_as_uint((float)x);
	if((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
	return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}
template <class VT> __device__ __forceinline__ void put_row(VT* p, const double* v);
template <> __device__ __forceinline__ void put_row<bf16>(bf16* p, const double* v)
{
	*reinterpret_cast<uint2*>(p) = make_uint2(bf16_bits(v[0]) | (bf16_bits(v[1]) << 16),
	                                          bf16_bits(v[2]) | (bf16_bits(v[3]) << 16));
}
template <> __device__ __forceinline__ void put_row<double>(double* p, const double* v)
{
	reinterpret_cast<double2*>(p)[0] = make_double2(v[0], v[1]);
	reinterpret_cast<double2*>(p)[1] = make_double2(v[2], v[3]);
}
template <> __device__ __forceinline__ void put_row<float>(float* p, const double* v)
{
	*reinterpret_cast<float4*>(p) = make_float4((float)v[0], (float)v[1], (float)v[2],
	                                            (float)v[3]);
}
template <class VT> __device__ __forceinline__ void load_block(const VT* p, double* b)
{
	for(int r = 0; r < 4; r++) load_row<VT>(p + 4*r, b + 4*r);
}
template <class VT> __device__ __forceinline__ void put_block(VT* p, const double* b)
{
	for(int r = 0; r < 4; r++) put_row<VT>(p + 4*r, b + 4*r);
}

__device__ __forceinline__ double dot4(const double* a, const double* x)
{
	return a[0]*x[0] + a[1]*x[1] + a[2]*x[2] + a[3]*x[3];
}

/// Value of lane k of the quad, on every lane of the quad.
template <int K> __device__ __forceinline__ double quad_bcast(double v)
{
	return dpp_d<K*0x55>(v);
}

}
#endif
