// What the convolution kernels share: the geometry of a layer, range-checked
// buffer loads and the forward epilogue.
#pragma once

#include "common.hpp"

namespace ach {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr unsigned kOOB = 0x80000000u;  // buffer offset that reads as 0

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *p, unsigned bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes,
                                             0x00020000);
}

// element offset -> byte offset, or the out-of-range offset when invalid
__device__ __forceinline__ int boff(bool ok, int elem)
{
    return ok ? elem * 4 : (int)kOOB;
}

// the builtin returns the loaded dword as an integer: reinterpret its bits
__device__ __forceinline__ float bload(__amdgpu_buffer_rsrc_t r, int byte_off)
{
    return __int_as_float((int)__builtin_amdgcn_raw_buffer_load_b32(r, byte_off, 0, 0));
}

// The same with a wave-uniform byte offset in the instruction's scalar
// offset operand (an SGPR): loaders with loop-invariant per-thread offsets
// add the k-tile's uniform advance there instead of in one VGPR per load.
// Callers keep voff + soff inside the buffer for every in-range voff (the
// prefetch past the last k-tile re-reads the last tile), so the address is
// valid whether or not the range check includes the scalar offset; an
// out-of-range voff (>= 2^31) reads zero either way.
__device__ __forceinline__ float bload_so(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff)
{
    return __int_as_float(
        (int)__builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, 0));
}

__device__ __forceinline__ float4 bload4(__amdgpu_buffer_rsrc_t r, int byte_off)
{
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, byte_off, 0, 0);
    return make_float4(__int_as_float((int)v[0]), __int_as_float((int)v[1]),
                       __int_as_float((int)v[2]), __int_as_float((int)v[3]));
}

__device__ __forceinline__ float4 bload4_so(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff)
{
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0);
    return make_float4(__int_as_float((int)v[0]), __int_as_float((int)v[1]),
                       __int_as_float((int)v[2]), __int_as_float((int)v[3]));
}

struct ConvGeom {
    int B, C, H, W;    // input
    int F, KS, S, P;   // filters, kernel, stride, pad
    int OH, OW;
    FastDiv dkk, dks;  // division by KS*KS and by KS
};

// ===========================================================================
// Output epilogue of the forward GEMMs: the layer's bias and activation
// applied to each finished sum, as the separate passes would apply them
// (IOData.addBias then activate, IOData.c:43-72), in one branch-free form
// so the kernel keeps a single epilogue.  Kernels instantiated with the
// epilogue (EPI) hold every accumulator in VGPRs at the end; tiles of at
// most 128 rows keep that within their occupancy.
//   v += bias[m]            (no bias: v + -0.0f, which is v for every v)
//   v = v > 0 ? v : (float)(slope * (double)v)
// slope 0.1 is act_forward's leaky; slope 0 gives relu's v * (v > 0)
// (+-0 with the sign of v, NaN kept); slope 1 is linear.  The default
// (no bias, slope 1) leaves v unchanged.  The logistic activation, with
// its double exp, stays a separate pass.
struct Epi {
    const float *bias = nullptr;
    double slope = 1.0;
    bool active() const { return bias != nullptr || slope != 1.0; }
    __device__ __forceinline__ float apply(float v, int m) const
    {
        const float b = bias ? bias[m] : -0.0f;
        v = v + b;
        return v > 0.f ? v : (float)(slope * (double)v);
    }
};

}  // namespace ach
