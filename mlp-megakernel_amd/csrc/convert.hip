// Element conversions of several tensors in one launch: the casts and zero
// padding around the fused kernels (x, the weights and dL/dout on the way in,
// dW on the way out), which as framework operations are a launch or two per
// tensor.
#include "device_common.h"
#include "host_common.h"

namespace mlpmk {
namespace convert {

constexpr int kMaxTensors = 16;
struct Item {
  const void* src;
  void* dst;
  uint32_t first;             // first workgroup of this tensor in the launch (2048 destination elements each)
  uint32_t src_rows, src_cols, dst_cols;
  uint32_t n;                 // destination elements
  int src_dt, dst_dt;
  int raw;                    // both the same 16-bit type: the bits as they are
  int flat;                   // equal columns: element i of dst is element i of src below src_rows * src_cols
  int vec;                    // flat and src 16-byte aligned
};
struct Params {
  int n;
  Item t[kMaxTensors];
};

__device__ __forceinline__ float load1(const void* p, uint32_t i, int dt) {
  if (dt == MLPMK_DTYPE_F32) return static_cast<const float*>(p)[i];
  if (dt == MLPMK_DTYPE_F16) return (float)static_cast<const _Float16*>(p)[i];
  return (float)static_cast<const __bf16*>(p)[i];
}
__device__ __forceinline__ void store1(void* p, uint32_t i, int dt, float v) {
  if (dt == MLPMK_DTYPE_F32) static_cast<float*>(p)[i] = v;
  else if (dt == MLPMK_DTYPE_F16) static_cast<_Float16*>(p)[i] = (_Float16)v;
  else static_cast<__bf16*>(p)[i] = (__bf16)v;
}

__global__ __launch_bounds__(256) void convert_kernel(Params p) {
  // One tensor per workgroup, so that its description stays in scalar
  // registers; 8 destination elements per thread.
  int k = 0;
  while (k + 1 < p.n && blockIdx.x >= p.t[k + 1].first) ++k;
  const Item& t = p.t[k];
  const uint32_t e = ((blockIdx.x - t.first) * 256 + threadIdx.x) * 8;
  if (e >= t.n) return;
  const uint32_t have = t.src_rows * t.src_cols;
  float v[8] = {};
  if (t.raw && !(t.vec && e + 8 <= have)) {
    const uint16_t* s = static_cast<const uint16_t*>(t.src);
    uint32_t r = e / t.dst_cols, c = e - r * t.dst_cols;
    typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
    u16x8 b = {};
    if (t.dst_cols % 8 == 0 && r < t.src_rows && c + 8 <= t.src_cols) {
      // Padding to whole pieces (every caller's): eight elements of one row, at
      // any element boundary of the source, in one load.  Element by element in
      // and out, 524,288 x 63 bf16 into 64 columns took 53 us, this way 29 (fp32 56 and 44).
      __builtin_memcpy(&b, s + r * t.src_cols + c, 16);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (r < t.src_rows && c < t.src_cols) b[j] = s[r * t.src_cols + c];
        if (++c == t.dst_cols) {
          c = 0;
          ++r;
        }
      }
    }
    uint16_t* d = static_cast<uint16_t*>(t.dst);
    if (e + 8 <= t.n) {  // dst is 16-byte aligned
      reinterpret_cast<u16x8*>(d)[e / 8] = b;
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (e + j < t.n) d[e + j] = b[j];
    }
    return;
  }
  if (t.flat) {
    if (t.vec && e + 8 <= have) {
      if (t.src_dt == MLPMK_DTYPE_F32) {
        const f32x4 a = reinterpret_cast<const f32x4*>(t.src)[e / 4], b = reinterpret_cast<const f32x4*>(t.src)[e / 4 + 1];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[j] = a[j];
          v[4 + j] = b[j];
        }
      } else {
        const f16x8 a = reinterpret_cast<const f16x8*>(t.src)[e / 8];
        if (t.raw && e + 8 <= t.n) {
          reinterpret_cast<f16x8*>(t.dst)[e / 8] = a;
          return;
        }
        const bool bf = t.src_dt == MLPMK_DTYPE_BF16;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = bf ? elem_to_f32<true>(a[j]) : elem_to_f32<false>(a[j]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (e + j < have) v[j] = load1(t.src, e + j, t.src_dt);
    }
  } else {
    uint32_t r = e / t.dst_cols, c = e - r * t.dst_cols;
    if (t.src_dt == MLPMK_DTYPE_F32 && t.dst_cols % 8 == 0 && r < t.src_rows && c + 8 <= t.src_cols) {
      __builtin_memcpy(v, static_cast<const float*>(t.src) + r * t.src_cols + c, 32);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (r < t.src_rows && c < t.src_cols) v[j] = load1(t.src, r * t.src_cols + c, t.src_dt);
        if (++c == t.dst_cols) {
          c = 0;
          ++r;
        }
      }
    }
  }
  if (e + 8 <= t.n) {  // dst is 16-byte aligned
    if (t.dst_dt == MLPMK_DTYPE_F32) {
      reinterpret_cast<f32x4*>(t.dst)[e / 4] = f32x4{v[0], v[1], v[2], v[3]};
      reinterpret_cast<f32x4*>(t.dst)[e / 4 + 1] = f32x4{v[4], v[5], v[6], v[7]};
    } else if (t.dst_dt == MLPMK_DTYPE_BF16) {
      reinterpret_cast<f16x8*>(t.dst)[e / 8] = pack8<true>(v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]);
    } else {
      reinterpret_cast<f16x8*>(t.dst)[e / 8] = pack8<false>(v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]);
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (e + j < t.n) store1(t.dst, e + j, t.dst_dt, v[j]);
  }
}

}  // namespace convert

// Arguments checked by the C ABI (api.cpp), except for the sizes a launch
// takes: MLPMK_ERR_UNSUPPORTED_SHAPE past 2^31 elements in all.
int convert_dispatch(int n, const void* const* src, const int* src_dt, void* const* dst, const int* dst_dt,
                     const int64_t* shapes, hipStream_t st) {
  convert::Params p = {};
  int64_t blocks = 0;
  for (int i = 0; i < n; ++i) {
    const int64_t sr = shapes[4 * i], sc = shapes[4 * i + 1], dr = shapes[4 * i + 2], dc = shapes[4 * i + 3];
    if (sr > 0x7fffffff || sc > 0x7fffffff || dr > 0x7fffffff || dc > 0x7fffffff || sr * sc > 0x7fffffff ||
        dr * dc > 0x7fffffff)
      return fail(MLPMK_ERR_UNSUPPORTED_SHAPE, "tensor %d has 2^31 elements or more", i);
    if (dr * dc == 0) continue;
    convert::Item& t = p.t[p.n++];
    t = {src[i], dst[i], (uint32_t)blocks, (uint32_t)sr, (uint32_t)sc, (uint32_t)dc, (uint32_t)(dr * dc), src_dt[i],
         dst_dt[i], src_dt[i] == dst_dt[i] && src_dt[i] != MLPMK_DTYPE_F32, sc == dc, sc == dc && (reinterpret_cast<uintptr_t>(src[i]) & 15u) == 0};
    blocks += (dr * dc + 2047) / 2048;
  }
  if (blocks == 0) return MLPMK_OK;
  int cus = 0;
  const int rc = current_device_cus(&cus);
  if (rc != MLPMK_OK) return rc;
  (void)hipGetLastError();
  hipLaunchKernelGGL(convert::convert_kernel, dim3((unsigned)blocks), dim3(256), 0, st, p);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? MLPMK_OK : hip_fail(e, "conversion kernel launch");
}

}  // namespace mlpmk
