// fp8 (OCP e4m3fn) quantisation of token embeddings, per token or per tensor
// (reference fp8.py:35-59): scale = max(amax, 1e-6) / 448 in fp32, bytes =
// e4m3(clamp(x / scale, +-448)), round to nearest even.
//
// What bounds it: HBM, each element read once (per tensor: twice, the second
// time partly from the memory-side cache) and one byte written. The same
// steps as separate elementwise passes (abs, amax, widen, divide, clamp, cast)
// move 11x the bytes: on 1,030,000 bf16 rows of d = 128 (396 MB of input and
// output) they take 860 us.
//
// The bytes equal those of the pass-by-pass form (IEEE division, then the
// cast). The quotient takes five instructions instead of the ten of a full
// fp32 division: with r = RN(1 / scale), q = RN(x r) and f = RN(q + (x - q scale) r),
// f is a faithful quotient and RN(f + (x - f scale) r) the correctly rounded one
// (Markstein, "Computation of elementary functions on the IBM RISC
// System/6000 processor", 1990) as long as nothing in it under- or overflows.
// scale is at least 1e-6 / 448 = 2.2e-9, so the remainders are normal numbers
// whenever |x / scale| reaches 2^-12, and below 2^-10 every quotient rounds to
// a zero of x's sign anyway; scales of 1e30 and above (infinite and NaN rows
// among them) take the full division.
#include "lik_common.h"

namespace lik {

constexpr float kE4m3Max = 448.0f;

// |x| as integer bits that order as the magnitudes do, NaN above everything.
template <int EK>
__device__ __forceinline__ uint32_t chunk_absmax(const u32x4& v, uint32_t m) {
  if constexpr (EK == EK_F32) {
#pragma unroll
    for (int i = 0; i < 4; ++i) m = max(m, v[i] & 0x7fffffffu);
    return m;
  } else {  // two 16-bit maxima side by side
    typedef unsigned short us2 __attribute__((ext_vector_type(2)));
    us2 a = __builtin_bit_cast(us2, m);
#pragma unroll
    for (int i = 0; i < 4; ++i) a = __builtin_elementwise_max(a, __builtin_bit_cast(us2, v[i] & 0x7fff7fffu));
    return __builtin_bit_cast(uint32_t, a);
  }
}

template <int EK>
__device__ __forceinline__ uint32_t absmax2(uint32_t a, uint32_t b) {
  if constexpr (EK == EK_F32) return max(a, b);
  typedef unsigned short us2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(us2, a), __builtin_bit_cast(us2, b)));
}

// The magnitude those bits stand for, at least 1e-6 rounded to the input type.
template <int EK>
__device__ __forceinline__ float absmax_value(uint32_t m) {
  float f;
  if constexpr (EK == EK_F32) f = __uint_as_float(m);
  else {
    const uint32_t h = max(m & 0xffffu, m >> 16);
    f = EK == EK_BF16 ? __uint_as_float(h << 16) : f16_to_f32((uint16_t)h);
  }
  const float lo = EK == EK_F32 ? 1e-6f : EK == EK_BF16 ? (float)(__bf16)1e-6f : (float)(_Float16)1e-6f;
  return f < lo ? lo : f;  // NaN stays
}

__device__ __forceinline__ float scale_of(float amax) { return amax * (1.0f / kE4m3Max); }

// e4m3fn of a value that may be NaN (0x7f with its sign); |f| <= 448 otherwise.
__device__ __forceinline__ uint32_t e4m3_any(float f) {
  if (f != f) return 0x7fu | ((__float_as_uint(f) >> 24) & 0x80u);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(f, 0.f, 0, false) & 0xffu;
}

__device__ __forceinline__ float quotient(float x, float s, float r) {
  const float q = x * r;
  const float f = fmaf(fmaf(-q, s, x), r, q);
  const float y = fmaf(fmaf(-f, s, x), r, f);
  return __builtin_amdgcn_fmed3f(copysignf(y, x), -kE4m3Max, kE4m3Max);
}

// The bytes of one 16-byte input chunk: 8 elements -> two words, fp32: 4 -> one.
template <int EK>
__device__ __forceinline__ void quant_chunk(const u32x4& v, float s, float r, bool plain, uint32_t* w) {
  constexpr int N = EK == EK_F32 ? 4 : 8;
  float x[N];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (EK == EK_F32) x[i] = __uint_as_float(v[i]);
    else if constexpr (EK == EK_BF16) { x[2 * i] = bf16lo_to_f32(v[i]); x[2 * i + 1] = bf16hi_to_f32(v[i]); }
    else { x[2 * i] = f16_to_f32((uint16_t)(v[i] & 0xffffu)); x[2 * i + 1] = f16_to_f32((uint16_t)(v[i] >> 16)); }
  }
#pragma unroll
  for (int g = 0; g < N / 4; ++g) {
    const float* y = x + 4 * g;
    if (plain) {
      int p = __builtin_amdgcn_cvt_pk_fp8_f32(quotient(y[0], s, r), quotient(y[1], s, r), 0, false);
      w[g] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(quotient(y[2], s, r), quotient(y[3], s, r), p, true);
    } else {
      uint32_t b = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float q = y[e] / s;
        q = q != q ? q : fminf(fmaxf(q, -kE4m3Max), kE4m3Max);
        b |= e4m3_any(q) << (8 * e);
      }
      w[g] = b;
    }
  }
}

template <int EK>
__device__ __forceinline__ void store_bytes(uint8_t* p, const uint32_t* w) {
  if constexpr (EK == EK_F32) *(uint32_t*)p = w[0];
  else *(u32x2*)p = u32x2{w[0], w[1]};
}

// One scale per row: 16 lanes a row, the row's 16-byte chunks lane + 16 k kept
// in registers between the maximum and the conversion, U rows a group with
// all their loads issued first (a wavefront reads 4 U consecutive rows).
template <int EK, int NCH>
__global__ void __launch_bounds__(256) quant_rows_kernel(const char* x, int64_t rows, int dim, uint8_t* out,
                                                         float* scale) {
  constexpr int EPC = EK == EK_F32 ? 4 : 8;
  constexpr int U = NCH == 1 ? 4 : NCH == 2 ? 2 : 1;
  const int q = threadIdx.x & 15, g = (threadIdx.x >> 4) & 3;
  const int64_t rowb = (int64_t)dim * (16 / EPC);
  const int64_t nblk = (rows + 16 * U - 1) / (16 * U);
  for (int64_t blk = blockIdx.x; blk < nblk; blk += gridDim.x) {
    const int64_t r0 = (blk * 4 + (threadIdx.x >> 6)) * (4 * U) + g;
    u32x4 v[U][NCH];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int k = 0; k < NCH; ++k) {
        const int c = q + 16 * k;
        v[u][k] = u32x4{0u, 0u, 0u, 0u};
        if (r0 + 4 * u < rows && c * EPC < dim)
          v[u][k] = __builtin_nontemporal_load((const u32x4*)(x + (r0 + 4 * u) * rowb) + c);
      }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      uint32_t m = 0;
#pragma unroll
      for (int k = 0; k < NCH; ++k) m = chunk_absmax<EK>(v[u][k], m);
#pragma unroll
      for (int o = 8; o >= 1; o >>= 1) m = absmax2<EK>(m, (uint32_t)__shfl_xor((int)m, o));
      const float s = scale_of(absmax_value<EK>(m));
      const bool plain = s < 1e30f;
      const float rc = 1.0f / s;
      const int64_t r = r0 + 4 * u;
      if (r >= rows) continue;
      if (q == 0) scale[r] = s;
#pragma unroll
      for (int k = 0; k < NCH; ++k) {
        const int c = q + 16 * k;
        if (c * EPC >= dim) break;
        uint32_t w[2];
        quant_chunk<EK>(v[u][k], s, rc, plain, w);
        store_bytes<EK>(out + r * dim + (int64_t)c * EPC, w);
      }
    }
  }
}

constexpr int kQuantParts = 1024;  // workgroups of the per-tensor maximum

// part[b] = the largest |x| bits seen by workgroup b.
template <int EK>
__global__ void __launch_bounds__(256) absmax_kernel(const u32x4* x, int64_t n, uint32_t* part) {
  __shared__ uint32_t s_m[4];
  uint32_t m = 0;
  const int64_t step = (int64_t)gridDim.x * 256;
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  for (; i + 3 * step < n; i += 4 * step) {
    const u32x4 a = x[i], b = x[i + step], c = x[i + 2 * step], d = x[i + 3 * step];
    m = chunk_absmax<EK>(d, chunk_absmax<EK>(c, chunk_absmax<EK>(b, chunk_absmax<EK>(a, m))));
  }
  for (; i < n; i += step) m = chunk_absmax<EK>(x[i], m);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = absmax2<EK>(m, (uint32_t)__shfl_xor((int)m, o));
  if ((threadIdx.x & 63) == 0) s_m[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = absmax2<EK>(absmax2<EK>(s_m[0], s_m[1]), absmax2<EK>(s_m[2], s_m[3]));
}

// Every workgroup takes the maximum of the parts (4 KB, from L2), then its chunks.
template <int EK>
__global__ void __launch_bounds__(256) quant_tensor_kernel(const u32x4* x, int64_t n, const uint32_t* part,
                                                           int nparts, uint8_t* out, float* scale) {
  constexpr int EPC = EK == EK_F32 ? 4 : 8;
  __shared__ uint32_t s_m[4];
  uint32_t m = 0;
  for (int i = threadIdx.x; i < nparts; i += 256) m = absmax2<EK>(m, part[i]);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = absmax2<EK>(m, (uint32_t)__shfl_xor((int)m, o));
  if ((threadIdx.x & 63) == 0) s_m[threadIdx.x >> 6] = m;
  __syncthreads();
  m = absmax2<EK>(absmax2<EK>(s_m[0], s_m[1]), absmax2<EK>(s_m[2], s_m[3]));
  const float s = scale_of(absmax_value<EK>(m));
  const bool plain = s < 1e30f;
  const float rc = 1.0f / s;
  if (blockIdx.x == 0 && threadIdx.x == 0) *scale = s;
  const int64_t step = (int64_t)gridDim.x * 256;
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  uint32_t w[2];
  for (; i + 3 * step < n; i += 4 * step) {
    u32x4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = x[i + k * step];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      quant_chunk<EK>(v[k], s, rc, plain, w);
      store_bytes<EK>(out + (i + k * step) * EPC, w);
    }
  }
  for (; i < n; i += step) {
    quant_chunk<EK>(x[i], s, rc, plain, w);
    store_bytes<EK>(out + i * EPC, w);
  }
}

template <int EK, int NCH>
int launch_quant_rows(const char* x, int64_t rows, int dim, uint8_t* out, float* scale, hipStream_t s) {
  constexpr int U = NCH == 1 ? 4 : NCH == 2 ? 2 : 1;
  const int64_t nblk = (rows + 16 * U - 1) / (16 * U);
  const unsigned grid = (unsigned)(nblk < (1 << 20) ? nblk : (1 << 20));
  hipLaunchKernelGGL((quant_rows_kernel<EK, NCH>), dim3(grid), dim3(256), 0, s, x, rows, dim, out, scale);
  return hipGetLastError() == hipSuccess ? LIK_OK : LIK_ERR_LAUNCH;
}

template <int EK>
int launch_quant(const char* x, int64_t rows, int dim, bool per_token, uint8_t* out, float* scale, uint32_t* part,
                 hipStream_t s) {
  constexpr int EPC = EK == EK_F32 ? 4 : 8;
  if (per_token) {
    const int ch = (dim / EPC + 15) / 16;
    if (ch <= 1) return launch_quant_rows<EK, 1>(x, rows, dim, out, scale, s);
    if (ch <= 2) return launch_quant_rows<EK, 2>(x, rows, dim, out, scale, s);
    if (ch <= 4) return launch_quant_rows<EK, 4>(x, rows, dim, out, scale, s);
    return launch_quant_rows<EK, 8>(x, rows, dim, out, scale, s);
  }
  const int64_t n = rows * dim / EPC;
  const int64_t want = (n + 255) / 256;
  const int parts = (int)(want < kQuantParts ? want : kQuantParts);
  hipLaunchKernelGGL((absmax_kernel<EK>), dim3(parts), dim3(256), 0, s, (const u32x4*)x, n, part);
  if (hipGetLastError() != hipSuccess) return LIK_ERR_LAUNCH;
  const unsigned grid = (unsigned)(want < 2048 ? want : 2048);
  hipLaunchKernelGGL((quant_tensor_kernel<EK>), dim3(grid), dim3(256), 0, s, (const u32x4*)x, n, part, parts, out,
                     scale);
  return hipGetLastError() == hipSuccess ? LIK_OK : LIK_ERR_LAUNCH;
}

}  // namespace lik

using namespace lik;

extern "C" {

size_t lik_quantize_fp8_workspace_size(uint32_t flags) {
  return (flags & LIK_PER_TOKEN) ? 0 : kQuantParts * sizeof(uint32_t);
}

int lik_quantize_fp8(const void* x, int32_t dtype, int64_t rows, int32_t dim, uint32_t flags, void* out, float* scale,
                     void* workspace, size_t workspace_bytes, lik_stream_t stream) {
  if (rows < 0 || dim <= 0 || (flags & ~(uint32_t)LIK_PER_TOKEN)) return LIK_ERR_INVALID;
  if (dtype != LIK_BF16 && dtype != LIK_F16 && dtype != LIK_F32) return LIK_ERR_UNSUPPORTED;
  if (rows == 0) return LIK_OK;
  if (!x || !out || !scale) return LIK_ERR_INVALID;
  const bool per_token = (flags & LIK_PER_TOKEN) != 0;
  // whole 16-byte chunks per row, rows that stay in a lane group's registers
  const int epc = dtype == LIK_F32 ? 4 : 8;
  if (dim % epc || (per_token && dim > 128 * epc)) return LIK_ERR_UNSUPPORTED;
  if ((uintptr_t)x % 16 || (uintptr_t)out % 8) return LIK_ERR_UNSUPPORTED;
  const size_t need = lik_quantize_fp8_workspace_size(flags);
  if (need && (!workspace || workspace_bytes < need)) return LIK_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  uint32_t* part = (uint32_t*)workspace;
  const char* xc = (const char*)x;
  uint8_t* o = (uint8_t*)out;
  switch (dtype) {
    case LIK_BF16: return launch_quant<EK_BF16>(xc, rows, dim, per_token, o, scale, part, s);
    case LIK_F16: return launch_quant<EK_F16>(xc, rows, dim, per_token, o, scale, part, s);
    default: return launch_quant<EK_F32>(xc, rows, dim, per_token, o, scale, part, s);
  }
}

}  // extern "C"
