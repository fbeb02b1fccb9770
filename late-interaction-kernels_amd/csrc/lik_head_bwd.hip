// Gradients of the projection head (maxsim_from_hidden training) for gfx950:
// from grad_D [Nd, Ld, dp], nonzero only on the doc rows that won some query
// token's max, and those winners (the forward's argmax)
//   grad_H[r] = grad_D[r] W          (zero rows elsewhere)
//   grad_W    = sum_r grad_D[r]^T H[r],  grad_b = sum_r grad_D[r]
// (reference fused_head.py:347-460). Products of 16-bit values are exact in
// fp32 and accumulate in fp32, as an fp32 GEMM on the widened operands would.
//
// As separate operators (unique of the winners, gathers, widening copies, two
// fp32 GEMMs, a scatter into a zeroed tensor) this took about 25 launches, a
// device -> host synchronisation and ~250 us of GPU time on 8 queries x 32 docs of
// 1024 rows (d_model 768, d_out 128), where the bytes (H rows that won, grad_H
// written once) need about 15. Four launches here, 69 us in all (head_grad_w
// 29.6, head_grad_h 24, its finish 10.7, the winners 4.5): the training step 540
// -> 212 us; at 1024 docs of 2048 rows grad_H's 3.2 GB bound both forms (2.13 ms).
// * head_winners_kernel: per doc, a bitmap of its winning rows and their
//   ascending list.
// * head_grad_h_kernel: per 32 rows, zeros where no row won; else W (held in
//   registers as A operands for the workgroup's lifetime) times grad_D's rows
//   (B operands as they lie in memory). All rows are written: no fill pass.
// * head_grad_w_kernel: 128 x 64 tiles of grad_W per wavefront on the fp32
//   matrix instruction (32x32x2), whose operands are one value per lane and row,
//   so rows need no transpose: an 8-byte load of a grad_D row gives a lane its
//   value for four 32-column blocks, a 4-byte load of an H row for two. Each workgroup sums its docs' rows; partial
//   tiles go to the workspace.
// * head_grad_w_finish_kernel: the partials added in a fixed order.
#include "lik_common.h"

namespace lik {

namespace {

struct HeadBwd {
  const int32_t* amax;  // [(i * nd + j) * lq + s]
  const char* gd;       // [nd * ld, dp] 16-bit
  const char* h;        // H rows: h + j * h_sn + t * h_sl (bytes)
  int64_t h_sn, h_sl;
  const char* w;        // W rows: w + o * w_sl (bytes)
  int64_t w_sl;
  char* gh;             // [nd * ld, dm] 16-bit, or null
  char* gw;             // [dout, dm] 16-bit, or null
  float* gb;            // [dout], or null
  int nq, lq, nd, ld, dp, dout, dm;
  uint32_t* bits;       // [nd][words]: bit t % 32 of word t / 32: row t won
  int words;
  int32_t* list;        // [nd][cap] winning rows, ascending
  int32_t* count;       // [nd]
  int cap;
  float* part;          // [splits][slices][128 * kSW] tiles of grad_W
  float* part_b;        // [splits][128] of grad_b
  int splits, slices, docs_per;
};

constexpr int kSW = 64;          // grad_W columns per tile (128 x 128 spilled its accumulators)
constexpr int kMaxWords = 2048;  // rows per doc / 32

__global__ void __launch_bounds__(256) head_winners_kernel(const HeadBwd p) {
  __shared__ uint32_t s_bits[kMaxWords];
  __shared__ int s_tot[4];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int j = blockIdx.x;
  for (int k = tid; k < p.words; k += 256) s_bits[k] = 0u;
  __syncthreads();
  const int np = p.nq * p.lq;
  for (int f = tid; f < np; f += 256) {
    const int i = f / p.lq, s = f - i * p.lq;
    const int a = p.amax[((int64_t)i * p.nd + j) * p.lq + s];
    if (a >= 0 && a < p.ld) atomicOr(&s_bits[a >> 5], 1u << (a & 31));
  }
  __syncthreads();
  int base = 0;
  for (int k0 = 0; k0 < p.words; k0 += 256) {
    const int k = k0 + tid;
    uint32_t b = k < p.words ? s_bits[k] : 0u;
    if (k < p.words) p.bits[(int64_t)j * p.words + k] = b;
    const int n = __builtin_popcount(b);
    int incl = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(incl, o);
      if (lane >= o) incl += t;
    }
    if (lane == 63) s_tot[wv] = incl;
    __syncthreads();
    int pos = base + incl - n;
    for (int w = 0; w < wv; ++w) pos += s_tot[w];
    while (b) {
      const int t = __builtin_ctz(b);
      b &= b - 1;
      if (pos < p.cap) p.list[(int64_t)j * p.cap + pos] = k * 32 + t;
      ++pos;
    }
    base += s_tot[0] + s_tot[1] + s_tot[2] + s_tot[3];
    __syncthreads();
  }
  if (tid == 0) p.count[j] = base < p.cap ? base : p.cap;
}

constexpr int kHB = 3;  // 32-column blocks of grad_H per wavefront (a workgroup covers 4 kHB of them)

template <int EK>
__global__ void __launch_bounds__(256) head_grad_h_kernel(const HeadBwd p) {
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = ((int)blockIdx.y * 4 + wv) * kHB * 32;  // first column of this wavefront
  if (m0 >= p.dm) return;
  // A operands: column m of W, output dims [64 h + 8 ks, +8). Each wavefront's
  // columns pass through LDS as they lie in memory (16-byte loads), 32 output
  // dims at a time; the column reads are one 2-byte read per element.
  __shared__ __attribute__((aligned(16))) uint16_t s_w[4][32][kHB * 32];
  u32x4 a[kHB][8];
#pragma unroll
  for (int c = 0; c < 4; ++c) {  // output dims [32 c, +32): half c / 2, k-steps 4 (c % 2) .. + 3
    constexpr int CPRW = kHB * 4;  // 16-byte chunks per row of the wavefront's columns
#pragma unroll
    for (int k = 0; k < 32 * CPRW / 64; ++k) {
      const int idx = k * 64 + lane, o = 32 * c + idx / CPRW, m = m0 + (idx % CPRW) * 8;
      u32x4 v = {0u, 0u, 0u, 0u};
      if (o < p.dout && m < p.dm) v = *(const u32x4*)(p.w + o * p.w_sl + (int64_t)m * 2);
      *(u32x4*)&s_w[wv][idx / CPRW][(idx % CPRW) * 8] = v;
    }
    // (a wavefront reads only what it wrote itself; its LDS operations are in order)
    __builtin_amdgcn_wave_barrier();
    if (h == c / 2) {
#pragma unroll
      for (int b = 0; b < kHB; ++b)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            a[b][4 * (c % 2) + ks][e] = (uint32_t)s_w[wv][8 * ks + 2 * e][32 * b + l32] |
                                        ((uint32_t)s_w[wv][8 * ks + 2 * e + 1][32 * b + l32] << 16);
    }
    __builtin_amdgcn_wave_barrier();
  }
  const int64_t nblk = (int64_t)p.nd * p.words;
  for (int64_t blk = blockIdx.x; blk < nblk; blk += gridDim.x) {
    const int64_t j = blk / p.words;
    const int t0 = (int)(blk - j * p.words) * 32;
    const bool in = t0 + l32 < p.ld;
    const int64_t row = j * p.ld + t0 + l32;
    char* out = p.gh + (row * p.dm + m0) * 2;
    const uint32_t won = p.bits[blk];
    if (won == 0u) {
      // 16 bytes a lane, the columns of a row by the lane's half and block
      if (in) {
#pragma unroll
        for (int c = 0; c < kHB * 4; c += 2)
          if (m0 + (c + h) * 8 < p.dm) *(u32x4*)(out + (c + h) * 16) = u32x4{0u, 0u, 0u, 0u};
      }
      continue;
    }
    u32x4 g[8];
    const bool live = (won >> l32) & 1u;  // rows without a winner: zeros (grad_D is not read)
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
      g[ks] = (live && 64 * h + 8 * ks < p.dp) ? *(const u32x4*)(p.gd + (row * p.dp + 64 * h + 8 * ks) * 2)
                                               : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int b = 0; b < kHB; ++b) {
      f32x16 acc = {};
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) acc = mfma32<EK>(acc, &a[b][ks], &g[ks]);
      // element e of lane (h, l32): column 8 (e / 4) + 4 h + e % 4 of row l32.
      // The halves swap groups so that a lane holds 16 consecutive columns.
      uint32_t w[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if constexpr (EK == EK_F16) w[e] = f32_to_f16_bits(acc[2 * e]) | (f32_to_f16_bits(acc[2 * e + 1]) << 16);
        else w[e] = __builtin_bit_cast(uint32_t, bf16x2{(__bf16)acc[2 * e], (__bf16)acc[2 * e + 1]});
      }
      // w[2 q], w[2 q + 1]: columns 8 q + 4 h .. + 3. The swap hands half 1 the
      // other half's groups 2, 3 and half 0 the other half's groups 0, 1.
      u32x4 v[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const auto s0 = __builtin_amdgcn_permlane32_swap(w[2 * q], w[2 * (q + 2)], false, false);
        const auto s1 = __builtin_amdgcn_permlane32_swap(w[2 * q + 1], w[2 * (q + 2) + 1], false, false);
        v[q] = live ? u32x4{s0[0], s1[0], s0[1], s1[1]} : u32x4{0u, 0u, 0u, 0u};
      }
      const int c0 = 32 * b + 16 * h;  // half h: columns c0 .. c0 + 15
      if (in) {
        if (m0 + c0 < p.dm) *(u32x4*)(out + c0 * 2) = v[0];
        if (m0 + c0 + 8 < p.dm) *(u32x4*)(out + c0 * 2 + 16) = v[1];
      }
    }
  }
}

template <int EK>
__device__ __forceinline__ float lo16(uint32_t w) {
  if constexpr (EK == EK_BF16) return bf16lo_to_f32(w);
  else return f16_to_f32((uint16_t)(w & 0xffffu));
}
template <int EK>
__device__ __forceinline__ float hi16(uint32_t w) {
  if constexpr (EK == EK_BF16) return bf16hi_to_f32(w);
  else return f16_to_f32((uint16_t)(w >> 16));
}

// Workgroup (split, slice): grad_W[:, kSW slice .. + kSW) over the winning rows
// of docs [split * docs_per, + docs_per), rows dealt to the 4 wavefronts in
// pairs. Column 4 l32 + a of a grad_D row (2 l32 + b of H's slice) is lane l32's
// value for block a (b).
template <int EK>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) head_grad_w_kernel(const HeadBwd p) {
  __shared__ __attribute__((aligned(16))) float s_t[128 * kSW];
  __shared__ float s_b[4][128];
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slice = blockIdx.x % p.slices, split = blockIdx.x / p.slices;
  f32x16 acc[4][2];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = f32x16{};
  float sb[4] = {0.f, 0.f, 0.f, 0.f};
  const int col = kSW * slice + 2 * l32;
  const int j1 = (split + 1) * p.docs_per < p.nd ? (split + 1) * p.docs_per : p.nd;
  for (int j = split * p.docs_per; j < j1; ++j) {
    const int n = __builtin_amdgcn_readfirstlane(p.count[j]);
    const int32_t* list = p.list + (int64_t)j * p.cap;
    // 8 row pairs per step: all loads first, the next step's row numbers
    // (one per lane, row pair u of half h in lane 2 u + h) on their way
    auto rows_at = [&](int k0) -> int {
      const int k = k0 + 8 * ((lane >> 1) & 7) + (lane & 1);
      return k < n ? list[k] : -1;
    };
    int next = rows_at(wv * 2);
    for (int k0 = wv * 2; k0 < n; k0 += 8 * 8) {
      const int rows = next;
      next = rows_at(k0 + 64);
      u32x2 gv[8];
      uint32_t hv[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int r0 = __builtin_amdgcn_readlane(rows, 2 * u), r1 = __builtin_amdgcn_readlane(rows, 2 * u + 1);
        const int64_t t = h ? r1 : r0;
        gv[u] = u32x2{0u, 0u};
        hv[u] = 0u;
        if (t >= 0) {
          if (4 * l32 < p.dp) gv[u] = *(const u32x2*)(p.gd + (((int64_t)j * p.ld + t) * p.dp + 4 * l32) * 2);
          if (col < p.dm) hv[u] = *(const uint32_t*)(p.h + j * p.h_sn + t * p.h_sl + (int64_t)col * 2);
        }
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float g[4] = {lo16<EK>(gv[u][0]), hi16<EK>(gv[u][0]), lo16<EK>(gv[u][1]), hi16<EK>(gv[u][1])};
        const float x[2] = {lo16<EK>(hv[u]), hi16<EK>(hv[u])};
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          sb[a] += g[a];
#pragma unroll
          for (int b = 0; b < 2; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(g[a], x[b], acc[a][b], 0, 0, 0);
        }
      }
    }
  }
  // the wavefronts' tiles added in order through LDS: element e of lane (h, l32)
  // is (row 8 (e / 4) + 4 h + e % 4, column l32) of block (a, b), i.e. grad_W
  // row 4 row + a, column 2 l32 + b of the slice
  for (int w = 0; w < 4; ++w) {
    if (wv == w) {
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          f32x2* t = (f32x2*)&s_t[(4 * (8 * (e >> 2) + 4 * h + (e & 3)) + a) * kSW + 2 * l32];
          const f32x2 v = {acc[a][0][e], acc[a][1][e]};
          *t = w == 0 ? v : *t + v;
        }
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const float v = sb[a] + __shfl_xor(sb[a], 32);
        if (h == 0) s_b[w][4 * l32 + a] = v;
      }
    }
    __syncthreads();
  }
  f32x4* out = (f32x4*)(p.part + ((int64_t)split * p.slices + slice) * (128 * kSW));
  for (int k = tid; k < 128 * kSW / 4; k += 256) out[k] = ((const f32x4*)s_t)[k];
  if (slice == 0 && tid < 128) p.part_b[split * 128 + tid] = ((s_b[0][tid] + s_b[1][tid]) + s_b[2][tid]) + s_b[3][tid];
}

// grad_W element (o, m) = sum of the splits' tiles, in split order; grad_b too.
template <int EK>
__global__ void __launch_bounds__(256) head_grad_w_finish_kernel(const HeadBwd p) {
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p.gw && k < (int64_t)p.dout * p.dm) {
    const int o = (int)(k / p.dm), m = (int)(k - (int64_t)o * p.dm);
    const float* t = p.part + (int64_t)(m / kSW) * (128 * kSW) + o * kSW + m % kSW;
    float s = 0.f;
#pragma unroll 8
    for (int c = 0; c < p.splits; ++c) s += t[(int64_t)c * p.slices * (128 * kSW)];
    ((uint16_t*)p.gw)[k] = (uint16_t)(EK == EK_F16 ? f32_to_f16_bits(s) : f32_to_bf16_bits(s));
  }
  if (p.gb && k < p.dout) {
    float s = 0.f;
    for (int c = 0; c < p.splits; ++c) s += p.part_b[c * 128 + k];
    p.gb[k] = s;
  }
}

size_t al(size_t x) { return (x + 255) & ~(size_t)255; }

struct HeadBwdWs {
  size_t bits, list, count, part, part_b, total;
};
// Sizes that follow from the shape: row splits of grad_W so that the slices
// give about 512 workgroups (two per CU: the tiles take 128 accumulators), each
// of whole docs.
void head_bwd_shape(HeadBwd& p, HeadBwdWs& w) {
  p.words = (p.ld + 31) / 32;
  p.cap = (int)((int64_t)p.nq * p.lq < p.ld ? (int64_t)p.nq * p.lq : p.ld);
  p.slices = (p.dm + kSW - 1) / kSW;
  const int want = 512 / p.slices < 1 ? 1 : 512 / p.slices;
  p.docs_per = (p.nd + want - 1) / want;
  p.splits = (p.nd + p.docs_per - 1) / p.docs_per;
  size_t o = 0;
  w.bits = o; o += al((size_t)p.nd * p.words * 4);
  w.list = o; o += al((size_t)p.nd * p.cap * 4);
  w.count = o; o += al((size_t)p.nd * 4);
  w.part = o; o += al((size_t)p.splits * p.slices * 128 * kSW * 4);
  w.part_b = o; o += al((size_t)p.splits * 128 * 4);
  w.total = o + 256;
}

bool head_bwd_takes(int32_t dtype, int64_t nq, int64_t lq, int64_t nd, int64_t ld, int64_t dp, int64_t dout, int64_t dm) {
  return (dtype == LIK_BF16 || dtype == LIK_F16) && nq > 0 && lq > 0 && nd > 0 && ld > 0 && nd <= 0x7fffffff &&
         nq * lq <= (1 << 24) && ld <= (int64_t)kMaxWords * 32 && dp % 8 == 0 && dp <= 128 && dout >= 1 && dout <= dp &&
         dm >= 8 && dm % 8 == 0 && dm <= (1 << 16);
}

template <int EK>
int launch_head_bwd(const HeadBwd& p, hipStream_t s) {
  hipLaunchKernelGGL(head_winners_kernel, dim3((unsigned)p.nd), dim3(256), 0, s, p);
  if (hipGetLastError() != hipSuccess) return LIK_ERR_LAUNCH;
  if (p.gh) {
    const int64_t nblk = (int64_t)p.nd * p.words;
    const unsigned gy = (unsigned)((p.dm + 128 * kHB - 1) / (128 * kHB));
    const int64_t most = gy < 512 ? 512 / gy : 1;  // two workgroups per CU
    const int64_t gx = nblk < most ? nblk : most;
    hipLaunchKernelGGL((head_grad_h_kernel<EK>), dim3((unsigned)gx, gy), dim3(256), 0, s, p);
    if (hipGetLastError() != hipSuccess) return LIK_ERR_LAUNCH;
  }
  if (p.gw || p.gb) {
    hipLaunchKernelGGL((head_grad_w_kernel<EK>), dim3((unsigned)(p.splits * p.slices)), dim3(256), 0, s, p);
    if (hipGetLastError() != hipSuccess) return LIK_ERR_LAUNCH;
    const int64_t n = (int64_t)p.dout * p.dm;
    hipLaunchKernelGGL((head_grad_w_finish_kernel<EK>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p);
    if (hipGetLastError() != hipSuccess) return LIK_ERR_LAUNCH;
  }
  return LIK_OK;
}

}  // namespace
}  // namespace lik

using namespace lik;

extern "C" {

size_t lik_head_backward_workspace_size(int32_t dtype, int64_t nq, int64_t lq, int64_t nd, int64_t ld, int64_t dp,
                                        int64_t d_out, int64_t d_model) {
  if (!head_bwd_takes(dtype, nq, lq, nd, ld, dp, d_out, d_model)) return 0;
  HeadBwd p{};
  HeadBwdWs w;
  p.nq = (int)nq; p.lq = (int)lq; p.nd = (int)nd; p.ld = (int)ld; p.dp = (int)dp; p.dout = (int)d_out; p.dm = (int)d_model;
  head_bwd_shape(p, w);
  return w.total;
}

int lik_head_backward(const int32_t* argmax, int64_t nq, int64_t lq, const void* grad_d, int64_t dp,
                      const lik_seqs_t* H, const void* W, int64_t w_stride, int64_t d_out, void* grad_h, void* grad_w,
                      float* grad_b, void* workspace, size_t workspace_bytes, lik_stream_t stream) {
  if (!H) return LIK_ERR_INVALID;
  if (!head_bwd_takes(H->dtype, nq, lq, H->n, H->len, dp, d_out, H->dim)) return LIK_ERR_UNSUPPORTED;
  if (!argmax || !grad_d || !H->data || !W || H->cu_seqlens) return LIK_ERR_INVALID;
  if ((uintptr_t)grad_d % 16 || (uintptr_t)H->data % 4 || H->stride_n % 2 || H->stride_l % 2 ||
      (uintptr_t)grad_h % 16 || (uintptr_t)W % 16 || (w_stride * 2) % 16 || (uintptr_t)grad_w % 2)
    return LIK_ERR_UNSUPPORTED;
  HeadBwd p{};
  HeadBwdWs w;
  p.amax = argmax;
  p.gd = (const char*)grad_d;
  p.h = (const char*)H->data;
  p.h_sn = H->stride_n * 2;
  p.h_sl = H->stride_l * 2;
  p.w = (const char*)W;
  p.w_sl = w_stride * 2;
  p.gh = (char*)grad_h;
  p.gw = (char*)grad_w;
  p.gb = grad_b;
  p.nq = (int)nq;
  p.lq = (int)lq;
  p.nd = (int)H->n;
  p.ld = (int)H->len;
  p.dp = (int)dp;
  p.dout = (int)d_out;
  p.dm = H->dim;
  head_bwd_shape(p, w);
  if (!workspace || workspace_bytes < w.total) return LIK_ERR_WORKSPACE;
  char* ws = (char*)(((uintptr_t)workspace + 255) & ~(uintptr_t)255);
  p.bits = (uint32_t*)(ws + w.bits);
  p.list = (int32_t*)(ws + w.list);
  p.count = (int32_t*)(ws + w.count);
  p.part = (float*)(ws + w.part);
  p.part_b = (float*)(ws + w.part_b);
  return H->dtype == LIK_F16 ? launch_head_bwd<EK_F16>(p, (hipStream_t)stream)
                             : launch_head_bwd<EK_BF16>(p, (hipStream_t)stream);
}

}  // extern "C"
