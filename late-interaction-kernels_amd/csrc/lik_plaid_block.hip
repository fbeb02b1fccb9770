// PLAID decode + MaxSim for query blocks of up to 512 tokens (gfx950).
//
// One 8-wavefront workgroup per (query group, doc range); wavefront w holds
// NSUB blocks of 32 query tokens as MFMA B fragments. The range's 32-token
// tiles are taken four at a time (a stage): 128 tokens are decoded into one of
// two LDS buffers while the wavefronts multiply the other, one barrier a stage.
//
// What bounds the fused decode is latency and decode arithmetic, not bytes:
// with one barrier per 32-token tile, each behind a code -> centroid row ->
// decode chain (the tile kernel, lik_kernel.h), 512 query tokens against 4.5 M
// tokens of 2-bit residuals took 1330 us, 256 query tokens 1146 us. Here 662
// and 504 us (the MFMAs alone: about 350 and 175):
// * a stage's codes and residual bits are loaded three stages ahead and its
//   centroid rows two ahead of their MFMAs, 4 rows per thread in flight;
// * the four passes of a decode go step by step together (one after the other,
//   with a branch per element, a stage took 7.3 us; 2.9 us now), one inverse
//   norm per lane instead of one per pass;
// * wavefronts w and w + 4 share a SIMD and run the two halves of a stage in
//   opposite order (multiply then decode, decode then multiply), so one's
//   decode arithmetic runs beside the other's MFMAs.
//
// Scores are bitwise the tile kernel's: the same fp32 adds, per-chunk fma
// chain, row reduction tree and rounding of a decoded row, the same k order,
// exact maxima, and its order of a query's column sum.
#include "lik_params.h"

namespace lik {

namespace {

constexpr int kBlkTiles = 4;  // tiles per stage
constexpr int kBlkRMax = 512;  // docs per workgroup (table in LDS)
constexpr uint32_t kOut = 0xffffffffu;  // byte offset past every buffer range: the load returns 0

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, uint32_t nbytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)nbytes, 0x00020000);
}
__device__ __forceinline__ uint32_t clamp_u32(int64_t x) {
  return x < 0 ? 0u : (x >= 0xffffffffLL ? 0xffffffffu : (uint32_t)x);
}

template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), CTRL, 0xf, 0xf, true));
}
// Sum over the N (8 or 16) lanes of a row. Each step's partner holds the value
// an xor shuffle by 1, 2, 4, 8 would bring (the lanes below it are equal by
// then), so the sum has the association of the tile kernel's shuffles.
template <int N>
__device__ __forceinline__ float row_sum(float v) {
  v = dpp_add<0xb1>(v);   // quad_perm [1, 0, 3, 2]
  v = dpp_add<0x4e>(v);   // quad_perm [2, 3, 0, 1]
  v = dpp_add<0x141>(v);  // row_half_mirror
  if constexpr (N == 16) v = dpp_add<0x140>(v);  // row_mirror
  return v;
}

// Two values rounded to the 16-bit type, packed (bf16: one conversion for both).
template <int EK>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  if constexpr (EK == EK_F16) return f32_to_f16_bits(a) | (f32_to_f16_bits(b) << 16);
  else return __builtin_bit_cast(uint32_t, bf16x2{(__bf16)a, (__bf16)b});
}
// Lane I of each quad, to the quad.
template <int I>
__device__ __forceinline__ float quad_lane(float v) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), I * 0x55, 0xf, 0xf, true));
}

}  // namespace

template <int EK, int CD, int DPAD, int NSUB, int NBITS>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) plaid_block_kernel(const Params p) {
  using T = KT<EK, DPAD>;
  constexpr int COLS = 8 * NSUB * 32;
  constexpr int KS = T::KSTEPS;
  constexpr int CPR = DPAD / 8;            // 8-element chunks (16 bytes decoded) per row
  constexpr int RPP = 512 / CPR;           // rows one pass of the workgroup decodes
  constexpr int NCH = kBlkTiles * 32 / RPP;  // passes per stage = chunks per thread
  constexpr int TPP = RPP / 32;            // tiles per pass
  constexpr float NEG_INF = -__builtin_huge_valf();

  __shared__ __attribute__((aligned(16))) char s_tile[2][kBlkTiles * 32 * T::ROW_B];
  // per-column maxima of docs that ended in the last two stages (at most one doc end per tile)
  __shared__ __attribute__((aligned(16))) float s_col[2][kBlkTiles][COLS];
  __shared__ int s_slotk[2][kBlkTiles];
  // bucket weights by code; 2-bit codes by pairs of codes (one 8-byte read for two)
  __shared__ __attribute__((aligned(16))) float s_bw[NBITS == 2 ? 32 : 256];
  __shared__ float* s_outp[COLS];
  __shared__ int64_t s_tok[kBlkRMax];
  __shared__ int32_t s_len[kBlkRMax];
  __shared__ __attribute__((aligned(16))) i32x4 s_nz[kBlkRMax + 1];  // {k, length, first token lo, hi}; [nnz] = sentinel
  __shared__ int s_nnz, s_ntiles;

  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, l32 = lane & 31;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  int64_t g, r;
  {
    const int64_t b = blockIdx.x;
    if (p.xcd_map) {  // all column groups of a doc range on one XCD, back to back
      const int64_t i = b >> 3;
      g = i % p.ngroups;
      r = (i / p.ngroups) * 8 + (b & 7);
    } else {
      g = b % p.ngroups;
      r = b / p.ngroups;
    }
  }
  if (r >= p.NR) return;

  // bucket codes past the last bucket read the last bucket's weight
  if (tid < (NBITS == 2 ? 32 : 256)) {
    const int c = NBITS == 2 ? ((tid >> 1) >> (2 * (tid & 1))) & 3 : tid;
    s_bw[tid] = p.pl.bw[c < p.pl.nb ? c : p.pl.nb - 1];
  }
  const int64_t j0 = r * (int64_t)p.R;
  const int64_t j1 = (j0 + p.R < p.ndocs_pg) ? j0 + p.R : p.ndocs_pg;
  const int nloc = (int)(j1 - j0);
  for (int t = tid; t < COLS; t += 512) {
    const int64_t u = g * p.QPG + t;
    s_outp[t] = (t < p.QPG && u < p.nunits) ? p.out + u * p.osq + j0 * p.osd : nullptr;
  }
  __syncthreads();
  for (int k = tid; k < nloc; k += 512) {
    const int64_t j = j0 + k;
    const int64_t L = doc_len<SRC_PLAID>(p, j);
    s_tok[k] = p.pl.cu ? (int64_t)p.pl.cu[j] : j * p.pl.codes_sn;
    s_len[k] = (int32_t)L;
    if (L <= 0)
      for (int t = 0; t < p.QPG; ++t)
        if (float* o = s_outp[t]) o[k * p.osd] = 0.f;
  }
  __syncthreads();
  if (wv == 0) {
    int base = 0, ntl = 0;
    for (int k0 = 0; k0 < nloc; k0 += 64) {
      const int k = k0 + lane;
      const int L = k < nloc ? s_len[k] : 0;
      const bool nz = L > 0;
      const uint64_t bal = __ballot(nz);
      const int pos = base + (int)__popcll(bal & ((1ull << lane) - 1ull));
      if (nz) s_nz[pos] = (i32x4){k, L, (int)(uint32_t)s_tok[k], (int)(s_tok[k] >> 32)};
      base += (int)__popcll(bal);
      int nt = nz ? (L + 31) >> 5 : 0;
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) nt += __shfl_xor(nt, o);
      ntl += nt;
    }
    if (lane == 0) {
      s_nnz = base;
      s_ntiles = ntl;
      s_nz[base] = (i32x4){0, 0, 0, 0};
    }
  }
  __syncthreads();
  const int nnz = __builtin_amdgcn_readfirstlane(s_nnz);
  if (nnz == 0) return;
  const int nstages = (__builtin_amdgcn_readfirstlane(s_ntiles) + kBlkTiles - 1) / kBlkTiles;

  // query block -> B fragments (lane l32: column, half h: elements [h * DPAD/2, +DPAD/2))
  u32x4 bq[NSUB][KS];
  float qsc[NSUB];
#pragma unroll
  for (int sub = 0; sub < NSUB; ++sub) {
    const int col = (wv * NSUB + sub) * 32 + l32;
    const int ul = col / p.LU;
    const int64_t tok = col - ul * p.LU;
    const int64_t u = g * p.QPG + ul;
    const bool valid = ul < p.QPG && u < p.nunits && tok < seq_len(p.q, u);
    const char* rowp = valid ? seq_row0(p.q, u) + tok * p.q.sl_b : nullptr;
    float ss = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int e = h * (DPAD / 2) + ks * 8;
      bq[sub][ks] = (valid && e < p.q.dim) ? *(const u32x4*)(rowp + (int64_t)e * 2) : (u32x4){0u, 0u, 0u, 0u};
      if (p.normalize & 1) ss += chunk_sumsq<EK>(bq[sub][ks]);
    }
    ss += __shfl_xor(ss, 32);
    const float sc = (p.normalize & 1) ? inv_norm(ss) : 1.f;
    qsc[sub] = valid ? sc : 0.f;
  }
  // a wavefront whose columns hold no query token only decodes
  const bool has_cols = (int64_t)wv * NSUB * 32 < (int64_t)p.QPG * p.LU && g * p.QPG + (wv * NSUB * 32) / p.LU < p.nunits;

  // Tile cursor: the workgroup's tiles in order (uniform). crem: tokens of the
  // doc from the tile's first on; the doc's codes and residual rows are buffers
  // that end with the doc (rows past its end read 0), the tile at byte offsets
  // coff_c, coff_r in them. (They start over at the tile once the offset
  // reaches 1 GiB, in a document of tens of millions of tokens.)
  int cm = 0, crem, ck;
  int64_t ct0;
  uint32_t coff_c, coff_r;
  const uint32_t tile_r = 32u * (uint32_t)p.pl.res_st;
  __amdgpu_buffer_rsrc_t rcode, rres;
  auto rebase = [&]() {
    rcode = rsrc(p.pl.codes + ct0, clamp_u32((int64_t)crem * 4));
    rres = rsrc(p.pl.res + ct0 * p.pl.res_st, clamp_u32((int64_t)crem * p.pl.res_st));
    coff_c = 0u;
    coff_r = 0u;
  };
  auto entry = [&](int m) {
    const i32x4 e = s_nz[m];
    cm = m;
    ck = __builtin_amdgcn_readfirstlane(e[0]);
    crem = __builtin_amdgcn_readfirstlane(e[1]);
    ct0 = (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane(e[2]) |
          ((int64_t)__builtin_amdgcn_readfirstlane(e[3]) << 32);
    rebase();
  };
  entry(0);
  // A stage's tiles: valid rows (bits 0..5, 0 past the last tile) and 1 + the
  // doc the tile ends (bits 8.., 0: none).
  struct Stage {
    int d[kBlkTiles];
  };
  auto rows_in = [](int d) -> int { return d & 63; };

  // thread's chunks: pass i covers rows [i * RPP, +RPP) of the stage: row prow of tile i * TPP + ptile
  const int cc = tid % CPR, prow = (tid / CPR) & 31;
  const int ptile = __builtin_amdgcn_readfirstlane(tid / CPR / 32);
  const bool cc_ok = cc * 8 < p.q.dim;
  const __amdgpu_buffer_rsrc_t rcent = rsrc(p.pl.cent, clamp_u32(p.pl.ncent * p.pl.cent_sb));
  const uint32_t vcode = (uint32_t)prow * 4u;
  const uint32_t vres = (uint32_t)prow * (uint32_t)p.pl.res_st + (uint32_t)(cc * NBITS);
  constexpr int NB = NBITS == 8 ? 2 : 1;  // dwords of a chunk's residual bits
  uint32_t code[NCH], bits[NCH][NB], bits_n[NCH][NB];
  u32x4 cv[NCH];
  // The next stage: its tiles off the cursor, the loads of its codes and residual bits.
  auto produce = [&]() -> Stage {
    Stage s;
#pragma unroll
    for (int t = 0; t < kBlkTiles; ++t) {
      if (TPP == 1 || (t & 1) == ptile) {
        const int i = t / TPP;
        // (the tile's offset is added to the lane's: the scalar offset of a
        // buffer load is not part of its bounds check)
        code[i] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rcode, vcode + coff_c, 0, 0);
        const uint32_t ro = cc_ok ? vres + coff_r : kOut;
        if constexpr (NBITS == 2) bits_n[i][0] = __builtin_amdgcn_raw_buffer_load_b16(rres, ro, 0, 0);
        else if constexpr (NBITS == 4) bits_n[i][0] = __builtin_amdgcn_raw_buffer_load_b32(rres, ro, 0, 0);
        else {
          const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rres, ro, 0, 0);
          bits_n[i][0] = v[0];
          bits_n[i][NB - 1] = v[1];
        }
      }
      s.d[t] = crem > 32 ? 32 : (crem > 0 ? crem | ((ck + 1) << 8) : 0);
      if (crem <= 32) entry(cm + 1 < nnz ? cm + 1 : nnz);
      else {
        crem -= 32;
        coff_c += 128u;
        coff_r += tile_r;
        if (coff_r >= 0x40000000u) {
          ct0 += coff_c >> 2;
          rebase();
        }
      }
    }
    return s;
  };
  // Centroid rows of the stage whose codes have arrived; its residual bits
  // move up. (Rows past a doc's end take centroid 0: finite or not, their
  // products are replaced by -inf.)
  auto load_rows = [&]() {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const uint32_t c = code[i] < (uint32_t)p.pl.ncent ? code[i] : 0u;
      cv[i] = __builtin_amdgcn_raw_buffer_load_b128(rcent, cc_ok ? c * (uint32_t)p.pl.cent_sb + (uint32_t)(cc * 16) : kOut,
                                                    0, 0);
#pragma unroll
      for (int b = 0; b < NB; ++b) bits[i][b] = bits_n[i][b];
    }
  };
  // The loaded rows decoded, normalised, rounded, into LDS buffer buf (dims
  // past the embedding's as zeros). All passes go step by step together, so
  // that their lookup and reduction latencies overlap.
  auto decode = [&](int buf) {
    float x[NCH][8], sc[NCH];
#pragma unroll
    for (int i = 0; i < NCH; ++i)
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        if constexpr (NBITS == 2) {
          const f32x2 v = *(const f32x2*)&s_bw[2 * ((bits[i][0] >> (2 * e)) & 15u)];
          x[i][e] = v[0];
          x[i][e + 1] = v[1];
        } else if constexpr (NBITS == 4) {
          x[i][e] = s_bw[(bits[i][0] >> (4 * e)) & 15u];
          x[i][e + 1] = s_bw[(bits[i][0] >> (4 * e + 4)) & 15u];
        } else {
          x[i][e] = s_bw[(bits[i][e >> 2] >> (8 * (e & 3))) & 255u];
          x[i][e + 1] = s_bw[(bits[i][e >> 2] >> (8 * (e & 3) + 8)) & 255u];
        }
      }
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      float ss = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if constexpr (CD == EK_BF16)
          x[i][e] = ((e & 1) ? bf16hi_to_f32(cv[i][e >> 1]) : bf16lo_to_f32(cv[i][e >> 1])) + x[i][e];
        else
          x[i][e] = f16_to_f32((uint16_t)((e & 1) ? (cv[i][e >> 1] >> 16) : (cv[i][e >> 1] & 0xffffu))) + x[i][e];
        ss = fmaf(x[i][e], x[i][e], ss);
      }
      sc[i] = cc_ok ? ss : 0.f;
    }
    if (p.normalize & 2) {
      // one inverse norm per lane: lane 4 k + i of a row takes pass i's, and
      // the passes read theirs back from their quad
#pragma unroll
      for (int i = 0; i < NCH; ++i) sc[i] = row_sum<CPR>(sc[i]);
      float v = sc[0];
#pragma unroll
      for (int i = 1; i < NCH; ++i) v = (lane & 3) == i ? sc[i] : v;
      v = inv_norm(v);
      sc[0] = quad_lane<0>(v);
      sc[1] = quad_lane<1>(v);
      if constexpr (NCH == 4) {
        sc[2] = quad_lane<2>(v);
        sc[3] = quad_lane<3>(v);
      }
    } else {
#pragma unroll
      for (int i = 0; i < NCH; ++i) sc[i] = 1.f;
    }
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      u32x4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        w[e] = pack2<EK>(x[i][2 * e] * sc[i], x[i][2 * e + 1] * sc[i]);
        w[e] = cc_ok ? w[e] : 0u;
      }
      *(u32x4*)(s_tile[buf] + ((i * TPP + ptile) * 32 + prow) * T::ROW_B + cc * 16) = w;
    }
  };

  float m[NSUB];
#pragma unroll
  for (int sub = 0; sub < NSUB; ++sub) m[sub] = NEG_INF;

  // MFMAs and running maxima of the stage in buffer buf; docs that end in it
  // are parked in s_col[buf]. A tile's A fragments are read while the tile
  // before it is multiplied.
  auto multiply = [&](const Stage& s, int buf) {
    const char* A = s_tile[buf] + l32 * T::ROW_B + h * T::HALF_B;
    u32x4 a[2][KS];
    if (has_cols) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) a[0][ks] = *(const u32x4*)(A + ks * 16);
    }
#pragma unroll
    for (int t = 0; t < kBlkTiles; ++t) {
      const int nv = rows_in(s.d[t]);
      if (has_cols) {
        if (t + 1 < kBlkTiles) {
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) a[(t + 1) & 1][ks] = *(const u32x4*)(A + (t + 1) * 32 * T::ROW_B + ks * 16);
        }
        __builtin_amdgcn_sched_barrier(0);
        f32x16 acc[NSUB];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int sub = 0; sub < NSUB; ++sub)
            acc[sub] = mfma32<EK>(ks == 0 ? f32x16{} : acc[sub], &a[t & 1][ks], &bq[sub][ks]);
        if (nv < 32) {
          // element e of lane half h is row 8 (e / 4) + 4 h + e % 4
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const bool in = 8 * (e >> 2) + 4 * h + (e & 3) < nv;
#pragma unroll
            for (int sub = 0; sub < NSUB; ++sub) acc[sub][e] = in ? acc[sub][e] : NEG_INF;
          }
        }
#pragma unroll
        for (int sub = 0; sub < NSUB; ++sub)
#pragma unroll
          for (int e = 0; e < 16; e += 2) m[sub] = max_nan(m[sub], max_nan(acc[sub][e], acc[sub][e + 1]));
        if ((s.d[t] >> 8) != 0) {
#pragma unroll
          for (int sub = 0; sub < NSUB; ++sub) {
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(m[sub]), __float_as_uint(m[sub]), false, false);
            const float mm = max_nan(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
            if (h == 0) s_col[buf][t][(wv * NSUB + sub) * 32 + l32] = __builtin_isfinite(mm) ? mm * qsc[sub] : 0.f;
            m[sub] = NEG_INF;
          }
        }
      }
    }
    if (tid == 0) {
#pragma unroll
      for (int t = 0; t < kBlkTiles; ++t) s_slotk[buf][t] = (s.d[t] >> 8) - 1;
    }
  };
  // Scores of the docs parked in s_col[buf] (after the barrier that ends their stage).
  const bool rot = (p.LU & 3) == 0;
  auto flush = [&](int buf) {
    for (int task = (tid & 63) * 8 + (tid >> 6); task < kBlkTiles * p.QPG; task += 512) {
      const int t = task / p.QPG, u = task - t * p.QPG;
      const int k = s_slotk[buf][t];
      float* const orow = s_outp[u];
      if (k < 0 || !orow) continue;
      const float* cvp = &s_col[buf][t][u * p.LU];
      float sum = 0.f;
      if (rot) {  // the tile kernel's order: 4-column groups, rotated by the unit
        const int nvec = p.LU >> 2;
        int c = u % nvec;
        for (int j = 0; j < nvec; ++j) {
          const f32x4 v = *(const f32x4*)(cvp + 4 * c);
          sum += v[0];
          sum += v[1];
          sum += v[2];
          sum += v[3];
          c = (c + 1 == nvec) ? 0 : c + 1;
        }
      } else {
        for (int j = 0; j < p.LU; ++j) sum += cvp[j];
      }
      ((__attribute__((address_space(1))) float*)orow)[k * p.osd] = sum * p.out_scale;
    }
  };

  // stages: s0 being multiplied, s1 decoded during it, s2's centroid rows and
  // s3's codes and residual bits on their way
  Stage s0 = produce();
  load_rows();
  Stage s1 = produce();
  decode(0);
  load_rows();
  Stage s2 = produce();
  __syncthreads();
  const bool mul_first = wv < 4;
  bool parked = false;  // the stage before s0 ended a doc
  for (int n = 0; n < nstages; ++n) {
    const int buf = n & 1;
    if (mul_first) multiply(s0, buf);
    if (parked) flush(buf ^ 1);
    parked = ((s0.d[0] | s0.d[1] | s0.d[2] | s0.d[3]) >> 8) != 0;
    decode(buf ^ 1);
    load_rows();
    const Stage s3 = produce();
    if (!mul_first) multiply(s0, buf);
    s0 = s1;
    s1 = s2;
    s2 = s3;
    __syncthreads();
  }
  if (parked) flush((nstages - 1) & 1);
}

namespace {

template <int EK, int CD, int DPAD, int NSUB>
int launch_block_bits(const Params& p, int64_t nb, hipStream_t s) {
  const dim3 grid((unsigned)nb), block(512);
  if (p.pl.nbits == 2) launch_kernel(plaid_block_kernel<EK, CD, DPAD, NSUB, 2>, grid, block, 0, s, p);
  else if (p.pl.nbits == 4) launch_kernel(plaid_block_kernel<EK, CD, DPAD, NSUB, 4>, grid, block, 0, s, p);
  else launch_kernel(plaid_block_kernel<EK, CD, DPAD, NSUB, 8>, grid, block, 0, s, p);
  return hipGetLastError() == hipSuccess ? LIK_OK : LIK_ERR_LAUNCH;
}
template <int EK, int CD>
int launch_block_dpad(int dpad, int cols, const Params& p, int64_t nb, hipStream_t s) {
  if (dpad == 64)
    return cols == 256 ? launch_block_bits<EK, CD, 64, 1>(p, nb, s) : launch_block_bits<EK, CD, 64, 2>(p, nb, s);
  return cols == 256 ? launch_block_bits<EK, CD, 128, 1>(p, nb, s) : launch_block_bits<EK, CD, 128, 2>(p, nb, s);
}

}  // namespace

// dpad 64 / 128, 16-bit centroids, cols 256 or 512 query tokens per group.
int launch_plaid_block(int ek, int cd, int dpad, int cols, const Params& p, int64_t nb, hipStream_t s) {
  if (nb <= 0) return LIK_OK;
  if (nb > 0x7fffffffLL) return LIK_ERR_UNSUPPORTED;
  if (ek == EK_BF16)
    return cd == EK_BF16 ? launch_block_dpad<EK_BF16, EK_BF16>(dpad, cols, p, nb, s)
                         : launch_block_dpad<EK_BF16, EK_F16>(dpad, cols, p, nb, s);
  return cd == EK_BF16 ? launch_block_dpad<EK_F16, EK_BF16>(dpad, cols, p, nb, s)
                       : launch_block_dpad<EK_F16, EK_F16>(dpad, cols, p, nb, s);
}

}  // namespace lik
