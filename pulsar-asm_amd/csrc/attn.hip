// attn.hip -- split-K flash-decode attention over an fp16 KV cache (gfx950).
//
// Positions are cut into splits of 64; pass 1 computes, per (kv head, split,
// query), the G = nh/nkv heads' partial softmax state (for many queries in
// matrix tiles), pass 2 merges the
// splits of each head in ascending order and applies the per-head sigmoid
// gate (optionally emitting the Q8_0 input of o_proj). head_dim 64 or 128; a
// sliding-window layer (win > 0) sees keys [npos - win, npos) once npos > win.
// Order (the same on the host side):
//   dot_p = fmaf chain over d ascending of q_d * f16(k_pd), s_p = fl(dot_p * scale)
//   split j: m_j = max s_p, e_p = expf(fl(s_p - m_j)), l_j = pairwise sum of the
//            64 slots (zero past npos), o_jd = fmaf chain over p ascending of e_p * v_pd
//   M = max m_j; w_j = expf(fl(m_j - M)); L = fmaf(l_j, w_j, L); O_d = fmaf(o_jd, w_j, O_d)
//   out_d = bf16(fl(O_d / L)), then bf16(out_d * sigmoid(gate_h)).
// Query t of a T-position call sits at position pos0 + t and sees keys
// [0, pos0 + t] (causal), so a prefill chunk and T single-position calls give
// the same bits. The GQA head map h -> h / (nh/nkv) is lfm3_nanode.cu:520.
#include "pq_device.h"
#include "pq_host.h"
#include "pq_internal.h"
#include "q8_common.h"

namespace pq {

constexpr int kSplit = 64;

// One wave per (kv head g, split j, query t); lane p = position 64j + p for the
// scores, lane l = dimensions l + 64e (e < HD/64) for the value sums; the G
// heads of the group share every K and V load. Splits with no key in the
// window write nothing (the merge starts at the window's first split); the
// slots before lo are absent (no score, e = 0, skipped in the value chain).
template <int G, int HD>
__global__ __launch_bounds__(64) void attn_split_kernel(const uint16_t *__restrict__ q, int q_stride,
                                                         const uint16_t *__restrict__ kc,
                                                         const uint16_t *__restrict__ vc, float *__restrict__ po,
                                                         float *__restrict__ pml, int pos0, int nh, int nkv, int nsplit_max, float scale,
                                                         int win, const int32_t *__restrict__ pos_dev) {
  constexpr int E = HD / 64;
  __shared__ __align__(16) float qs[G][HD];
  __shared__ float es[G][kSplit];
  const int g = blockIdx.x, j = blockIdx.y, t = blockIdx.z, lane = threadIdx.x;
  const int npos = (pos_dev != nullptr ? *pos_dev : pos0) + t + 1;
  const int lo = window_lo(npos, win);
  const int p0 = j * kSplit;
  if (p0 >= npos || p0 + kSplit <= lo) return;
  const int pn = npos - p0 < kSplit ? npos - p0 : kSplit;
  const int i0 = lo > p0 ? lo - p0 : 0;
  const int kvd = nkv * HD;
#pragma unroll
  for (int h = 0; h < G; h++)
#pragma unroll
    for (int e = 0; e < E; e++) qs[h][lane + 64 * e] = bf2f(q[(size_t)t * q_stride + (g * G + h) * HD + lane + 64 * e]);
  __syncthreads();
  const bool valid = lane >= i0 && lane < pn;
  float dot[G];
#pragma unroll
  for (int h = 0; h < G; h++) dot[h] = 0.0f;
  if (valid) {
    const uint16_t *kr = kc + (size_t)(p0 + lane) * kvd + g * HD;
    for (int d0 = 0; d0 < HD; d0 += 8) {
      const uint4 k8 = *reinterpret_cast<const uint4 *>(kr + d0);
      const uint32_t kw[4] = {k8.x, k8.y, k8.z, k8.w};
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float kf = h2f((uint16_t)(kw[i >> 1] >> (16 * (i & 1))));
#pragma unroll
        for (int h = 0; h < G; h++) dot[h] = __builtin_fmaf(qs[h][d0 + i], kf, dot[h]);
      }
    }
  }
  float m[G], l[G];
#pragma unroll
  for (int h = 0; h < G; h++) {
    const float sc = valid ? dot[h] * scale : -__builtin_inff();
    m[h] = wave_max(sc);
    const float e = valid ? expf_pq(sc - m[h]) : 0.0f;
    l[h] = wave_pairwise_sum(e);
    es[h][lane] = e;
  }
  __syncthreads();
  float o[G][E];
#pragma unroll
  for (int h = 0; h < G; h++)
#pragma unroll
    for (int e = 0; e < E; e++) o[h][e] = 0.0f;
  for (int p = i0; p < pn; p++) {
#pragma unroll
    for (int e = 0; e < E; e++) {
      const float v = h2f(vc[(size_t)(p0 + p) * kvd + g * HD + lane + 64 * e]);
#pragma unroll
      for (int h = 0; h < G; h++) o[h][e] = __builtin_fmaf(es[h][p], v, o[h][e]);
    }
  }
#pragma unroll
  for (int h = 0; h < G; h++) {
    const size_t pj = ((size_t)t * nh + g * G + h) * nsplit_max + j;
#pragma unroll
    for (int e = 0; e < E; e++) po[pj * HD + lane + 64 * e] = o[h][e];
    if (lane == 0) {
      pml[2 * pj] = m[h];
      pml[2 * pj + 1] = l[h];
    }
  }
}

// The same partials for many queries, on the fp32 matrix cores: one wave per
// (kv head g, split j, tile of 32 rows), row i = head g*G + i % G of query
// t0 + i / G, so the G heads of 32 / G queries share the split's K and V. A
// step of v_mfma_f32_32x32x2 computes fma(a_1, b_1, fma(a_0, b_0, c)), each fma
// rounded once, k ascending: the score's chain over d and the value chain over
// p are such steps from C = 0 (a masked key adds fma(0, v, o) = o).
//
// Scores: A = K (32 keys), B = q, so a lane holds 32 scores of its own row (key
// 32u + 8i + 4h + c, h its half): the max is in-lane but for one half swap,
// the pairwise tree likewise (its first two levels and the last three within
// the lane, the third across the halves). e stays in registers: one half swap
// per pair turns keys (4h + 2b + c) into the order (2b + h) that the value
// steps read them in, A = V (32 dims), B = e. K comes in half rows per lane
// (the same swap hands each lane its parity of d), V as HD/32 adjacent dims
// per lane, straight from the cache: no LDS.
//
// A split that some row sees only in part may hold keys whose V a row must not
// touch; if V is not finite there, 0 * v would reach it, so that wave takes the
// value sums key by key instead (es in LDS).
//
// What bounds it: per split and 32 rows 2 HD MFMA steps (64 cycles and more)
// and about 1400 vector instructions (head_dim 64), 900 of them e^x. 512
// queries from 0, 32 q and 8 kv heads of 64: 60.4 -> 25.6 us (a wave per query
// read each K and V once per query and formed every chain on the vector unit).
typedef float v16f __attribute__((ext_vector_type(16)));

// a's upper with b's lower half of the wave exchanged
__device__ __forceinline__ void swap_halves(float &a, float &b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}

template <int G, int HD>
__global__ __launch_bounds__(64, 2) void attn_tile_kernel(const uint16_t *__restrict__ q, int q_stride, int qvec,
                                                        const uint16_t *__restrict__ kc,
                                                        const uint16_t *__restrict__ vc, float *__restrict__ po,
                                                        float *__restrict__ pml, int pos0, int T, int nh, int nkv,
                                                        int nsplit_max, float scale, int win) {
  constexpr int TP = 32 / G, MS = HD / 2, VD = HD / 32;
  __shared__ float es[32][kSplit + 1];
  const int g = blockIdx.x, j = blockIdx.y, t0 = blockIdx.z * TP, lane = threadIdx.x;
  const int l32 = lane & 31, h = lane >> 5;
  const int tl = (t0 + TP < T ? t0 + TP : T) - 1;   // the tile's last query
  const int p0 = j * kSplit, first = pos0 + t0 + 1, last = pos0 + tl + 1;   // npos of the first and the last query
  if (p0 >= last || p0 + kSplit <= window_lo(first, win)) return;
  const bool mixed = p0 + kSplit > first || p0 < window_lo(last, win);   // some row sees only a part of the split
  const int t = t0 + l32 / G, tc = t < tl ? t : tl, head = g * G + l32 % G;
  const int npos = pos0 + tc + 1, lo = window_lo(npos, win);
  const int kvd = nkv * HD;
  // the split's rows of the cache up to the last query's position; rows past it read zeros
  const int rows = last - p0 < kSplit ? last - p0 : kSplit;
  const size_t base = (size_t)p0 * kvd + (size_t)g * HD;
  const int lim = ((rows - 1) * kvd + HD) * 2;
  const __amdgpu_buffer_rsrc_t rk =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(kc + base), (short)0, lim, kRsrcWord3);
  const __amdgpu_buffer_rsrc_t rv =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(vc + base), (short)0, lim, kRsrcWord3);
  v4i kw[2][HD / 16];
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int i = 0; i < HD / 16; i++)
      kw[u][i] = __builtin_amdgcn_raw_buffer_load_b128(rk, ((32 * u + l32) * kvd + h * (HD / 2)) * 2 + 16 * i, 0, 0);
  // q: element 2m + h of the lane's row
  float qf[MS];
  const uint16_t *qr = q + (size_t)tc * q_stride + (size_t)head * HD;
  if (qvec) {
#pragma unroll
    for (int i = 0; i < HD / 16; i++) {
      const v4i w = *reinterpret_cast<const v4i *>(qr + h * (HD / 2) + 8 * i);
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int m = 4 * i + k;
        qf[m] = __uint_as_float((uint32_t)w[k] << 16);
        qf[MS / 2 + m] = __uint_as_float((uint32_t)w[k] & 0xffff0000u);
        swap_halves(qf[m], qf[MS / 2 + m]);
      }
    }
  } else {
#pragma unroll
    for (int m = 0; m < MS; m++) qf[m] = bf2f(qr[2 * m + h]);
  }
  const v16f zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  v16f sc[2];
#pragma unroll
  for (int u = 0; u < 2; u++) {
    float kf[MS];
#pragma unroll
    for (int i = 0; i < HD / 16; i++)
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int m = 4 * i + k;
        const uint32_t w = (uint32_t)kw[u][i][k];
        kf[m] = h2f((uint16_t)(w & 0xffffu));
        kf[MS / 2 + m] = h2f((uint16_t)(w >> 16));
        swap_halves(kf[m], kf[MS / 2 + m]);
      }
    sc[u] = zero;
#pragma unroll
    for (int m = 0; m < MS; m++) sc[u] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[m], qf[m], sc[u], 0, 0, 0);
  }
  // V on its way while the softmax runs: key 2m + h, dims VD * l32 and on
  uint32_t vw[32][VD / 2];
#pragma unroll
  for (int m = 0; m < 32; m++) {
    const int off = (2 * m + h) * kvd * 2 + l32 * VD * 2;
    if constexpr (VD == 2) {
      vw[m][0] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rv, off, 0, 0);
    } else {
      const v2i w = __builtin_amdgcn_raw_buffer_load_b64(rv, off, 0, 0);
      vw[m][0] = (uint32_t)w.x;
      vw[m][1] = (uint32_t)w.y;
    }
  }
  const int kn = npos - p0, kl = lo - p0;   // the row's keys of the split: [kl, kn)
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      sc[u][r] = sc[u][r] * scale;
      const int p = 32 * u + 8 * (r >> 2) + 4 * h + (r & 3);
      if (mixed) sc[u][r] = p >= kl && p < kn ? sc[u][r] : -__builtin_inff();
    }
  float m = fmaxf(sc[0][0], sc[1][0]);
#pragma unroll
  for (int r = 1; r < 16; r++) m = fmaxf(m, fmaxf(sc[0][r], sc[1][r]));
  m = max_half_pair(m);
  // e (0 at absent keys: e^-inf; a row with no key here is not stored) and its pairwise sum
  float ls[8];
#pragma unroll
  for (int u = 0; u < 2; u++) {
#pragma unroll
    for (int r = 0; r < 16; r++) sc[u][r] = expf_pq(sc[u][r] - m);
#pragma unroll
    for (int i = 0; i < 4; i++)
      ls[4 * u + i] = add_half_pair((sc[u][4 * i] + sc[u][4 * i + 1]) + (sc[u][4 * i + 2] + sc[u][4 * i + 3]));
  }
  const float l = ((ls[0] + ls[1]) + (ls[2] + ls[3])) + ((ls[4] + ls[5]) + (ls[6] + ls[7]));
  const bool store = t <= tl && p0 < npos && p0 + kSplit > lo;
  const size_t pj = ((size_t)tc * nh + head) * nsplit_max + j;
  if (store && h == 0) *reinterpret_cast<float2 *>(pml + 2 * pj) = make_float2(m, l);
  if (mixed) {
    bool odd = false;
#pragma unroll
    for (int k = 0; k < 32; k++)
#pragma unroll
      for (int d = 0; d < VD / 2; d++)
        odd = odd || (vw[k][d] & 0x7c00u) == 0x7c00u || (vw[k][d] & 0x7c000000u) == 0x7c000000u;
    if (__any(odd)) {   // key by key: lane = dims lane + 64e of one row after the other
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int r = 0; r < 16; r++) es[l32][32 * u + 8 * (r >> 2) + 4 * h + (r & 3)] = sc[u][r];
      __syncthreads();
      for (int i = 0; i < 32; i++) {
        const int ti = t0 + i / G;
        if (ti > tl) break;
        const int np = pos0 + ti + 1, pl = window_lo(np, win);
        if (p0 >= np || p0 + kSplit <= pl) continue;
        const int b = np - p0 < kSplit ? np - p0 : kSplit;
        for (int d = lane; d < HD; d += 64) {
          float o = 0.0f;
          for (int p = pl > p0 ? pl - p0 : 0; p < b; p++)
            o = __builtin_fmaf(es[i][p], h2f(vc[base + (size_t)p * kvd + d]), o);
          po[(((size_t)ti * nh + g * G + i % G) * nsplit_max + j) * HD + d] = o;
        }
      }
      return;
    }
  }
  // value steps: key pair (2m, 2m + 1) of e
  float ev[32];
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int b = 0; b < 2; b++) {
        float a0 = sc[u][4 * i + 2 * b], a1 = sc[u][4 * i + 2 * b + 1];
        swap_halves(a0, a1);
        ev[16 * u + 4 * i + b] = a0;
        ev[16 * u + 4 * i + 2 + b] = a1;
      }
  v16f o[VD];
#pragma unroll
  for (int d = 0; d < VD; d++) o[d] = zero;
#pragma unroll
  for (int k = 0; k < 32; k++)
#pragma unroll
    for (int d = 0; d < VD; d++) {
      const float vf = h2f((uint16_t)((vw[k][d >> 1] >> (16 * (d & 1))) & 0xffffu));
      o[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf, ev[k], o[d], 0, 0, 0);
    }
  // the lane's dims VD * (8i + 4h + c) + d of its row: 4 VD adjacent floats per i
  if (!store) return;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    float f[4 * VD];
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int d = 0; d < VD; d++) f[c * VD + d] = o[d][4 * i + c];
    float4 *dst = reinterpret_cast<float4 *>(po + pj * HD + VD * (8 * i + 4 * h));
#pragma unroll
    for (int k = 0; k < VD; k++) dst[k] = make_float4(f[4 * k], f[4 * k + 1], f[4 * k + 2], f[4 * k + 3]);
  }
}

// One wave per (head, query), 4 heads a workgroup; lane l = dimensions l + 64e.
// The window's splits merge in ascending order; lane i forms the weight of
// split c + i of a run of 64, and the partials load 8 at a time ahead of the
// chain -- a load a step, waited for, bound it: 512 queries of 32 heads over 1 to
// 8 splits 15.0 -> 9.9 us, one query over 24 about 14 us less.
template <int HD>
__global__ __launch_bounds__(256) void attn_merge_kernel(const float *__restrict__ po, const float *__restrict__ pml,
                                                          int pos0, int nh, int nsplit_max,
                                                          const uint16_t *__restrict__ gate, int gate_stride,
                                                          uint16_t *__restrict__ out, int out_stride,
                                                          int8_t *__restrict__ qx, float *__restrict__ dx, int win,
                                                          const int32_t *__restrict__ pos_dev) {
  constexpr int E = HD / 64;
  const int h = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t = blockIdx.y;
  const int d = threadIdx.x & 63;
  if (h >= nh) return;
  const int npos = (pos_dev != nullptr ? *pos_dev : pos0) + t + 1;
  const int j0 = window_lo(npos, win) / kSplit;
  const int ns = (npos + kSplit - 1) / kSplit;
  const size_t row = ((size_t)t * nh + h) * nsplit_max;
  const float2 *ml = reinterpret_cast<const float2 *>(pml) + row;
  const float *pr = po + row * HD + d;
  float M = -__builtin_inff();
  for (int c = j0; c < ns; c += 64) M = fmaxf(M, c + d < ns ? ml[c + d].x : -__builtin_inff());
  M = wave_max(M);
  float L = 0.0f, O[E];
#pragma unroll
  for (int e = 0; e < E; e++) O[e] = 0.0f;
  for (int c = j0; c < ns; c += 64) {
    const float2 mine = c + d < ns ? ml[c + d] : make_float2(0.0f, 0.0f);
    const float wl = expf_pq(mine.x - M);
    const int n = ns - c < 64 ? ns - c : 64;
    for (int i0 = 0; i0 < n; i0 += 8) {
      float p[8][E];
#pragma unroll
      for (int i = 0; i < 8; i++)
#pragma unroll
        for (int e = 0; e < E; e++) p[i][e] = i0 + i < n ? pr[(size_t)(c + i0 + i) * HD + 64 * e] : 0.0f;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        if (i0 + i >= n) break;
        const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wl), i0 + i));
        L = __builtin_fmaf(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(mine.y), i0 + i)), w, L);
#pragma unroll
        for (int e = 0; e < E; e++) O[e] = __builtin_fmaf(p[i][e], w, O[e]);
      }
    }
  }
  const float gs = gate != nullptr ? 1.0f / (1.0f + expf_pq(-bf2f(gate[(size_t)t * gate_stride + h]))) : 0.0f;
#pragma unroll
  for (int e = 0; e < E; e++) {
    uint16_t r = f2bf(O[e] / L);
    if (gate != nullptr) r = f2bf(bf2f(r) * gs);
    const int dd = d + 64 * e;
    if (out != nullptr) out[(size_t)t * out_stride + h * HD + dd] = r;
    if (qx != nullptr) {
      const float v = bf2f(r);
      float a = fabsf(v);
#pragma unroll
      for (int o = 1; o < 32; o <<= 1) a = fmaxf(a, __shfl_xor(a, o, 64));
      const float dq = a / 127.0f;
      // d = 0 only when every |x| of the block is below 127 * 2^-149: dividing
      // by 1 then gives q = 0 as the zero-block rule does, with no branch
      int qv = (int)__builtin_rintf(v / (dq != 0.0f ? dq : 1.0f));
      qv = qv > 127 ? 127 : (qv < -127 ? -127 : qv);
      const size_t K = (size_t)nh * HD;
      qx[(size_t)t * K + h * HD + dd] = (int8_t)qv;
      if ((d & 31) == 0) dx[(size_t)t * (K / 32) + (h * HD + dd) / 32] = dq;
    }
  }
}

}  // namespace pq

using namespace pq;

extern "C" size_t pq_attn_workspace_bytes(int nh, int hd, int max_pos, int T) {
  if (nh <= 0 || (hd != 64 && hd != 128) || max_pos <= 0 || T <= 0) return 0;
  const size_t ns = (size_t)(max_pos + kSplit - 1) / kSplit;
  return (size_t)T * nh * ns * (hd + 2) * sizeof(float);
}

// Matrix tiles when the per-query kernel's waves (one per kv head, query and
// split that the query sees; each costs by its G heads) fill the chip several
// times over: a tile wave takes about 7 us (head_dim 128: 14) however few of its
// rows are queries. Measured with the merge, per query / tiles (us): 32 q and 8
// kv heads of 64, 64 queries from 0 (512 waves) 13.3 / 15.8, 16 from 1500 (3072)
// 17.8 / 17.2, 203 from 0 (3424) 22.9 / 18.1, 512 from 0 (18432) 62.8 / 34.9, 512
// from 1500 263 / 129; 16 and 4 heads of 128, 203 from 0 (1712) 23.1 / 25.2, 203 in
// a window of 256 (4060) 33.2 / 34.2, 64 from 1500 (6400) 50.6 / 29.8, 512 from
// 1500 235 / 128; 8 and 1 of 128, 203 from 0 (428) 22.1 / 23.3, 512 (2304) 39.3 / 29.6.
// One query has as many tile waves as per-query ones. The per-query wave, which
// costs by its heads, is then the cheaper one but for 8 heads, or 4 of 128 once
// 4096 of its waves fill the chip: from 30000 keys 32 and 8 heads of 64 71.8 /
// 72.8, from 64000 128 / 142, 32 and 32 from 16000 56.5 / 74.7, 32 and 16 of 128 from
// 24000 85.0 / 115; 64 and 8 of 64 from 12500 45.2 / 37.0, 64 and 8 of 128 from 48000
// 207 / 159, 16 and 4 of 128 from 66000 (4128 waves) 165 / 176, from 90000 272 / 228, 32
// and 8 from 36000 (4504) 146 / 126. Two queries share the tiles: 32 and 8 of 64 from
// 64000 161 / 143, 32 and 32 from 16000 85.5 / 77.3.
static bool attn_tiles(int HD, int G, int nkv, int pos0, int T, int win) {
  auto splits = [&](long long npos) {
    const long long lo = win > 0 && npos > win ? npos - win : 0;
    return (npos + kSplit - 1) / kSplit - lo / kSplit;
  };
  const long long waves = nkv * (long long)T * (splits(pos0 + 1LL) + splits((long long)pos0 + T)) / 2;
  if (T < 2 && G <= 4 && !(G == 4 && HD == 128 && waves >= 4500)) return false;
  return waves * (G > 4 ? 2 : 1) >= (HD == 64 ? 3072 : 4096);
}

extern "C" int pq_attn_decode_form(int nh, int nkv, int hd, int pos0, int T, int win) {
  if (nkv <= 0 || nh <= 0 || nh % nkv || (hd != 64 && hd != 128) || pos0 < 0 || T <= 0 || win < 0) return -1;
  const int G = nh / nkv;
  if (G != 1 && G != 2 && G != 4 && G != 8) return -1;
  return attn_tiles(hd, G, nkv, pos0, T, win) ? 1 : 0;
}

template <int HD>
static int attn_launch(const uint16_t *q, int q_stride, const uint16_t *kcache, const uint16_t *vcache,
                       const uint16_t *gate, int gate_stride, uint16_t *out, int out_stride, int8_t *qx, float *dx,
                       int pos0, const int32_t *pos_dev, int nh, int nkv, int T, float scale, int win, float *part,
                       int nsplit, hipStream_t st) {
  const int G = nh / nkv;
  // the partials: o [T][nh][nsplit][HD], then the (m, l) pairs
  float *pml = part + (size_t)T * nh * nsplit * HD;
  const int TP = G > 0 && G <= 8 ? 32 / G : 0;
  const bool tiles = pos_dev == nullptr && aligned(part, 16) && attn_tiles(HD, G, nkv, pos0, T, win);
  const int qvec = aligned(q, 16) && q_stride % 8 == 0 ? 1 : 0;
  const dim3 g1(nkv, nsplit, T), b1(64), g2(nkv, nsplit, TP > 0 ? (T + TP - 1) / TP : 1);
#define PQ_ATTN(GG)                                                                                                 \
  if (tiles)                                                                                                        \
    launch(attn_tile_kernel<GG, HD>, g2, b1, 0, st, q, q_stride, qvec, kcache, vcache, part, pml, pos0, T, nh, nkv, \
           nsplit, scale, win);                                                                                     \
  else                                                                                                              \
    launch(attn_split_kernel<GG, HD>, g1, b1, 0, st, q, q_stride, kcache, vcache, part, pml, pos0, nh, nkv, nsplit, \
           scale, win, pos_dev)
  switch (G) {
    case 1: PQ_ATTN(1); break;
    case 2: PQ_ATTN(2); break;
    case 4: PQ_ATTN(4); break;
    case 8: PQ_ATTN(8); break;
    default: return fail(PQ_ERR_ARG, "pq_attn_decode: %d q heads per kv head (1, 2, 4 or 8)", G);
  }
#undef PQ_ATTN
  int rc = check_launch("pq_attn_decode split");
  if (rc) return rc;
  launch(attn_merge_kernel<HD>, dim3((nh + 3) / 4, T), dim3(256), 0, st, part, pml, pos0, nh, nsplit, gate,
         gate_stride, out, out_stride, qx, dx, win, pos_dev);
  return check_launch("pq_attn_decode merge");
}

extern "C" int pq_attn_decode(const uint16_t *q, int q_stride, const uint16_t *kcache, const uint16_t *vcache,
                              const uint16_t *gate, int gate_stride, uint16_t *out, int out_stride, int8_t *qx,
                              float *dx, int pos0, int nh, int nkv, int hd, int T, float scale, int win, void *ws,
                              size_t ws_bytes, void *stream) {
  PQ_REQUIRE(q && kcache && vcache && (out || qx) && (!qx || dx), PQ_ERR_ARG, "pq_attn_decode: null pointer");
  PQ_REQUIRE(hd == 64 || hd == 128, PQ_ERR_ARG, "pq_attn_decode: head_dim %d (64 or 128)", hd);
  PQ_REQUIRE(nh > 0 && nkv > 0 && nh % nkv == 0 && T > 0 && pos0 >= 0 && win >= 0, PQ_ERR_ARG,
             "pq_attn_decode: nh=%d nkv=%d T=%d pos0=%d win=%d", nh, nkv, T, pos0, win);
  PQ_REQUIRE(aligned(kcache, 16) && aligned(vcache, 16), PQ_ERR_ALIGN, "pq_attn_decode: KV cache must be 16-byte aligned");
  const int max_pos = pos0 + T;
  const int nsplit = (max_pos + kSplit - 1) / kSplit;
  const size_t need = pq_attn_workspace_bytes(nh, hd, max_pos, T);
  PQ_REQUIRE(ws && ws_bytes >= need, PQ_ERR_WORKSPACE, "pq_attn_decode: workspace of %zu bytes needed (got %zu)", need,
             ws_bytes);
  float *part = reinterpret_cast<float *>(ws);
  hipStream_t st = as_stream(stream);
  if (hd == 64)
    return attn_launch<64>(q, q_stride, kcache, vcache, gate, gate_stride, out, out_stride, qx, dx, pos0, nullptr, nh,
                           nkv, T, scale, win, part, nsplit, st);
  return attn_launch<128>(q, q_stride, kcache, vcache, gate, gate_stride, out, out_stride, qx, dx, pos0, nullptr, nh,
                          nkv, T, scale, win, part, nsplit, st);
}

namespace pq {
// One query (T = 1) at the position *pos_dev holds: the split grid and the
// workspace cover positions below ctx, and the splits past the position
// return at once, so a captured launch replays for any position.
int attn_decode_dev(const uint16_t *q, int q_stride, const uint16_t *kcache, const uint16_t *vcache,
                    const uint16_t *gate, int gate_stride, uint16_t *out, int out_stride, int8_t *qx, float *dx,
                    const int32_t *pos_dev, int ctx, int nh, int nkv, int hd, float scale, int win, void *ws,
                    size_t ws_bytes, hipStream_t st) {
  PQ_REQUIRE(q && kcache && vcache && pos_dev && (out || qx) && (!qx || dx) && ctx > 0, PQ_ERR_ARG,
             "attn_decode_dev: bad arguments");
  PQ_REQUIRE(hd == 64 || hd == 128, PQ_ERR_ARG, "attn_decode_dev: head_dim %d", hd);
  const int nsplit = (ctx + kSplit - 1) / kSplit;
  PQ_REQUIRE(ws && ws_bytes >= pq_attn_workspace_bytes(nh, hd, ctx, 1), PQ_ERR_WORKSPACE,
             "attn_decode_dev: workspace too small");
  float *part = reinterpret_cast<float *>(ws);
  if (hd == 64)
    return attn_launch<64>(q, q_stride, kcache, vcache, gate, gate_stride, out, out_stride, qx, dx, 0, pos_dev, nh,
                           nkv, 1, scale, win, part, nsplit, st);
  return attn_launch<128>(q, q_stride, kcache, vcache, gate, gate_stride, out, out_stride, qx, dx, 0, pos_dev, nh,
                          nkv, 1, scale, win, part, nsplit, st);
}
}  // namespace pq
