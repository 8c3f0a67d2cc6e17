// qlow_gemm.hip -- the Q4 / Q5 GEMM over many positions on the fp32 matrix
// cores (gfx950), bit for bit pq_qlow_gemv's order (qlow.hip).
//
// Per output and 32-group the order needs four chains a_b of 8 steps
// fmaf(1 + q_k/128, x_k, a_b), k = b, b + 4, ..., b + 28. A step of
// v_mfma_f32_32x32x2 computes fma(a_1, b_1, fma(a_0, b_0, c)), each fma rounded
// once (q8r_gemm.hip), so 4 steps from C = 0 form one chain of a 32 x 32 tile,
// 16 steps the four. The step m of chain b takes k = 8m + b from lanes 0..31
// and k = 8m + 4 + b from lanes 32..63: the low and the high nibble of byte b
// of the packed word m. The rest -- (a0 + a1) + (a2 + a3), - sg, the two fmas
// of the slice's chain -- stays on the vector unit.
//
// 16 x 16 tiles do the same with v_mfma_f32_16x16x4 (4 k's a step, lanes of 16:
// 2 steps a chain, nibble h mod 2 of words h / 2 and h / 2 + 2), for shapes
// whose 32-wide tiles would leave SIMDs idle or be mostly padding.
//
// A = the codes (row = lane % MT), B = x (position = lane % MT), so a lane's
// outputs are rows of its own position: the group sum sg is one register of
// the lane, and the scale pairs are read as they lie, 4 rows a load, and widen
// inside the fma (v_fma_mix_f32).
//
// A wave walks one K slice of a tile, KG = 64 / MT groups at a time: lane
// (position, h) loads the 64 bytes of x of group g + h, widens them, sums them
// in order (sg of its group), and swaps between the lane groups hand every
// group's operands to the lanes that feed them -- x passes through no LDS and
// no barrier. A workgroup is 4 waves: the KS slices of 4 / KS row tiles, which
// meet in LDS once at the end, where they add in slice order.
//
// What bounds it: the fp32 MFMA steps, and beside them the vector instructions
// (the two exclude each other on a SIMD): per group of a 32-wide tile 96 for
// the epilogue's 6 per output, 41 to bring x into place, 24 (Q5: 33) for the
// codes, against 16 steps of 64 cycles or more. Per launch, before (every chain
// on the vector unit, 16 - 26 TFLOP/s) and now: Q5 16384 x 2048 at 77 positions
// 206 -> 84 us, at 256 660 -> 213 us (81 TFLOP/s); 2048 x 8192 at 77 166 -> 66 us,
// at 256 530 -> 114 us; Q4 2048 x 2048 at 256 77 -> 35 us.
#include "pq_device.h"
#include "pq_host.h"
#include "pq_internal.h"
#include "q8_common.h"

namespace pq {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));

constexpr int kQmNT = 256;   // 4 waves

template <int MT>
struct QmTile;
template <>
struct QmTile<32> {
  typedef v16f Acc;
  static __device__ __forceinline__ Acc mfma(float a, float b, Acc c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
  }
};
template <>
struct QmTile<16> {
  typedef f4v Acc;
  static __device__ __forceinline__ Acc mfma(float a, float b, Acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// Lane groups: MT lanes each, KG = 64 / MT of them (the k's of one MFMA step,
// and the groups a pass takes); M = 8 / KG steps a chain, R outputs a lane.
template <int MT>
struct QmLoad {   // KG groups of a wave's operands on their way
  static constexpr int KG = 64 / MT, M = 8 / KG;
  v4i x[4];            // the lane group's group: 32 bf16 of the lane's position
  uint32_t w[KG][M];   // the words the lane takes codes from
  uint32_t hp[KG];
};

// v[i] of lane group h becomes v[h] of lane group i (KG x KG, over the lane
// groups): swaps of halves, then of adjacent 16-lane rows.
__device__ __forceinline__ void qm_swap32(float &a, float &b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void qm_swap16(float &a, float &b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
template <int KG>
__device__ __forceinline__ void qm_transpose(float *v) {
  if constexpr (KG == 2) {
    qm_swap32(v[0], v[1]);
  } else {
    qm_swap32(v[0], v[2]);
    qm_swap32(v[1], v[3]);
    qm_swap16(v[0], v[1]);
    qm_swap16(v[2], v[3]);
  }
}

template <int B, int KS, int MT>
__global__ __launch_bounds__(kQmNT, 2) void qlow_mfma_kernel(const uint8_t *__restrict__ pc,
                                                              const uint32_t *__restrict__ ps,
                                                              const uint16_t *__restrict__ x, void *__restrict__ y,
                                                              int y_bf16, int N, int K, int T, int ldy, int npt) {
  using Load = QmLoad<MT>;
  using Acc = typename QmTile<MT>::Acc;
  constexpr int RT = 4 / KS, GW = B == 4 ? 32 : 40, KG = Load::KG, M = Load::M, R = MT * MT / 64;
  constexpr int kPart = MT * (MT + 1);   // floats of a wave's outputs in LDS: [row][MT + 1] positions
  __shared__ float part[4 * kPart];
  const int G = K / kQ, GL = G / KS;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lm = lane & (MT - 1), h = lane / MT;
  // Workgroups go round-robin over the 8 XCDs: the position tiles of one group
  // of row tiles run on one XCD, whose L2 then serves the codes again.
  const int idx = blockIdx.x >> 3, rg = (idx / npt) * 8 + (blockIdx.x & 7), t0 = (idx % npt) * MT;
  if (rg * RT * MT >= N) return;
  const int r0 = (rg * RT + wave / KS) * MT, s = wave % KS;   // the wave's first row, its K slice
  const int nt = T - t0 < MT ? T - t0 : MT;
  if (r0 < N) {
    const int tile = r0 >> 5, sub = r0 & 31;
    const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(pc + (size_t)tile * G * GW * 16), (short)0, G * GW * 16, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t *>(ps + (size_t)tile * G * 32), (short)0, G * 32 * 4, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t *>(x + (size_t)t0 * K), (short)0, nt * K * 2, kRsrcWord3);
    const int g1 = (s + 1) * GL;
    const int xo = (lm * K + h * kQ) * 2, wo = (sub + lm) * 16 + (MT == 16 ? (h >> 1) * 4 : 0);
    const int po = 32 * 16 + (sub + lm) * 4, so = (sub + 4 * h) * 4;
    auto load = [&](Load &L, int g) {   // groups past the slice repeat its last one, or (x) read another's: not used
#pragma unroll
      for (int i = 0; i < 4; i++) L.x[i] = __builtin_amdgcn_raw_buffer_load_b128(rx, xo + g * kQ * 2 + i * 16, 0, 0);
#pragma unroll
      for (int i = 0; i < KG; i++) {
        const int gi = (g + i < g1 ? g + i : g1 - 1) * GW * 16;
        if constexpr (MT == 32) {
          const v4i v = __builtin_amdgcn_raw_buffer_load_b128(rc, wo, gi, 0);
#pragma unroll
          for (int m = 0; m < M; m++) L.w[i][m] = (uint32_t)v[m];
        } else {
#pragma unroll
          for (int m = 0; m < M; m++) L.w[i][m] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rc, wo + 8 * m, gi, 0);
        }
        L.hp[i] = B == 5 ? (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rc, po, gi, 0) : 0u;
      }
    };
    Acc yv;
#pragma unroll
    for (int r = 0; r < R; r++) yv[r] = 0.0f;
    // One group: the chains' steps, then the slice chain's step of the lane's outputs.
    auto group = [&](const uint32_t *w, uint32_t hp, const float (*xv)[4], const v4i *sc, float sg) {
      Acc zero;
#pragma unroll
      for (int r = 0; r < R; r++) zero[r] = 0.0f;
      const uint32_t hs = hp >> h, sh = 4 * (h & 1);
      Acc a[4];
#pragma unroll
      for (int m = 0; m < M; m++) {
        // 0x80 | code of weight 4 (KG m + h) + b in byte b: with 0x3F above it, the float 1 + q/128
        uint32_t c = ((w[m] >> sh) & 0x0f0f0f0fu) | 0x80808080u;
        if constexpr (B == 5) {   // bit 4: the plane's bit 8b + KG m + h
          const uint32_t p = KG * m < 4 ? hs << (4 - KG * m) : hs >> (KG * m - 4);
          c = (p & 0x10101010u) | c;
        }
#pragma unroll
        for (int b = 0; b < 4; b++) {
          const float cf = __uint_as_float(__builtin_amdgcn_perm(0x3fu, c, 0x04000c0cu + ((uint32_t)b << 16)));
          a[b] = QmTile<MT>::mfma(cf, xv[m][b], m == 0 ? zero : a[b]);
        }
      }
#pragma unroll
      for (int r = 0; r < R; r++) {
        const float u = ((a[0][r] + a[1][r]) + (a[2][r] + a[3][r])) - sg;
        const h2v d = __builtin_bit_cast(h2v, (uint32_t)sc[r >> 2][r & 3]);   // (d', mn)
        yv[r] = __builtin_fmaf((float)d.x, u, __builtin_fmaf((float)d.y, sg, yv[r]));
      }
    };
    auto step = [&](const Load &L, Load &nxt, int g) {
      v4i sc[KG][R / 4];   // group g + i, rows 8q + 4h .. + 3
#pragma unroll
      for (int i = 0; i < KG; i++)
#pragma unroll
        for (int q = 0; q < R / 4; q++)
          sc[i][q] = __builtin_amdgcn_raw_buffer_load_b128(rs, so + q * 32, (g + i < g1 ? g + i : g1 - 1) * 128, 0);
      load(nxt, g + KG < g1 ? g + KG : g);
      float f[32];
#pragma unroll
      for (int k = 0; k < 16; k++) {
        const uint32_t v = (uint32_t)L.x[k >> 2][k & 3];
        f[2 * k] = __uint_as_float(v << 16);
        f[2 * k + 1] = __uint_as_float(v & 0xffff0000u);
      }
      float sg[KG];
      sg[0] = 0.0f;
#pragma unroll
      for (int k = 0; k < 32; k++) sg[0] = sg[0] + f[k];
#pragma unroll
      for (int i = 1; i < KG; i++) sg[i] = sg[0];
      qm_transpose<KG>(sg);   // lane group h's sum of group g + h: to every lane group
      // lane group h holds the quads of group g + h and takes quad KG m + h of each group
      float xv[KG][M][4];
#pragma unroll
      for (int m = 0; m < M; m++)
#pragma unroll
        for (int b = 0; b < 4; b++) {
          float v[KG];
#pragma unroll
          for (int i = 0; i < KG; i++) v[i] = f[4 * (KG * m + i) + b];
          qm_transpose<KG>(v);
#pragma unroll
          for (int i = 0; i < KG; i++) xv[i][m][b] = v[i];
        }
#pragma unroll
      for (int i = 0; i < KG; i++)
        if (KG == 2 || g + i < g1) group(L.w[i], L.hp[i], xv[i], sc[i], sg[i]);   // GL is even
    };
    // two register sets passed by name: no copy of a set still being loaded
    Load La, Lb;
    load(La, s * GL);
    for (int g = s * GL; g < g1; g += 2 * KG) {
      step(La, Lb, g);
      if (g + KG >= g1) break;
      step(Lb, La, g + KG);
    }
    float *pp = part + wave * kPart + lm;
#pragma unroll
    for (int r = 0; r < R; r++) pp[(MT / 4 * (r >> 2) + 4 * h + (r & 3)) * (MT + 1)] = yv[r];
  }
  __syncthreads();
  // outputs of the workgroup's row tiles: MT lanes write MT rows of one position
  for (int i = tid; i < RT * MT * MT; i += kQmNT) {
    const int rt = i / (MT * MT), p = i / MT % MT, row = i % MT;
    const int n = (rg * RT + rt) * MT + row;
    if (p >= nt || n >= N) continue;
    float v = 0.0f;
#pragma unroll
    for (int k = 0; k < KS; k++) v = v + part[(rt * KS + k) * kPart + row * (MT + 1) + p];
    const size_t o = (size_t)(t0 + p) * ldy + n;
    if (y_bf16) reinterpret_cast<uint16_t *>(y)[o] = f2bf(v);
    else reinterpret_cast<float *>(y)[o] = v;
  }
}

template <int MT>
static int qlow_mfma_go(const uint8_t *pc, const uint32_t *ps, const uint16_t *x, void *y, int yb, int N, int K, int T,
                        int ldy, int bits, int ks, hipStream_t st) {
  const int rt = 4 / ks, nrg = (N / MT + rt - 1) / rt, npt = (T + MT - 1) / MT;
  const dim3 grid((unsigned)((nrg + 7) / 8 * 8 * npt)), block(kQmNT);
#define PQ_QM(BB, SS) launch(qlow_mfma_kernel<BB, SS, MT>, grid, block, 0, st, pc, ps, x, y, yb, N, K, T, ldy, npt)
  if (bits == 4) {
    if (ks == 2) PQ_QM(4, 2);
    else PQ_QM(4, 4);
  } else {
    if (ks == 2) PQ_QM(5, 2);
    else PQ_QM(5, 4);
  }
#undef PQ_QM
  return check_launch("pq_qlow_gemm");
}

// Which form runs a T-position GEMM: 32 or 16 (the matrix tiles here) or 0 (the
// vector kernel of qlow.hip, rv rounds of 256 workgroups of rs x tb outputs),
// by the time of the busiest SIMD or CU, in ns per launch. A wave takes one
// slice of GL groups; the 1024 SIMDs run the waves in rounds, the first of them
// latency-bound. Fitted to (us, vector / 16 / 32; * the form taken), Q5:
//   16384 x 2048 at 8 positions 23.9* / 24.8 / 35, at 9 44.7 / 24.6* / 35, at
//   64 166 / 81 / 58*, at 77 206 / 99 / 84*, at 256 660 / 300 / 213*;
//   2048 x 8192 at 8 17.5* / 30 / 64, at 16 33.5 / 32.8* / 64, at 64 132 / 50* /
//   65, at 256 530 / 153 / 114*;
// Q4: 3072 x 2048 at 16 10.7* / 17.5 / 33, at 24 20.1 / 17.7* / 33; 64 x 1024 at
//   256 7.2* / 10.2 / 18.5.
int qlow_mfma_tile(int N, int K, int T, int ks, long long rv, int rs, int tb) {
  const long long GL = K / kQ / ks;
  auto rounds = [&](int mt) { return ((long long)(N / mt) * ((T + mt - 1) / mt) * ks + 1023) / 1024; };
  const long long t16 = GL * (250 + 280 * rounds(16)), t32 = GL * (300 + 800 * rounds(32));
  const long long tv = rv * (1500 + (long long)rs * tb * K / 75 + K * 5 / 12);
  if (tv <= t16 && tv <= t32) return 0;
  return t16 <= t32 ? 16 : 32;
}

int qlow_mfma(int mt, const uint8_t *pc, const uint32_t *ps, const uint16_t *x, void *y, int yb, int N, int K, int T,
              int ldy, int bits, int ks, hipStream_t st) {
  if (mt == 16) return qlow_mfma_go<16>(pc, ps, x, y, yb, N, K, T, ldy, bits, ks, st);
  return qlow_mfma_go<32>(pc, ps, x, y, yb, N, K, T, ldy, bits, ks, st);
}

}  // namespace pq
