// q8r_gemm.hip -- the reference-numerics Q8_0 GEMM over many positions on the
// fp32 matrix cores (gfx950), bit for bit pq_q8r_gemv's order (q8r.hip).
//
// The order needs, per output and 32-block, the chain dot = fmaf(c_j, x_j, dot)
// over j ascending from 0. gfx950's fp32 MFMA is that chain: a step of
// v_mfma_f32_32x32x2 computes fma(a_1, b_1, fma(a_0, b_0, c)), every fma rounded
// once and subnormals kept (compared with fmaf chains of 32: the same bits for
// 524288 outputs each of ordinary, wide-exponent, subnormal and overflowing
// inputs), so 16 steps from C = 0 give a block's 32 x 32 dots. The rest of the
// order -- acc = fmaf(s_b, dot, acc) over a leaf's blocks, the leaf tree, the
// sum over chunks -- stays on the vector unit.
//
// What bounds it: an fp32 MFMA step and vector instructions of any wave of the
// SIMD exclude each other (72 cycles a 32x32x2 step, 4 to 5 more for every
// vector instruction beside it, measured), so beyond the matrix rate (138
// TFLOP/s, measured) every vector instruction costs: 83 a block of 16 steps, of
// which 16 widen x, 16 convert codes, 16 scale, 12 fold the tree. Per launch
// with cold weights, before (each output's chain on the vector unit) and now:
// 15360 x 2048 at 256 positions 440 -> 171 us (94 TFLOP/s), 2048 x 7680 at 256
// 347 -> 82 us, 2048 x 2048 at 203 54 -> 25 us. Measured and left out: 64-row
// or 64-position workgroups of 16 waves with 4 classes (spills, 191 - 217 us at
// the first shape).
//
// A workgroup of S = 8 waves owns a tile of MT rows x MT positions (MT = 32, or
// 16 through v_mfma_f32_16x16x4). Wave w takes one class of leaves, L = w mod S:
// the first levels of the leaf tree (offsets 16 .. S) add leaves of one class,
// so the wave folds them by itself, walking its 32/S leaves in bit-reversed
// order with one held partial per level; the last log2(S) levels add the S
// waves' partials through LDS at the end of a chunk. The workgroup stages S
// adjacent blocks (one leaf per class) of its rows and positions at a time:
// whole cache lines from global memory, two stages ahead of their use in
// registers and one in LDS, one barrier per stage, and on through the chunks
// and the workgroup's next tiles, so only its first tile waits for memory.
// The staging sorts k by the lane group that an MFMA step reads it from (KH = 2
// or 4 groups: k mod KH) and places pieces by an xor of their block, which
// spreads the writes over the banks; a wave then reads its operands of a block
// in whole 16-byte (8-byte) pieces.
#include "pq_device.h"
#include "pq_host.h"
#include "q8_common.h"
#include "q8r_common.h"

namespace pq {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kRgS = 8;           // leaf classes = waves per workgroup
constexpr int kRgJ = 32 / kRgS;   // leaves per class
constexpr int kRgNT = 64 * kRgS;

template <int MT>
struct RTile;
template <>
struct RTile<32> {
  typedef v16f Acc;
  static __device__ __forceinline__ Acc mfma(float a, float b, Acc c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
  }
  // output register r of a lane: position of the tile (the row is lane % 32)
  static __device__ __forceinline__ int pos(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }
};
template <>
struct RTile<16> {
  typedef f4v Acc;
  static __device__ __forceinline__ Acc mfma(float a, float b, Acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int pos(int r, int h) { return 4 * h + r; }
};

template <int MT>
struct RGemm {
  static constexpr int R = MT * MT / 64;                 // output registers per lane
  static constexpr int kXP = MT / 16;                    // 16-byte pieces of x per thread and stage
  static constexpr int kXRow = kRgS * 64 + 16;           // bytes per staged position (16 B pad: rows 4 banks apart)
  static constexpr int kXBytes = MT * kXRow, kWBytes = MT * kRgS * 32, kStage = kXBytes + kWBytes;
  // [buffer 0][gap][buffer 1]: a buffer and the gap hold the S waves' partials
  static constexpr int kPart = kRgS * MT * MT * 4, kGap = kPart > kStage ? kPart - kStage : 0;
  static constexpr size_t kLds = 2 * (size_t)kStage + kGap;
  static constexpr int kPerCU = MT == 32 ? 2 : 4;        // workgroups a CU holds
};

// A stage: block i of leaves S*j .. S*j + S - 1 (j the bit reversal of jj) of
// chunk c of a tile (rows from r0, positions from t0).
struct RStage {
  int tile, r0, t0, c, jj, i;
};

template <int MT>
__global__ __launch_bounds__(kRgNT) void q8r_mfma_kernel(const int8_t *__restrict__ codes,
                                                          const float *__restrict__ scales,
                                                          const uint16_t *__restrict__ x, void *__restrict__ y,
                                                          int y_bf16, int N, int K, int T, int npt, int ntile) {
  using C = RGemm<MT>;
  using Acc = typename RTile<MT>::Acc;
  constexpr int S = kRgS, J = kRgJ, R = C::R, kXP = C::kXP, kLog = 2;
  constexpr int kYQ = R >= S ? R / S : 1;   // outputs per thread after the last tree levels (R < S: waves below R)
  static_assert(J == 1 << kLog, "tree levels of a class");
  extern __shared__ __align__(16) unsigned char gm[];
  const int nb = K / kQ, nbc = q8r_chunk(K) / kQ, nch = nb / nbc;
  const int tid = threadIdx.x, sl = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lm = lane & (MT - 1), h = lane / MT;
  // Workgroups go round-robin over the 8 XCDs: the position tiles of one row
  // tile run one after the other on one XCD, which then reads the row tile's
  // codes from its own L2.
  auto place = [&](RStage &st) {
    for (; st.tile < ntile; st.tile += gridDim.x) {
      const int idx = st.tile >> 3, q = idx / npt;
      st.r0 = (q * 8 + (st.tile & 7)) * MT;
      st.t0 = (idx - q * npt) * MT;
      if (st.r0 < N) return;
    }
  };
  // This thread's pieces of a stage: x piece xq (8 k) of positions xp + 16 q,
  // weight piece wq (16 codes) of row wr, and its lane's scale. Offsets from
  // the stage's first element are fixed; the resources move, ending where the
  // tensor ends (rows past N and positions past T read zeros).
  const int xp = tid / (4 * S), xq = tid % (4 * S), wr = tid / (2 * S), wq = tid % (2 * S);
  const bool has_w = wr < MT;
  const int xoff = xp * K * 2 + xq * 16, woff = has_w ? wr * K + wq * 16 : kRsrcOob, soff = (lm * nb + sl) * 4;
  v4i xr[kXP], wv;
  float sr;
  auto first = [&](int jj, int i) { return S * (int)(__builtin_bitreverse32((uint32_t)jj) >> (32 - kLog)) + 32 * i; };
  auto load = [&](const RStage &st) {
    if (st.tile >= ntile) return;
    const int b0 = st.c * nbc + first(st.jj, st.i), k0 = b0 * kQ;   // the stage's first block and k
    const int np = T - st.t0 < MT ? T - st.t0 : MT, nr = N - st.r0 < MT ? N - st.r0 : MT;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t *>(x + (size_t)st.t0 * K + k0), (short)0, (np * K - k0) * 2, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t *>(codes + (size_t)st.r0 * K + k0), (short)0, nr * K - k0, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(scales + (size_t)st.r0 * nb + b0), (short)0, (nr * nb - b0) * 4, kRsrcWord3);
#pragma unroll
    for (int q = 0; q < kXP; q++) xr[q] = __builtin_amdgcn_raw_buffer_load_b128(rx, xoff + q * 32 * K, 0, 0);
    wv = __builtin_amdgcn_raw_buffer_load_b128(rc, woff, 0, 0);
    sr = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, soff, 0, 0));
  };
  // Stage buffers: x as it is, [position][512 B + pad]; the codes sorted by
  // the lane group that an MFMA step reads them from, k mod (64 / MT): MT = 32
  // [block][k mod 2][row^g][16 B], MT = 16 [k mod 4][block][row^g][8 B], the
  // xor spreading a wave's writes over the banks.
  const int bk = wq >> 1;
  const int xst = xp * C::kXRow + xq * 16;
  const int wst = C::kXBytes + (MT == 32 ? (bk * 2 * MT + (wr ^ ((bk & 3) * 4))) * 16 + (wq & 1) * 8
                                         : (bk * MT + (wr ^ ((bk >> 1) * 4))) * 8 + (wq & 1) * 4);
  auto store = [&](unsigned char *buf) {
#pragma unroll
    for (int q = 0; q < kXP; q++) *reinterpret_cast<v4i *>(buf + xst + q * 16 * C::kXRow) = xr[q];
    const uint32_t w[4] = {(uint32_t)wv.x, (uint32_t)wv.y, (uint32_t)wv.z, (uint32_t)wv.w};
    unsigned char *d = buf + wst;
    if constexpr (MT == 32) {
      *reinterpret_cast<uint2 *>(d) = make_uint2(__builtin_amdgcn_perm(w[1], w[0], 0x06040200u),
                                                 __builtin_amdgcn_perm(w[3], w[2], 0x06040200u));
      *reinterpret_cast<uint2 *>(d + MT * 16) = make_uint2(__builtin_amdgcn_perm(w[1], w[0], 0x07050301u),
                                                           __builtin_amdgcn_perm(w[3], w[2], 0x07050301u));
    } else if (has_w) {
      const uint32_t a0 = __builtin_amdgcn_perm(w[1], w[0], 0x05010400u);
      const uint32_t a1 = __builtin_amdgcn_perm(w[1], w[0], 0x07030602u);
      const uint32_t b0 = __builtin_amdgcn_perm(w[3], w[2], 0x05010400u);
      const uint32_t b1 = __builtin_amdgcn_perm(w[3], w[2], 0x07030602u);
      *reinterpret_cast<uint32_t *>(d) = __builtin_amdgcn_perm(b0, a0, 0x05040100u);
      *reinterpret_cast<uint32_t *>(d + S * MT * 8) = __builtin_amdgcn_perm(b0, a0, 0x07060302u);
      *reinterpret_cast<uint32_t *>(d + 2 * S * MT * 8) = __builtin_amdgcn_perm(b1, a1, 0x05040100u);
      *reinterpret_cast<uint32_t *>(d + 3 * S * MT * 8) = __builtin_amdgcn_perm(b1, a1, 0x07060302u);
    }
  };
  // where this lane reads its operands of block sl, and the byte permute that widens its half of an x word pair
  const int xld = lm * C::kXRow + sl * 64;
  const int wld = C::kXBytes + (MT == 32 ? ((sl * 2 + h) * MT + (lm ^ ((sl & 3) * 4))) * 16
                                         : ((h * S + sl) * MT + (lm ^ ((sl >> 1) * 4))) * 8);
  const uint32_t xsel = 0x01000c0cu + (uint32_t)h * 0x02020000u;
  auto dots = [&](const unsigned char *buf) {
    Acc dot;
#pragma unroll
    for (int r = 0; r < R; r++) dot[r] = 0.0f;
    v4i xd[4];
#pragma unroll
    for (int p = 0; p < 4; p++) xd[p] = *reinterpret_cast<const v4i *>(buf + xld + p * 16);
    if constexpr (MT == 32) {
      const v4i wd = *reinterpret_cast<const v4i *>(buf + wld);
#pragma unroll
      for (int m = 0; m < 16; m++) {
        const uint32_t xw = (uint32_t)xd[m >> 2][m & 3], ww = (uint32_t)wd[m >> 2];
        dot = RTile<MT>::mfma(__uint_as_float(__builtin_amdgcn_perm(0u, xw, xsel)),
                              (float)(int8_t)((ww >> (8 * (m & 3))) & 0xffu), dot);
      }
    } else {
      const v2i wd = *reinterpret_cast<const v2i *>(buf + wld);
#pragma unroll
      for (int m = 0; m < 8; m++) {
        const uint32_t x0 = (uint32_t)xd[m >> 1][2 * (m & 1)], x1 = (uint32_t)xd[m >> 1][2 * (m & 1) + 1];
        const uint32_t ww = (uint32_t)wd[m >> 2];
        dot = RTile<MT>::mfma(__uint_as_float(__builtin_amdgcn_perm(x1, x0, xsel)),
                              (float)(int8_t)((ww >> (8 * (m & 3))) & 0xffu), dot);
      }
    }
    return dot;
  };
  auto next = [&](RStage st) {   // the next stage that holds a block of its chunk, through the workgroup's tiles
    st.i++;
    while (first(st.jj, st.i) >= nbc) {
      st.i = 0;
      if (++st.jj < J) continue;
      st.jj = 0;
      if (++st.c < nch) break;   // block 0 always is one
      st.c = 0;
      st.tile += gridDim.x;
      place(st);
      break;
    }
    return st;
  };
  RStage ld;
  ld.tile = blockIdx.x;
  ld.c = ld.jj = ld.i = 0;
  place(ld);
  RStage cst = ld;   // the tile being computed
  load(ld);
  float s_now = sr;
  unsigned char *b_cur = gm, *b_nxt = gm + C::kStage + C::kGap;
  store(b_cur);
  ld = next(ld);
  load(ld);
  lds_barrier();
  while (cst.tile < ntile) {
    float ysum[kYQ];
#pragma unroll
    for (int q = 0; q < kYQ; q++) ysum[q] = 0.0f;
    for (int c = 0; c < nch; c++) {
      Acc held[kLog + 1];
#pragma unroll
      for (int jj = 0; jj < J; jj++) {
        // One stage: the next one into the other buffer (every wave is past
        // it), the one after it on its way, then this wave's block of it.
        Acc acc;
#pragma unroll
        for (int r = 0; r < R; r++) acc[r] = 0.0f;
        for (int i = 0; first(jj, i) < nbc; i++) {
          const float s_next = sr;
          store(b_nxt);
          ld = next(ld);
          load(ld);
          if (first(jj, i) + sl < nbc) {
            const Acc dot = dots(b_cur);
#pragma unroll
            for (int r = 0; r < R; r++) acc[r] = __builtin_fmaf(s_now, dot[r], acc[r]);
          }
          s_now = s_next;
          unsigned char *b = b_cur;
          b_cur = b_nxt;
          b_nxt = b;
          lds_barrier();
        }
        // the leaf tree's levels within the class: leaf jj completes a pair on every level whose bits below are set
        int lv = 0;
#pragma unroll
        for (; (jj >> lv) & 1; lv++)
#pragma unroll
          for (int r = 0; r < R; r++) acc[r] = held[lv][r] + acc[r];
        held[lv] = acc;
      }
      // The last levels over the classes, in the free buffer and the gap:
      // thread (wave sl, lane) adds registers sl * kYQ .. of the lane.
      float *part = reinterpret_cast<float *>(b_nxt == gm ? gm : gm + C::kStage);
#pragma unroll
      for (int r = 0; r < R; r++) part[(sl * R + r) * 64 + lane] = held[kLog][r];
      lds_barrier();
      if (sl * kYQ < R) {
#pragma unroll
        for (int q = 0; q < kYQ; q++) {
          const float *pp = part + (sl * kYQ + q) * 64 + lane;
          float v[S];
#pragma unroll
          for (int w = 0; w < S; w++) v[w] = pp[w * R * 64];
#pragma unroll
          for (int o = S / 2; o >= 1; o >>= 1)
#pragma unroll
            for (int w = 0; w < o; w++) v[w] = v[w] + v[w + o];
          ysum[q] = ysum[q] + v[0];
        }
      }
      lds_barrier();   // the next stage is stored over the partials
    }
    const int row = cst.r0 + lm;
    if (sl * kYQ < R && row < N) {
#pragma unroll
      for (int q = 0; q < kYQ; q++) {
        const int pos = cst.t0 + RTile<MT>::pos(sl * kYQ + q, h);
        if (pos < T) {
          if (y_bf16) reinterpret_cast<uint16_t *>(y)[(size_t)pos * N + row] = f2bf(ysum[q]);
          else reinterpret_cast<float *>(y)[(size_t)pos * N + row] = ysum[q];
        }
      }
    }
    cst.tile += gridDim.x;
    place(cst);
  }
}

template <int MT>
static int q8r_mfma_go(const int8_t *codes, const float *scales, const uint16_t *x, void *y, int yb, int N, int K,
                       int T, hipStream_t st) {
  using C = RGemm<MT>;
  const int nrt = (N + MT - 1) / MT, npt = (T + MT - 1) / MT, ntile = (nrt + 7) / 8 * 8 * npt;
  const int most = C::kPerCU * 256;   // a multiple of 8: a workgroup's tiles keep their XCD
  const dim3 grid((unsigned)(ntile < most ? ntile : most)), block(kRgNT);
  launch(q8r_mfma_kernel<MT>, grid, block, C::kLds, st, codes, scales, x, y, yb, N, K, T, npt, ntile);
  return check_launch("pq_q8r_gemv");
}

// 16-position, 16-row tiles where 32-wide ones leave CUs idle or are mostly
// padding: a CU takes about 0.4 of a 32-wide tile's time for one (the 16x16x4
// step runs at 112 TFLOP/s and its operands serve half as many outputs: 63
// against 94 TFLOP/s where both fill the chip), so the form with less time on
// the busiest CU is taken. Measured, 32 / 16: 15360 x 2048 at 256 positions
// 171 / 257 us, 4096 x 4096 at 48 28.4 / 28.5, 2048 x 8192 at 64 53 / 40,
// 16384 x 2048 at 16 27 / 23, 2048 x 8192 at 32 53 / 29.
int q8r_mfma_tile(int N, int T) {
  auto rounds = [&](int mt) {
    return ((long long)((N + mt - 1) / mt) * ((T + mt - 1) / mt) + 255) / 256;   // tiles of the busiest of 256 CUs
  };
  return 2 * rounds(16) < 5 * rounds(32) ? 16 : 32;
}

int q8r_mfma(int mt, const int8_t *codes, const float *scales, const uint16_t *x, void *y, int yb, int N, int K, int T,
             hipStream_t st) {
  if (mt == 16) return q8r_mfma_go<16>(codes, scales, x, y, yb, N, K, T, st);
  return q8r_mfma_go<32>(codes, scales, x, y, yb, N, K, T, st);
}

}  // namespace pq
