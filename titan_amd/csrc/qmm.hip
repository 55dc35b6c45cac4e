// Dense quantized matmul for a batch of rows (mx.quantized_matmul with M > 1;
// smallm/kernel.py:38, 319-391): out[m, n] = x[m] . W[n]^T over MLX-layout
// weights with the exact affine values, fp32 accumulation.
//
// The GEMV (qmv.hip) streams the weights once per row of x; here each weight
// is read once per 16 * MT rows.  The codes go to the matrix cores as they
// are -- 4-bit codes as the bf16 values 1 + q / 128 (0x3F80 | q), 8-bit codes as
// the integers 0..255, all exact -- and the group's scale and bias are applied
// to the products' sums in fp32, so nothing is rounded to bf16 before the
// result, as in the GEMV:
//   acc += s * sum_k x q + b * sum_k x            per group
// with sum_k x from the same matrix instruction over a constant: for 4 bits
// the constant is -1, so that the sum is also what the products start from
// (sum x (1 + q / 128) - sum x), and the scale is multiplied by 128.  (128 + q
// would do without that and give the same bits, but 128 sum x overflows from
// sums of 2.7e36 on.)
//
// Work: a block owns 16 output columns of 16 * MT rows and its eight waves
// take the K = 256 batches (four 64-column units) in turn; their partial sums
// meet in LDS at the end and are added in wave order.  Lane (n = lane % 16,
// q = lane / 16) feeds the MFMAs codes 16 q .. 16 q + 15 of column n and the same
// columns of x row n of each unit.  Read straight into that layout, 16 rows
// under 16 neighbouring lanes, every load instruction costs its 64 lanes a
// cycle or more each (measured 70 to 80 cycles per instruction, the bound of
// the kernel built so: 5.9 us for 2 rows, 12.5 us for 64 at N = 4096, K = 2048, of
// which 2.8 without its loads), so each wave copies whole rows' lines into LDS
// instead (global_load_lds, 16-byte units XOR-swizzled by row) and reads its
// operands from there; its buffers are its own, so nothing waits on a barrier.
// One scale and one bias load per batch bring unit q's to lane (n, q), and
// lanes exchange them.
//
// Per call in a graph (us), against the GEMV's one weight pass per row:
//   N x K, bits, group    rows:   2          4          8         24         64
//   4096 x 2048, 4, 64      4.2/4.5    5.4/4.6    7.9/4.5   17.4/5.5   39.7/7.3
//   4096 x 2048, 8, 64      6.1/4.9    9.3/5.0   14.2/5.0   31.5/6.1   63.2/7.5
//   9216 x 2048, 4, 64      6.2/7.3    9.4/7.3   14.3/7.4   36.9/10.1  79.1/17.3
//   1000 x 2048, 4, 32      3.1/4.2    3.6/4.2    4.2/4.2    6.6/5.6   12.3/6.3
//   5120 x 2560, 8, 32     10.5/10.1  14.6/10.2  23.8/10.2  55.6/13.2 137.9/17.8
// A launch and its first dependent read take ~2.8 us of each; the error against
// 64-bit products is the GEMV's to four digits (0.0016 to 0.0017, the result's
// bf16 rounding).  Twice the units of x staged at a time measured 2-25% slower
// (144 KB of LDS and more: one block per CU.  The 8-bit form's 96 KB allow no
// second one as it is, but for three row tiles, 80 KB.)
#include "qmm.h"

#include "gemm_common.h"

namespace {

using qmoe_gemm::dma16;

constexpr int kWaves = 8;
constexpr int kMaxMT = 4;

struct QmmArgs {
  const uint16_t* x;
  int64_t M;
  int K;
  const uint32_t* w;
  const uint16_t* s;
  const uint16_t* b;
  int N;
  uint16_t* out;
};

typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4_t;

// x[8] as the bf16 pairs that match a code word's nibble pairs: (0,4) (1,5) (2,6) (3,7)
__device__ __forceinline__ u32x4_t pair_nibbles(const u32x4_t& a) {
  return u32x4_t{__builtin_amdgcn_perm(a[2], a[0], 0x05040100u), __builtin_amdgcn_perm(a[2], a[0], 0x07060302u),
                 __builtin_amdgcn_perm(a[3], a[1], 0x05040100u), __builtin_amdgcn_perm(a[3], a[1], 0x07060302u)};
}
// the eight 4-bit codes of a word as bf16 1 + q / 128, in that order
__device__ __forceinline__ u32x4_t codes4(uint32_t v) {
  constexpr uint32_t m = 0x000F000Fu, c = 0x3F803F80u;
  return u32x4_t{(v & m) | c, ((v >> 4) & m) | c, ((v >> 8) & m) | c, ((v >> 12) & m) | c};
}
// eight 8-bit codes of two words as bf16 integers (exact: the float's top half)
__device__ __forceinline__ u32x4_t codes8(uint32_t v0, uint32_t v1) {
  auto f = [](uint32_t v, int i) { return __float_as_uint((float)((v >> (8 * i)) & 0xFFu)); };
  return u32x4_t{__builtin_amdgcn_perm(f(v0, 1), f(v0, 0), 0x07060302u),
                 __builtin_amdgcn_perm(f(v0, 3), f(v0, 2), 0x07060302u),
                 __builtin_amdgcn_perm(f(v1, 1), f(v1, 0), 0x07060302u),
                 __builtin_amdgcn_perm(f(v1, 3), f(v1, 2), 0x07060302u)};
}
__device__ __forceinline__ f32x4_t mfma(const u32x4_t& a, const u32x4_t& b, const f32x4_t& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                 0, 0, 0);
}

template <int BITS, int GS, int MT>
struct Cfg {
  static constexpr int kUnits = 4;                           // units per batch
  static constexpr int kUX = MT == 1 ? 4 : MT == 2 ? 2 : 1;  // units of x staged at a time
  static constexpr int kSubs = kUnits / kUX;
  static constexpr int kXRow = 16 * MT * 128;                // bytes of one unit of x
  static constexpr int kXBytes = kUX * kXRow;
  static constexpr int kWRow = kUnits * 8 * BITS;            // bytes of a column's batch of codes
  static constexpr int kWBytes = 16 * kWRow;
  static constexpr int kWaveBytes = kXBytes + kWBytes;
  static constexpr int SG = GS == 32 ? 2 : 1;                // groups per unit
  static_assert(kWaves * kWaveBytes <= 96 * 1024 && kWaves * 16 * MT * 17 * 4 <= kWaves * kWaveBytes, "LDS");
};

// The wave's share of x for units u .. u + kUX - 1 (past the last: the last)
template <int BITS, int GS, int MT>
__device__ __forceinline__ void stage_x(const QmmArgs& a, int64_t m0, int u, uint32_t lds) {
  using C = Cfg<BITS, GS, MT>;
  const int lane = threadIdx.x % 64, U = a.K / 64;
#pragma unroll
  for (int j = 0; j < C::kUX; ++j) {
    const int uu = min(u + j, U - 1);
#pragma unroll
    for (int c = 0; c < 2 * MT; ++c) {
      const int r = 8 * c + lane / 8;
      const uint16_t* src = a.x + min(m0 + r, a.M - 1) * (int64_t)a.K + uu * 64 + ((lane & 7) ^ (r & 7)) * 8;
      dma16(src, lds + j * C::kXRow + c * 1024);
    }
  }
}

// The codes of the block's 16 columns for units u .. u + 3 (past the last: the last)
template <int BITS, int GS, int MT>
__device__ __forceinline__ void stage_w(const QmmArgs& a, int n0, int u, uint32_t lds) {
  using C = Cfg<BITS, GS, MT>;
  constexpr int PR = C::kWRow / 16;  // 16-byte pieces per column: 8 or 16
  constexpr int PU = PR / 4;         // and per unit
  const int lane = threadIdx.x % 64, U = a.K / 64;
#pragma unroll
  for (int c = 0; c < C::kWBytes / 1024; ++c) {
    const int r = (64 / PR) * c + lane / PR;
    const int piece = (lane % PR) ^ (r % PR);
    const int uu = min(u + piece / PU, U - 1);
    const uint32_t* src = a.w + min(n0 + r, a.N - 1) * (int64_t)(a.K * BITS / 32) + uu * (2 * BITS) + (piece % PU) * 4;
    dma16(src, lds + c * 1024);
  }
}

template <int BITS, int GS, int MT>
__global__ __launch_bounds__(64 * kWaves) void qmm_kernel(QmmArgs a) {
  using C = Cfg<BITS, GS, MT>;
  constexpr int SG = C::SG, UX = C::kUX;
  __shared__ __attribute__((aligned(1024))) char smem[kWaves * C::kWaveBytes];
  const int lane = threadIdx.x % 64, n16 = lane % 16, q = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  const int n0 = blockIdx.x * 16;
  const int64_t m0 = (int64_t)blockIdx.y * (16 * MT);
  const int G = a.K / GS, U = a.K / 64, batches = (U + 3) / 4;
  char* xl = smem + wave * C::kWaveBytes;
  char* wl = xl + C::kXBytes;
  const uint32_t xlds = __builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)xl), wlds = xlds + C::kXBytes;
  const int64_t n = min(n0 + n16, a.N - 1);  // columns and rows past the end repeat the last, and are not stored
  const uint16_t* srow = a.s + n * G;
  const uint16_t* brow = a.b + n * G;
  // scale | bias << 16 of the groups of unit u + q
  auto load_sb = [&](int u, uint32_t (&sb)[SG]) {
    const int uu = min(u + q, U - 1);
#pragma unroll
    for (int t = 0; t < SG; ++t) {
      const int g = GS == 128 ? uu / 2 : uu * SG + t;
      sb[t] = (uint32_t)srow[g] | (uint32_t)brow[g] << 16;
    }
  };

  const uint32_t one = BITS == 4 ? 0xBF80BF80u : 0x3F803F80u;  // bf16 -1 or 1
  const u32x4_t ones = {one, one, one, one};
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  f32x4_t acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = zero;

  uint32_t sb[SG];
  if (wave < batches) {
    stage_w<BITS, GS, MT>(a, n0, 4 * wave, wlds);
    stage_x<BITS, GS, MT>(a, m0, 4 * wave, xlds);
    load_sb(4 * wave, sb);
  }
  for (int bt = wave; bt < batches; bt += kWaves) {
    const int ub = 4 * bt;
    const int nb = min(bt + kWaves, batches - 1) * 4;  // the next batch (the last repeats itself)
    uint32_t cw[4][BITS / 2];
    uint32_t sbj[4][SG];
#pragma unroll
    for (int sub = 0; sub < C::kSubs; ++sub) {
      qmoe_gemm::wait_vmem<0>();
      if (sub == 0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (BITS == 4) {
            const uint2 t = *reinterpret_cast<const uint2*>(wl + n16 * C::kWRow + (((2 * j + (q >> 1)) ^ (n16 & 7)) * 16) +
                                                            8 * (q & 1));
            cw[j][0] = t.x;
            cw[j][1] = t.y;
          } else {
            const uint4 t = *reinterpret_cast<const uint4*>(wl + n16 * C::kWRow + ((4 * j + q) ^ n16) * 16);
            cw[j][0] = t.x;
            cw[j][1] = t.y;
            cw[j][2] = t.z;
            cw[j][3] = t.w;
          }
#pragma unroll
          for (int t = 0; t < SG; ++t) sbj[j][t] = (uint32_t)__shfl((int)sb[t], n16 + 16 * j, 64);
        }
      }
      u32x4_t xv[UX][MT][2];
#pragma unroll
      for (int j = 0; j < UX; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int t = 0; t < 2; ++t)
            xv[j][i][t] = *reinterpret_cast<const u32x4_t*>(xl + j * C::kXRow + (16 * i + n16) * 128 +
                                                            (((2 * q + t) ^ (n16 & 7)) * 16));
      // the reads are done before their buffers are filled again
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      const bool more = sub + 1 < C::kSubs;
      if (more || bt + kWaves < batches) {  // wave-uniform
        stage_x<BITS, GS, MT>(a, m0, more ? ub + (sub + 1) * UX : nb, xlds);
        if (!more) {
          stage_w<BITS, GS, MT>(a, n0, nb, wlds);
          load_sb(nb, sb);
        }
      }
#pragma unroll
      for (int jj = 0; jj < UX; ++jj) {
        const int j = sub * UX + jj;
        const bool live = ub + j < U;  // a unit past the end: scale and bias zero
        u32x4_t wf[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          if constexpr (BITS == 4) wf[t] = codes4(cw[j][t]);
          else wf[t] = codes8(cw[j][2 * t], cw[j][2 * t + 1]);
        }
#pragma unroll
        for (int sg = 0; sg < SG; ++sg) {
          const uint32_t w = live ? sbj[j][sg] : 0u;
          const float s = __uint_as_float(w << 16) * (BITS == 4 ? 128.0f : 1.0f);  // exact
          const float b = BITS == 4 ? -__uint_as_float(w & 0xFFFF0000u) : __uint_as_float(w & 0xFFFF0000u);
#pragma unroll
          for (int i = 0; i < MT; ++i) {
            u32x4_t xf[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
              xf[t] = BITS == 4 ? pair_nibbles(xv[jj][i][t]) : xv[jj][i][t];
              // group 32: lanes q < 2 hold the unit's first group, the others its second
              if (SG == 2 && (q >> 1) != sg) xf[t] = u32x4_t{0u, 0u, 0u, 0u};
            }
            const f32x4_t xs = mfma(xf[1], ones, mfma(xf[0], ones, zero));
            const f32x4_t d = mfma(xf[1], wf[1], mfma(xf[0], wf[0], BITS == 4 ? xs : zero));
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][r] = fmaf(b, xs[r], fmaf(s, d[r], acc[i][r]));
          }
        }
      }
    }
  }
  __syncthreads();  // every wave is done with its buffers
  float(*red)[16 * MT][17] = reinterpret_cast<float(*)[16 * MT][17]>(smem);

  // lane: column n16, rows 16 i + 4 q + r
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave][16 * i + 4 * q + r][n16] = acc[i][r];
  __syncthreads();
  for (int o = threadIdx.x; o < 256 * MT; o += 64 * kWaves) {
    const int m = o / 16, c = o % 16;
    float v = red[0][m][c];
#pragma unroll
    for (int wv = 1; wv < kWaves; ++wv) v += red[wv][m][c];
    if (m0 + m < a.M && n0 + c < a.N) a.out[(m0 + m) * a.N + n0 + c] = (uint16_t)f32_to_bf16(v);
  }
}

template <int BITS, int GS>
int launch_mt(const QmmArgs& a, hipStream_t st) {
  const int64_t tiles = (a.M + 15) / 16;
  // group 32 keeps each operand twice, masked by group: two row tiles are what its registers hold
  constexpr int kMax = GS == 32 ? 2 : kMaxMT;
  const int mt = tiles >= kMax ? kMax : (int)tiles;
  const dim3 grid((unsigned)((a.N + 15) / 16), (unsigned)((tiles + mt - 1) / mt)), block(64 * kWaves);
  switch (mt) {
    case 1: qmm_kernel<BITS, GS, 1><<<grid, block, 0, st>>>(a); break;
    case 2: qmm_kernel<BITS, GS, 2><<<grid, block, 0, st>>>(a); break;
    default:
      if constexpr (kMax > 2) {
        if (mt == 3) qmm_kernel<BITS, GS, 3><<<grid, block, 0, st>>>(a);
        else qmm_kernel<BITS, GS, 4><<<grid, block, 0, st>>>(a);
      }
  }
  return qmoe::launch_status("qmm_kernel");
}

template <int BITS>
int launch_gs(const QmmArgs& a, int group_size, hipStream_t st) {
  switch (group_size) {
    case 32: return launch_mt<BITS, 32>(a, st);
    case 64: return launch_mt<BITS, 64>(a, st);
    default: return launch_mt<BITS, 128>(a, st);
  }
}

}  // namespace

namespace qmoe_qmm {

bool takes(int64_t M, int64_t N, int64_t K, int group_size, int bits) {
  if (K % 64 || K > (1 << 24) || M > 65535LL * 32 || (bits != 4 && bits != 8)) return false;
  // The GEMV re-reads the weights for every row, at about 7 TB/s from the
  // caches; this kernel's time hardly depends on the rows up to 16 but starts
  // from a longer chain.  Over 1000 x 2048 to 9216 x 2048 and 2048 x 4096 they
  // meet between two and five rows of 4-bit codes (at four rows 5.2/4.5 us for
  // 4096 x 2048 but 5.2/5.6 for 2048 x 4096) and between two and three of 8-bit
  // ones (at three 7.1/4.9 and 7.5/6.1); group 32, whose units cost it twice
  // the matrix work, at up to eight (4.1/4.2 at 1000 x 2048) and five rows.
  // Larger K, and K with a tail chunk for the GEMV, meet earlier: at four rows of
  // 4-bit codes 9.6/6.8 for 5120 x 2560 and 11.8/7.5 for 4096 x 6144, 6.8/6.8 and
  // 8.2/7.5 at two; the line, drawn by the rows alone, leaves those to the GEMV.
  // Below a few MB of weight reads both are launch-bound and the GEMV's chain
  // is the shorter one.
  const int64_t min_rows = bits == 4 ? (group_size == 32 ? 8 : 5) : (group_size == 32 ? 5 : 3);
  return M >= min_rows && M * (N * K * bits / 8) >= (4 << 20);
}

int launch(const uint16_t* x, int64_t M, int64_t K, const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
           int64_t N, int group_size, int bits, uint16_t* out, hipStream_t st) {
  const QmmArgs a{x, M, (int)K, w, scales, biases, (int)N, out};
  return bits == 4 ? launch_gs<4>(a, group_size, st) : launch_gs<8>(a, group_size, st);
}

}  // namespace qmoe_qmm
