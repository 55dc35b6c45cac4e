// Un-permute + router-weighted top-k sum (titan/kernels/moe_weighted_sum.py:44-98).
//
// Each thread owns 8 adjacent columns of one output row and walks the k
// expert outputs in order, keeping eight partial sums per column (slot j mod 8)
// that are combined in slot order at the end.  Rows are fetched eight slots
// at a time, so a thread has eight 16-byte loads in flight.  Rows are read
// and the output written with non-temporal hints: each byte is touched once
// (measured 36.8 -> 32.4 us at 4096 tokens x top-10 x 2048 columns, 185 MB,
// most of it from the store).  The arithmetic is spelled out
// with contraction switched off so no multiply-add is fused: every mode is a
// fixed sequence of IEEE operations and bf16 roundings, bit-for-bit
// reproducible against a CPU restatement of the same sequence.
#include "common.h"

namespace {

// SH: one more row per output row, shared[r], with the score in the last of
// the row's k + 1 scores; added in fp32 after the k slots (after their sum's
// bf16 rounding in the ops and clone modes, whose k-slot result is defined as
// rounded).
template <int MODE, bool SH>  // QMOE_WSUM_FAST, _OPS, _CLONE
__global__ __launch_bounds__(256) void wsum_kernel(const uint16_t* __restrict__ xs,
                                                   const int32_t* __restrict__ inv,
                                                   const float* __restrict__ scores, int64_t rows, int k,
                                                   int64_t dim, const uint16_t* __restrict__ shared,
                                                   uint16_t* __restrict__ out) {
#pragma clang fp contract(off)
  constexpr bool kRoundProd = MODE >= QMOE_WSUM_OPS;
  constexpr bool kBfAcc = MODE == QMOE_WSUM_CLONE;
  const int64_t c8 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8;
  const int64_t r = blockIdx.y;
  if (c8 >= dim || r >= rows) return;
  i32x4_t shq = {0, 0, 0, 0};
  float shs = 0.f;
  if constexpr (SH) {
    shq = __builtin_nontemporal_load(reinterpret_cast<const i32x4_t*>(shared + r * dim + c8));
    shs = scores[r * (k + 1) + k];
  }
  const int64_t ss = SH ? k + 1 : k;  // scores per row
  float acc[8][8];
#pragma unroll
  for (int a = 0; a < 8; ++a)
#pragma unroll
    for (int v = 0; v < 8; ++v) acc[a][v] = 0.f;
  // slots in batches of eight: the batch's indices, scores and rows are all
  // requested before any is used (eight loads in flight per thread), and
  // slot j mod 8 is the batch position, a compile-time index
  for (int j0 = 0; j0 < k; j0 += 8) {
    uint4 q[8];
    float sc[8];
#pragma unroll
    for (int jj = 0; jj < 8; ++jj) {
      if (j0 + jj < k) {
        const int64_t p = r * k + j0 + jj;
        const int64_t src = inv ? (int64_t)inv[p] : p;
        sc[jj] = scores[r * ss + j0 + jj];
        const i32x4_t t = __builtin_nontemporal_load(reinterpret_cast<const i32x4_t*>(xs + src * dim + c8));
        q[jj] = make_uint4((uint32_t)t[0], (uint32_t)t[1], (uint32_t)t[2], (uint32_t)t[3]);
      }
    }
#pragma unroll
    for (int jj = 0; jj < 8; ++jj) {
      if (j0 + jj >= k) break;
      float s = sc[jj];
      if (MODE >= QMOE_WSUM_OPS) s = round_bf16(s);
      const uint32_t pr[4] = {q[jj].x, q[jj].y, q[jj].z, q[jj].w};
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        const float xv = (v & 1) ? bf16hi(pr[v >> 1]) : bf16lo(pr[v >> 1]);
        float prod = s * xv;
        if (kRoundProd) prod = round_bf16(prod);
        const float t = acc[jj][v] + prod;
        acc[jj][v] = kBfAcc ? round_bf16(t) : t;
      }
    }
  }
  uint32_t o[4];
#pragma unroll
  for (int v = 0; v < 8; v += 2) {
    float r0 = acc[0][v], r1 = acc[0][v + 1];
#pragma unroll
    for (int a = 1; a < 8; ++a) {
      r0 = r0 + acc[a][v];
      r1 = r1 + acc[a][v + 1];
      if (kBfAcc) {
        r0 = round_bf16(r0);
        r1 = round_bf16(r1);
      }
    }
    if constexpr (SH) {
      if (MODE >= QMOE_WSUM_OPS) {
        r0 = round_bf16(r0);
        r1 = round_bf16(r1);
      }
      const uint32_t pr = (uint32_t)shq[v >> 1];
      r0 = r0 + shs * bf16lo(pr);
      r1 = r1 + shs * bf16hi(pr);
    }
    o[v >> 1] = pack_bf16x2(r0, r1);
  }
  const i32x4_t ov = {(int)o[0], (int)o[1], (int)o[2], (int)o[3]};
  __builtin_nontemporal_store(ov, reinterpret_cast<i32x4_t*>(out + r * dim + c8));
}

template <bool SH>
int weighted_sum(const uint16_t* xs, const int32_t* inv_order, const float* scores, int64_t rows, int64_t top_k,
                 int64_t dim, int mode, const uint16_t* shared, uint16_t* out, void* stream) {
  if (rows < 0 || top_k <= 0 || dim <= 0) return qmoe::fail(QMOE_ERR_INVALID, "bad sizes");
  if (rows == 0) return QMOE_OK;
  if (!xs || !scores || !out) return qmoe::fail(QMOE_ERR_INVALID, "null pointer");
  if (mode < QMOE_WSUM_FAST || mode > QMOE_WSUM_CLONE) return qmoe::fail(QMOE_ERR_UNSUPPORTED, "mode=%d", mode);
  if (dim % 8) return qmoe::fail(QMOE_ERR_UNSUPPORTED, "dim=%lld: must be a multiple of 8", (long long)dim);
  if (!qmoe::aligned16(xs) || !qmoe::aligned16(out))
    return qmoe::fail(QMOE_ERR_UNSUPPORTED, "xs and out must be 16-byte aligned");
  if (rows > 65535) return qmoe::fail(QMOE_ERR_UNSUPPORTED, "rows=%lld > 65535", (long long)rows);
  if (SH && !shared) return qmoe::fail(QMOE_ERR_INVALID, "null pointer");
  if (SH && !qmoe::aligned16(shared)) return qmoe::fail(QMOE_ERR_UNSUPPORTED, "shared must be 16-byte aligned");
  if (top_k > (SH ? 0x7FFFFFFE : 0x7FFFFFFF)) return qmoe::fail(QMOE_ERR_INVALID, "top_k too large");
  const int64_t threads = dim / 8;
  dim3 block((unsigned)(threads < 256 ? threads : 256));
  dim3 grid((unsigned)((threads + block.x - 1) / block.x), (unsigned)rows);
  hipStream_t st = qmoe::as_stream(stream);
  switch (mode) {
    case QMOE_WSUM_FAST:
      wsum_kernel<QMOE_WSUM_FAST, SH><<<grid, block, 0, st>>>(xs, inv_order, scores, rows, (int)top_k, dim, shared,
                                                             out);
      break;
    case QMOE_WSUM_OPS:
      wsum_kernel<QMOE_WSUM_OPS, SH><<<grid, block, 0, st>>>(xs, inv_order, scores, rows, (int)top_k, dim, shared,
                                                             out);
      break;
    default:
      wsum_kernel<QMOE_WSUM_CLONE, SH><<<grid, block, 0, st>>>(xs, inv_order, scores, rows, (int)top_k, dim, shared,
                                                             out);
      break;
  }
  return qmoe::launch_status("wsum_kernel");
}

}  // namespace

extern "C" int qmoe_weighted_sum(const uint16_t* xs, const int32_t* inv_order, const float* scores,
                                 int64_t rows, int64_t top_k, int64_t dim, int mode, uint16_t* out,
                                 void* stream) {
  return weighted_sum<false>(xs, inv_order, scores, rows, top_k, dim, mode, nullptr, out, stream);
}

extern "C" int qmoe_weighted_sum_shared(const uint16_t* xs, const int32_t* inv_order, const float* scores,
                                        int64_t rows, int64_t top_k, int64_t dim, int mode, const uint16_t* shared,
                                        uint16_t* out, void* stream) {
  return weighted_sum<true>(xs, inv_order, scores, rows, top_k, dim, mode, shared, out, stream);
}
