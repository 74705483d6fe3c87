// W8A8 GS128 GEMM for few rows: Y (M, N) = A (M, K) . W (N, K)^T under the contract of gemm.hip,
// bit for bit (acc = fmaf(float(P_g), sa * sw, acc), groups in order, the same K parts added in
// order, the same epilogue).
//
// What bounds it: latency. gemm.hip's kernel walks all groups of a 128 x 128 tile one after the
// other, so a decode call on 1536 x 1536 weights is 12 workgroups of 12 dependent steps, whatever
// M is. Only the fold over groups has to be in order, the exact int32 products need not be: here
// a workgroup owns 16 output columns and MT * 16 rows (MT = 1, 2, 4) and each of its up to 16
// waves takes one group, loads its slices of A and W straight into MFMA registers (they are used
// once, so LDS staging would only add a trip) and leaves its products in LDS, where 256 threads
// per row tile fold up to 16 groups in order. The next round's slices load during the fold.
// Measured (device time in a graph, 16-bit output, gemm.hip's kernel -> this one): 1 x 1536 -> 1536
// 11.8 -> 4.4 us, 64 x 1536 -> 1536 11.8 -> 8.2, 16 x 1536 -> 4096 11.9 -> 5.1, 16 x 5888 -> 1536
// (5 K parts and their combine launch) 15.0 -> 12.1, 512 x 1536 -> 512 11.9 -> 8.3.
#include "ksd_common.h"

namespace ksd {
namespace rows {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kMaxWaves = 16;

struct Prob {
  const int8_t *A, *W;
  const uint16_t *As, *Ws;
  const float *bias;
  const void *R;
  void *Y;
  int M, N, G, splits, out;
};

// A wave's 16 rows x 128 columns of one operand: lane l holds the 16-byte chunks q and 4 + q
// (q = l / 16) of row l % 16, so four lanes read 64 contiguous bytes. Both operands use this
// mapping; which k a slot of the MFMA holds does not matter then.
struct Tile {
  v4i c[2];
  uint16_t s;
  __device__ __forceinline__ void load(const int8_t *codes, const uint16_t *scales, int row, int G, int g, int lane) {
    const int64_t at = (int64_t)row * G + g;
    const int8_t *r = codes + at * 128 + 16 * (lane >> 4);
    c[0] = *(const v4i *)r;
    c[1] = *(const v4i *)(r + 64);
    s = scales[at];
  }
};

__device__ __forceinline__ void finish(const Prob &p, float y, int row, int col) {
  const int64_t i = (int64_t)row * p.N + col;
  if (p.bias) y = y + p.bias[col];
  switch (p.out) {
    case KSD_F32:
      if (p.R) y = y + ((const float *)p.R)[i];
      ((float *)p.Y)[i] = y;
      break;
    case KSD_BF16:
      if (p.R) y = bf16_to_f32(f32_to_bf16(y)) + bf16_to_f32(((const uint16_t *)p.R)[i]);
      ((uint16_t *)p.Y)[i] = f32_to_bf16(y);
      break;
    case KSD_F16:
      if (p.R) y = f16_round(y) + f16_to_f32(((const uint16_t *)p.R)[i]);
      ((uint16_t *)p.Y)[i] = f16_bits(y);
      break;
    default: {  // KSD_F16_SAT: fp16, then clamp to +-65504
      _Float16 h = (_Float16)opaque(y);
      const float hf = (float)h;
      if (hf > kScaleMax) h = (_Float16)kScaleMax;
      if (hf < -kScaleMax) h = (_Float16)(-kScaleMax);
      ((uint16_t *)p.Y)[i] = __builtin_bit_cast(uint16_t, h);
    }
  }
}

// blockDim.x = 64 * waves(G), a multiple of 256. Rows past M and columns past N load the last
// valid row and are not stored.
template <int MT>
__device__ __forceinline__ void rows_gemm_block(const Prob &p) {
  __shared__ float part[kMaxWaves][MT][256];  // float(P_g) of the round's groups
  __shared__ float sa[kMaxWaves][MT * 16], sw[kMaxWaves][16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = blockDim.x >> 6;
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * (MT * 16);
  const int wrow = min(n0 + (lane & 15), p.N - 1);
  Tile w, a[MT];
  auto load = [&](int g) {
    w.load(p.W, p.Ws, wrow, p.G, g, lane);
#pragma unroll
    for (int t = 0; t < MT; ++t) a[t].load(p.A, p.As, min(m0 + t * 16 + (lane & 15), p.M - 1), p.G, g, lane);
  };
  if (wave < p.G) load(wave);
  float acc[MT], y[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = y[i] = 0.0f;
  auto part_end = [&](int q) { return (int)((int64_t)(q + 1) * p.G / p.splits); };
  int q0 = 0;  // the K part that the round starts in

  for (int g0 = 0; g0 < p.G; g0 += nw) {
    const int g = g0 + wave, ng = min(nw, p.G - g0);
    if (g < p.G) {  // wave-uniform
      if (lane < 16) sw[wave][lane] = f16_to_f32(w.s);
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        v4i c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[t].c[0], w.c[0], (v4i){0, 0, 0, 0}, 0, 0, 0);
        c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[t].c[1], w.c[1], c, 0, 0, 0);
        if (lane < 16) sa[wave][t * 16 + lane] = f16_to_f32(a[t].s);
#pragma unroll
        for (int r = 0; r < 4; ++r) part[wave][t][(4 * (lane >> 4) + r) * 16 + (lane & 15)] = (float)c[r];
      }
      if (g + nw < p.G) load(g + nw);
    }
    __syncthreads();
    const int e = tid & 255;
    int q1 = q0;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int t = (tid >> 8) + i * (nw >> 2);
      if (t >= MT) break;
      q1 = q0;
      int end = part_end(q1);
      for (int k = 0; k < ng; ++k) {
        if (g0 + k == end) {  // the next K part starts: add the finished one
          y[i] = q1 == 0 ? acc[i] : y[i] + acc[i];
          acc[i] = 0.0f;
          end = part_end(++q1);
        }
        acc[i] = fmaf(part[k][t][e], sa[k][t * 16 + (e >> 4)] * sw[k][e & 15], acc[i]);
      }
    }
    while (q0 + 1 < p.splits && part_end(q0) < g0 + ng) ++q0;
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int t = (tid >> 8) + i * (nw >> 2);
    if (t >= MT) break;
    const int row = m0 + t * 16 + ((tid & 255) >> 4), col = n0 + (tid & 15);
    if (row < p.M && col < p.N) finish(p, p.splits > 1 ? y[i] + acc[i] : acc[i], row, col);
  }
}

template <int MT>
__global__ __launch_bounds__(64 * kMaxWaves) void rows_gemm_kernel(const Prob p) {
  rows_gemm_block<MT>(p);
}

// Three problems of one shape (a mixer's q, k and v) in one launch, blockIdx.z the problem: each
// alone leaves CUs idle. 301 x 1536 -> 512: three launches 26.3 us of device time, this one 15.6.
struct Prob3 {
  Prob p[3];
};
template <int MT>
__global__ __launch_bounds__(64 * kMaxWaves) void rows_gemm3_kernel(const Prob3 a) {
  rows_gemm_block<MT>(a.p[blockIdx.z]);
}

// The fewest rounds over the groups, then the fewest waves for them; whole 256-thread folds.
static int waves(int G) {
  const int rounds = (G + kMaxWaves - 1) / kMaxWaves, per = (G + rounds - 1) / rounds;
  return (per + 3) / 4 * 4;
}

static int tiles(int M) { return M <= 16 ? 1 : M <= 32 ? 2 : 4; }
}  // namespace rows

// Its time grows with the row tiles that a CU works through, f = MT * ceil(workgroups / CUs), and the G
// groups: about 3 us and, for each group, 0.2 at f = 1, 0.3 at f = 2, 0.4 to 0.6 at f = 4. gemm.hip's kernel
// takes 5.2 and 0.55 G / splits, and 3 more for the combine launch of a split K. So up to f = 4, and f G = 64
// where K is long enough to be split. At f G = 64 K is 2048, 4096 or 8192, whose rows all start in the same
// cache channels: a full row tile's 16 of them lose there (M above 10), fewer rows and several tiles do not.
// Both sides (us, gemm.hip's kernel and this one, M x N x K): 32 x 8192 x 1536 12.1, 8.2; 16 x 16384 x 1920
// 14.9, 12.9; 16 x 16384 x 2048 14.1, 16.3; 16 x 6144 x 4096 14.3, 15.8; 16 x 4096 x 8192 18.0, 18.4; 8 x 8192
// x 4096 14.9, 14.0; 64 x 4096 x 2048 13.4, 11.2; 64 x 5888 x 1536 (f = 8) 11.2, 13.4.
// CUs are counted as 256 whatever the device has.
bool rows_gemm_fits(int64_t M, int64_t N, int64_t K) {
  if (M > 4096) return false;
  const int mt = rows::tiles((int)M);
  const int64_t groups = K / 128, f = mt * cdiv(cdiv(N, 16) * cdiv(M, 16 * mt), 256);
  return f <= 4 && f * groups <= (mt == 1 && M > 10 ? 63 : 64);
}

void rows_gemm(const int8_t *a, const uint16_t *as, const int8_t *w, const uint16_t *ws, int M, int N, int K,
               int splits, const float *bias, const void *residual, void *y, int out, hipStream_t st) {
  const rows::Prob p{a, w, as, ws, bias, residual, y, M, N, K / 128, splits, out};
  const int mt = rows::tiles(M);
  const dim3 grid((unsigned)cdiv(N, 16), (unsigned)cdiv(M, 16 * mt)), block(64 * rows::waves(p.G));
  if (mt == 1) rows::rows_gemm_kernel<1><<<grid, block, 0, st>>>(p);
  else if (mt == 2) rows::rows_gemm_kernel<2><<<grid, block, 0, st>>>(p);
  else rows::rows_gemm_kernel<4><<<grid, block, 0, st>>>(p);
}

void rows_gemm3(const int8_t *const a[3], const uint16_t *const as[3], const int8_t *const w[3],
                const uint16_t *const ws[3], int M, int N, int K, int splits, const float *const bias[3],
                void *const y[3], int out, hipStream_t st) {
  rows::Prob3 p;
  for (int i = 0; i < 3; ++i)
    p.p[i] = rows::Prob{a[i], w[i], as[i], ws[i], bias[i], nullptr, y[i], M, N, K / 128, splits, out};
  const int mt = rows::tiles(M);
  const dim3 grid((unsigned)cdiv(N, 16), (unsigned)cdiv(M, 16 * mt), 3), block(64 * rows::waves(K / 128));
  if (mt == 1) rows::rows_gemm3_kernel<1><<<grid, block, 0, st>>>(p);
  else if (mt == 2) rows::rows_gemm3_kernel<2><<<grid, block, 0, st>>>(p);
  else rows::rows_gemm3_kernel<4><<<grid, block, 0, st>>>(p);
}
}  // namespace ksd
