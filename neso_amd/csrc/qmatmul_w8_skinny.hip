// W8A16 for few rows of A (M <= 64): column strips of B streamed once from
// HBM, K split over waves and workgroups.
//
// Bound: HBM, K * N bytes of int8 weights (B is [K][N], N-contiguous).  One
// CU draws at most ~35 GB/s from HBM, so the whole chip is needed even for
// one projection, while a strip of whole 128-byte lines per workgroup gives
// only N / 128 workgroups.  K is therefore split over workgroups as well
// (launch_w8a16_skinny); each writes its partial tile to a workspace of the
// caller, and w8a16_reduce_kernel adds the partials in a fixed order.
//
// A wave walks 32 k-rows of a 128-column strip per step.  Lane (j = l % 16,
// g = l / 16) loads 8 bytes, columns 8 j .. 8 j + 7, of the rows 8 g .. 8 g +
// 7: four whole lines per instruction.  Byte c of those eight rows is then
// the B operand of a v_mfma_f32_16x16x32_f16 over the columns 8 j + c, so the
// transposition costs one v_perm per pair of rows (which the int8 -> f16
// conversion needs anyway) and B never passes through LDS.  The A operand is
// 16 contiguous bytes of X per lane, read straight from global memory (L2
// holds it): 1/4 of the weight bytes at M <= 16.
//
// int8 -> f16 is exact: 0x6400 | (b ^ 0x80) is f16 1024 + 128 + b.
//
// Measured per call, both launches (rotated weights, graph of launches),
// against the 128 x 128-tile kernel that served these calls, M = 1 / 16 / 64:
// K 4096, N 4096 44.4 / 44.5 / 45.0 -> 8.4 / 9.3 / 17.5 us (M = 1 2.0 TB/s);
// K 4096, N 11008 48.6 / 48.7 / 49.2 -> 13.6 / 15.4 / 27.6 (3.3 TB/s);
// K 11008, N 4096 122.6 / 122.2 / 122.8 -> 12.5 / 14.6 / 25.2 (3.6 TB/s).  A
// kernel that only reads such strips takes 4.9, 9.1 and 9.2 us; the
// reduction's launch is about 2.5 us of the rest.  Four or eight waves per
// workgroup, the order of strips and splits over the XCDs, and more than two
// steps in flight measured the same within 4%.
#include "common.h"
#include "neso_internal.h"

namespace neso {

namespace {

constexpr int kStrip = 128;  // columns per workgroup
constexpr int kStepK = 32;   // k-rows per wave and step
constexpr int kWaves = 4;
constexpr int kRedRow = kStrip + 4;

typedef uint32_t uint2v __attribute__((ext_vector_type(2)));

// MT: 16-row tiles of A.  part != nullptr: partial sums of this workgroup's
// K range to part[split][m][n]; else the scaled result to C.
template <int MT>
__global__ __launch_bounds__(kWaves * kWave) void w8a16_skinny_kernel(W8Args a, float* part,
                                                                      int32_t splits) {
  constexpr uint32_t kOut = 0x80000000u;  // offset past every buffer
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, g = lane >> 4;
  const int nstrips = (a.N + kStrip - 1) / kStrip;
  const int strip = blockIdx.x % nstrips, split = blockIdx.x / nstrips;
  const int n0 = strip * kStrip;
  const int steps = (a.K + kStepK - 1) / kStepK;
  const int per = (steps + splits - 1) / splits;
  const int t0 = split * per, t1 = min(t0 + per, steps);

  __shared__ __attribute__((aligned(16))) float red[kWaves][16 * kRedRow];

  // Lane offsets within a step; columns past N and rows of A past M are
  // masked here, k past K by the steps' buffer extents (B) and per step (A).
  uint32_t bo[8], xo[MT];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    bo[i] = ((uint32_t)(8 * g + i) * (uint32_t)a.ldb + 8u * j) | (n0 + 8 * j < a.N ? 0u : kOut);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    xo[mt] = ((uint32_t)(16 * mt + j) * (uint32_t)a.lda + 8u * g) * 2u | (16 * mt + j < a.M ? 0u : kOut);

  struct Step {
    uint2v b[8];
    half8v x[MT];
  };
  auto load = [&](Step& s, int t) {
    // Steps past the range get empty buffers: their loads return zeros.
    const int k0 = t * kStepK;
    const int rows = t < t1 ? min(kStepK, a.K - k0) : 0;
    const int at = rows ? k0 : 0;
    const rsrc_t rb = make_rsrc(a.B + (int64_t)at * a.ldb + n0,
                                rows ? (uint32_t)((rows - 1) * (int64_t)a.ldb + min(kStrip, a.N - n0)) : 0u);
    const rsrc_t rx = make_rsrc(a.A + at, rows ? (uint32_t)(((int64_t)(a.M - 1) * a.lda + rows) * 2) : 0u);
    const uint32_t xoob = 8 * g < rows ? 0u : kOut;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) s.x[mt] = buf_load_half8(rx, xo[mt] | xoob);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      s.b[i] = __builtin_bit_cast(uint2v, __builtin_amdgcn_raw_buffer_load_b64(rb, bo[i], 0, kNonTemporal));
  };

  float4v acc[MT][8];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int c = 0; c < 8; ++c) acc[mt][c] = float4v{};
  const half2v bias = {(half_t)1152, (half_t)1152};
  auto compute = [&](const Step& s) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      half8v w;
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        // Byte c of rows 2 p and 2 p + 1 as two f16.
        const uint32_t sel = 0x0c000c00u | (uint32_t)((4 + c % 4) << 16) | (uint32_t)(c % 4);
        const uint32_t pr =
            __builtin_amdgcn_perm(s.b[2 * p + 1][c / 4], s.b[2 * p][c / 4], sel) ^ 0x64806480u;
        const half2v v = __builtin_bit_cast(half2v, pr) - bias;
        w[2 * p] = v[0];
        w[2 * p + 1] = v[1];
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt][c] = mfma16x16x32(s.x[mt], w, acc[mt][c]);
    }
  };

  // Wave w takes steps t0 + w, t0 + w + 8, ..., two in flight.
  Step sA, sB;
  load(sA, t0 + wave);
  for (int t = t0 + wave; t < t1; t += 2 * kWaves) {
    load(sB, t + kWaves);
    compute(sA);
    load(sA, t + 2 * kWaves);
    compute(sB);
  }

  // Sum of the waves' tiles, 16 rows at a time.  acc[mt][c] register r of
  // lane (j, g) is row 16 mt + 4 g + r, column n0 + 8 j + c.
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    if (mt) lds_barrier();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float* row = &red[wave][(4 * g + r) * kRedRow + 8 * j];
      *reinterpret_cast<float4v*>(row) = float4v{acc[mt][0][r], acc[mt][1][r], acc[mt][2][r], acc[mt][3][r]};
      *reinterpret_cast<float4v*>(row + 4) =
          float4v{acc[mt][4][r], acc[mt][5][r], acc[mt][6][r], acc[mt][7][r]};
    }
    lds_barrier();
#pragma unroll
    for (int h = 0; h < 8 / kWaves; ++h) {
      const int row = (int)(threadIdx.x >> 5) + 2 * kWaves * h, col = 4 * (threadIdx.x & 31);
      float4v v = float4v{};
#pragma unroll
      for (int w = 0; w < kWaves; ++w) v += *reinterpret_cast<const float4v*>(&red[w][row * kRedRow + col]);
      const int m = 16 * mt + row, n = n0 + col;
      if (m >= a.M || n >= a.N) continue;  // N is a multiple of 8
      if (part) {
        *reinterpret_cast<float4v*>(part + ((int64_t)split * a.M + m) * a.N + n) = v;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          a.C[(int64_t)m * a.ldc + n + i] = v[i] * (a.scale ? (float)a.scale[n + i] : 1.f);
      }
    }
  }
}

// C[m][n] = scale[n] * sum over splits of part[s][m][n], in split order.
// Rows of part are w8a16_part_stride(N) floats.
__global__ __launch_bounds__(kWave) void w8a16_reduce_kernel(W8Args a, const float* part, int32_t splits,
                                                             int32_t np) {
  const int quads = np / 4;
  const int64_t e = (int64_t)blockIdx.x * kWave + threadIdx.x;
  const int m = (int)(e / quads), n = 4 * (int)(e % quads);
  if (m >= a.M) return;
  const int64_t mn = (int64_t)a.M * np;
  const float* p = part + (int64_t)m * np + n;
  // Eight loads at a time, the last batch clamped to the last partial.
  float4v v = float4v{};
  for (int s0 = 0; s0 < splits; s0 += 8) {
    float4v x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = *reinterpret_cast<const float4v*>(p + min(s0 + i, splits - 1) * mn);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (s0 + i < splits) v += x[i];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (n + i < a.N) a.C[(int64_t)m * a.ldc + n + i] = v[i] * (a.scale ? (float)a.scale[n + i] : 1.f);
}

int mtiles(int m) { return m <= 16 ? 1 : m <= 32 ? 2 : 4; }

}  // namespace

int w8a16_skinny_max_m() { return 64; }

// As many splits as give every CU a workgroup, at most 8 and at most one per
// two steps of each wave.  One CU draws ~35 GB/s, so the strips alone leave
// most of the chip's bandwidth unused, and past eight partials the reduction
// and the half-empty steps cost more than they bring.  M = 16, us for
// splits 1 / 2 / 4 / 8 / 16:
//   K 4096, N 4096:  22.3 / 15.3 / 11.2 /  9.4 / 11.4  (8 chosen)
//   K 4096, N 11008: 20.4 / 15.6 / 16.4 / 16.4 / 20.7  (2)
//   K 11008, N 4096: 56.0 / 32.2 / 20.2 / 14.8 / 16.4  (8)
//   K 1024, N 1024:   7.1 /  6.9 /  6.4 /  6.4 /   -   (4)
//   K 256, N 1024:    4.6 /  5.9                       (1)
int w8a16_skinny_splits(const W8Args& a) {
  const int strips = (a.N + kStrip - 1) / kStrip;
  const int splits = min(min(device_cu_count() / strips, a.K / (2 * kStepK * kWaves)), 8);
  return splits < 2 ? 1 : splits;
}

hipError_t launch_w8a16_skinny(const W8Args& a, int splits, float* workspace, hipStream_t s) {
  const int strips = (a.N + kStrip - 1) / kStrip;
  const dim3 grid(strips * splits), block(kWaves * kWave);
  const int mt = mtiles(a.M);
  float* part = splits > 1 ? workspace : nullptr;
  const KernelTag tag = ktag("w8a16_skinny_kernel", mt);
  hipError_t e = mt == 1   ? launch<&w8a16_skinny_kernel<1>>(tag, grid, block, s, a, part, splits)
                 : mt == 2 ? launch<&w8a16_skinny_kernel<2>>(tag, grid, block, s, a, part, splits)
                           : launch<&w8a16_skinny_kernel<4>>(tag, grid, block, s, a, part, splits);
  return e != hipSuccess || splits == 1 ? e : launch_w8a16_reduce(a, splits, workspace, s);
}

hipError_t launch_w8a16_reduce(const W8Args& a, int splits, const float* part, hipStream_t s) {
  const int np = w8a16_part_stride(a.N);
  const int64_t quads = (int64_t)a.M * (np / 4);
  return launch<&w8a16_reduce_kernel>(ktag("w8a16_reduce_kernel"), dim3((quads + kWave - 1) / kWave), dim3(kWave), s,
                                      a, part, splits, np);
}

}  // namespace neso
