// int4 W4A16 skinny-M kernel with X resident in LDS (M <= 32, K % 128 == 0,
// power-of-two scale groups): its own translation unit so that it can be
// compiled with its own scheduler options (see build.py).
#include "common.h"
#include "neso_internal.h"
#include "qmatmul_common.h"

namespace neso {

namespace {

// Skinny-M regime with X resident in LDS.
//
// The workload is one burst of N*K/2 bytes.  One persistent workgroup per
// CU owns row tiles blockIdx.x + i * gridDim.x (16 rows each, i < T).  Its
// WV waves split K (wave w takes chunk quads [w*QW, (w+1)*QW)) and request
// the weights and scales of tile i + 1 before computing tile i, tile 0
// right after X (plain loads: the non-temporal hint measured slower for
// these 64-byte row pieces).  X is copied
// once per workgroup into LDS, already in MFMA A-fragment order (slot
// (4q + t) * 64 + lane holds X[m][32(4q+t) + 8g + {0,4,1,5,2,6,3,7}] for
// lane = m + 16g), so the per-tile A operand is one conflict-free
// ds_read_b128 per MFMA.  MFMA, transpose and dequantisation are those of
// w4a16_skinny_kernel.  The WV partial tiles are reduced through LDS.
// (The slot's row index is XOR-swizzled; see the X loads below.)
//
// LDS holds 4096 codes of 16 rows or 2048 of 32 (MT = 2: each dequantised
// fragment feeds two MFMAs).  Longer K runs in equal phases (MP), the next
// phase's X on its way in registers while this one computes.  The phase loop
// is rolled and keeps one W item ahead: each wave runs this code once or a
// few times per launch, so its size counts (K = 11008 N = 4096 M = 16, four
// phases unrolled with three items ahead 18.4 us, two with one 14.7, rolled
// with per-row buffer bases instead of per-piece offsets 13.5).
// GS scales per quad of 128 codes: 4, 2, or 1 (groups of 128 and up).
//
// Bound: HBM at K <= 4096 (9.1 us for N = 11008, 2.5 TB/s with a ~2 us
// launch); a phase's X store and barriers (~1 us) beyond.
constexpr int kLdsQuads = 32;  // K <= 4096 / MT per phase

template <int WV, int T, int QWMAX, int GS, bool MP>
__global__ __launch_bounds__(WV * kWave) void w4a16_skinny_lds_kernel(W4Args a) {
  static_assert(WV * QWMAX * 4 == kLdsQuads * QWMAX && kLdsQuads / WV == 4, "waves share out a phase");
  static_assert(QWMAX == 4 || QWMAX == 2, "quads per wave and phase");
  constexpr uint32_t kOut = 0x80000000u;
  constexpr int MT = 4 / QWMAX;            // 16-row tiles of X
  constexpr int QPM = kLdsQuads / MT;      // quads per phase, at most
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const int gshift = __builtin_ctz(a.group >> 7);  // GS = 1: 2^gshift quads per scale
  // Scales per row by shifts: a division here delays the first loads (1-2%
  // of a launch).
  const int KW = a.K >> 3, SG = GS == 4 ? a.K >> 5 : GS == 2 ? a.K >> 6 : a.K >> (7 + gshift);
  const int Q = a.K >> 7;                  // K % 128 == 0
  const int P = MP ? (Q + QPM - 1) / QPM : 1;
  const int QP = (Q + P - 1) / P, QW = (QP + WV - 1) / WV;
  const int ntiles = (a.N + 15) >> 4;
  const ZeroPoint zp = zero_point(a.zero);
  const Nibbles nib = nibble_consts();

  // The partial tiles have LDS of their own beside X at MT = 1 and take X's
  // place, after a barrier, at MT = 2.
  constexpr int kRed = T * WV * 4 * MT * kWave;
  __shared__ half8v xs[kLdsQuads * 4 * kWave];
  __shared__ float red_own[MT == 1 ? kRed : 1];
  static_assert(kRed * sizeof(float) <= sizeof(xs) && sizeof(xs) + sizeof(red_own) <= 160 * 1024, "LDS");
  float* const red = MT == 1 ? red_own : reinterpret_cast<float*>(xs);
  auto red_at = [&](int i, int wv, int r, int ln) { return ((i * WV + wv) * (4 * MT) + r) * kWave + ln; };

  // X first: loads complete in issue order, so X (L2-resident) reaches LDS
  // while the weight burst is still arriving; issued after the weights, it
  // waited behind them (measured: 15.7 -> 14.2 us at M = 16).  Each wave
  // instruction reads 1 KiB of one X row (piece e: row m, pieces pp of 8
  // halves; 16 rows x 64 B per instruction measured 14.2 vs 12.9 us).  Piece
  // (m, chunk ct, quarter g) goes to A-fragment slot ct*64 + 16g + m' of its
  // 16-row tile, with the row index swizzled, m' = m ^ (4 (ct % 4) + g), so
  // that the 64 same-row stores of an instruction and the 16-lane fragment
  // reads both spread over all banks.
  constexpr int kXPer = (kLdsQuads * 4 * kWave) / (WV * kWave);
  constexpr int kRowPieces = 16 * QPM;
  // Thread t takes piece t % kRowPieces of rows t / kRowPieces + MT i.
  static_assert(WV * kWave == MT * kRowPieces, "MT rows per pass");
  const int xr = threadIdx.x / kRowPieces, pp = threadIdx.x % kRowPieces, ct = pp >> 2;
  const int xsw = 4 * (ct & 3) + (pp & 3);
  half8v* const xdst = &xs[ct * 64 + 16 * (pp & 3)];
  half8v xv[kXPer];
  uint32_t xslot[MP ? 1 : kXPer];
  auto xload = [&](int p) {
    if constexpr (!MP) {
      // One phase: per-piece offsets and slots into one buffer, which issue
      // sooner than a buffer base per row (1-3% of a launch).
      const rsrc_t rx = make_rsrc(a.X, (uint32_t)(((int64_t)(a.M - 1) * a.ldx + a.K) * 2));
#pragma unroll
      for (int i = 0; i < kXPer; ++i) {
        const uint32_t e = threadIdx.x + i * WV * kWave;
        const uint32_t m = e / kRowPieces, pc = e % kRowPieces, c = pc >> 2, g = pc & 3;
        const uint32_t oob = ((int)c < 4 * Q && (int)m < a.M) ? 0u : kOut;
        xv[i] = buf_load_half8(rx, ((m * (uint32_t)a.ldx + 8u * pc) * 2u) | oob);
        xslot[i] = c * 64 + 16 * g + (m ^ (4 * (c & 3) + g));
      }
      return;
    }
    const int cend = 4 * (min((p + 1) * QP, Q) - p * QP);  // chunks of the phase
    const uint32_t off = ((uint32_t)xr * (uint32_t)a.ldx + 8u * pp) * 2u | (ct < cend ? 0u : kOut);
#pragma unroll
    for (int i = 0; i < kXPer; ++i) {
      const int rows = a.M - MT * i;  // left from row MT i on
      const rsrc_t rx = make_rsrc(a.X + (int64_t)(rows > 0 ? MT * i : 0) * a.ldx + 128 * p * QP,
                                  rows > 0 ? (uint32_t)(((int64_t)(rows - 1) * a.ldx + a.K - 128 * p * QP) * 2) : 0u);
      xv[i] = buf_load_half8(rx, off);
    }
  };
  auto xstore = [&]() {
#pragma unroll
    for (int i = 0; i < kXPer; ++i) {
      const int m = xr + MT * i;
      const half8v x = xv[i];
      half8v* const dst = MP ? xdst + (m >> 4) * (4 * QPM * 64) + ((m & 15) ^ xsw) : xs + xslot[MP ? 0 : i];
      *dst = half8v{x[0], x[4], x[1], x[5], x[2], x[6], x[3], x[7]};
    }
  };

  // Weight and scale loads of this wave for tile i in phase p.
  // Scales: one load per lane and item, lane (li, lg) taking quad q0 + lg of
  // row li (8, 4 or 2 bytes; no four lanes loading the same bytes); quad qi
  // reaches lane (li, *) from lane (li, qi) by ds_bpermute (measured 12.9 ->
  // 11.7 us at M = 16).
  typedef uint32_t uint2v __attribute__((ext_vector_type(2)));
  struct Item {
    uint4v w[QWMAX];
    uint2v s;
  };
  auto load_item = [&](Item& it, int p, int i) {
    const int tile = blockIdx.x + i * gridDim.x;
    const int n0 = tile * 16;
    const int nrows = tile < ntiles && p < P ? min(16, a.N - n0) : 0;
    const rsrc_t rw = make_rsrc(a.W + (int64_t)(nrows ? n0 : 0) * KW, (uint32_t)nrows * KW * 4u);
    const rsrc_t rs = make_rsrc(a.S + (int64_t)(nrows ? n0 : 0) * SG, (uint32_t)nrows * SG * 2u);
    const int q0 = p * QP + wave * QW, qend = min(min(q0 + QW, (p + 1) * QP), Q);
#pragma unroll
    for (int qi = 0; qi < QWMAX; ++qi) {
      const uint32_t c = 4 * (q0 + qi) + lg;
      const uint32_t wo = (li * (uint32_t)KW * 4u + c * 16u) | (q0 + qi < qend ? 0u : kOut);
      it.w[qi] = __builtin_bit_cast(uint4v, __builtin_amdgcn_raw_buffer_load_b128(rw, wo, 0, 0));
    }
    const uint32_t q = q0 + lg;
    const uint32_t sidx = GS > 1 ? GS * q : q >> gshift;
    const uint32_t so = ((li * (uint32_t)SG + sidx) * 2u) | ((int)q < qend ? 0u : kOut);
    if constexpr (GS == 4)
      it.s = __builtin_bit_cast(uint2v, __builtin_amdgcn_raw_buffer_load_b64(rs, so, 0, 0));
    else if constexpr (GS == 2)
      it.s[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, so, 0, 0);
    else
      it.s[0] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, so, 0, 0);
  };

  float4v acc[T][MT];
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[i][mt] = float4v{};
  auto compute = [&](const Item& it, int i) {
#pragma unroll
    for (int qi = 0; qi < QWMAX; ++qi) {
      if (qi >= QW) break;  // uniform
      const int q = wave * QW + qi;  // of the phase
      uint32_t wt[4] = {it.w[qi][0], it.w[qi][1], it.w[qi][2], it.w[qi][3]};
      const int src = (li + 16 * qi) * 4;
      const uint32_t s01 = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)it.s[0]);
      const uint32_t s23 = GS == 4 ? (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)it.s[1]) : 0u;
      transpose_rows4(wt[0], wt[1], wt[2], wt[3]);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const uint32_t sw = GS == 4 ? (t < 2 ? s01 : s23) >> (16 * (t & 1)) : GS == 2 ? s01 >> (16 * (t >> 1)) : s01;
        const half_t s = __builtin_bit_cast(half_t, (uint16_t)sw);
        const half2v s1 = {s, s};
        half2v r[4];
        unpack_word(wt[t], nib, zp, r);
        const half2v d0 = r[0] * s1, d1 = r[1] * s1, d2 = r[2] * s1, d3 = r[3] * s1;
        const half8v bv = {d0[0], d0[1], d1[0], d1[1], d2[0], d2[1], d3[0], d3[1]};
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const half8v xa = xs[(mt * 4 * QPM + 4 * q + t) * kWave + 16 * lg + (li ^ (4 * t + lg))];
          acc[i][mt] = mfma16x16x32(xa, bv, acc[i][mt]);
        }
      }
    }
  };

  // One phase: tile 0 now, tile i + 1 when tile i's compute starts.  With
  // every tile requested up front, the wave stalls at the load instructions
  // once the CU's outstanding-request capacity is full, and X, compute and
  // the weight stream run one after another (M = 16: 12.0 -> 9.3 us).
  auto put = [&](int i) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[red_at(i, wave, 4 * mt + r, lane)] = acc[i][mt][r];
  };

  Item it[T + 1];
  xload(0);
  load_item(it[0], 0, 0);
  xstore();
  lds_barrier();
  if constexpr (!MP) {
#pragma unroll
    for (int i = 0; i < T; ++i) {
      if (i + 1 < T) load_item(it[i + 1], 0, i + 1);
      compute(it[i], i);
      put(i);
    }
  } else {
    for (int p = 0; p < P; ++p) {
      if (p + 1 < P) xload(p + 1);
#pragma unroll
      for (int i = 0; i < T; ++i) {
        if (i + 1 < T)
          load_item(it[i + 1], p, i + 1);
        else
          load_item(it[T], p + 1, 0);
        compute(it[i], i);
      }
      if (p + 1 < P) {
        lds_barrier();
        xstore();
        lds_barrier();
        it[0] = it[T];
      }
    }
    if (MT > 1) lds_barrier();
#pragma unroll
    for (int i = 0; i < T; ++i) put(i);
  }
  lds_barrier();

  // acc[i][mt] register r of lane l is D[16 mt + 4(l/16) + r][l%16] of tile i.
  for (int e = threadIdx.x; e < T * MT * 4 * kWave; e += WV * kWave) {
    const int i = e / (MT * 4 * kWave), r = (e / kWave) % (4 * MT), ln = e & 63;
    const int tile = blockIdx.x + i * gridDim.x;
    float v = 0.f;
#pragma unroll
    for (int wv = 0; wv < WV; ++wv) v += red[red_at(i, wv, r, ln)];
    const int m = 16 * (r >> 2) + 4 * (ln >> 4) + (r & 3);
    const int n = tile * 16 + (ln & 15);
    if (tile < ntiles && m < a.M && n < a.N) a.Y[(int64_t)m * a.ldy + n] = (half_t)v;
  }
}

template <int QWMAX, int GS, bool MP>
hipError_t launch_lds(const W4Args& a, hipStream_t s) {
  const int ntiles = (a.N + 15) / 16;
  const int cus = device_cu_count();
  int T = (ntiles + cus - 1) / cus;
  if (T > 4) T = 4;
  const dim3 grid((ntiles + T - 1) / T);
  constexpr int WV = 8;
  const dim3 block(WV * kWave);
  switch (T) {
    case 1: return launch<&w4a16_skinny_lds_kernel<WV, 1, QWMAX, GS, MP>>(
        ktag("w4a16_skinny_lds_kernel", WV, 1, QWMAX, GS, MP), grid, block, s, a);
    case 2: return launch<&w4a16_skinny_lds_kernel<WV, 2, QWMAX, GS, MP>>(
        ktag("w4a16_skinny_lds_kernel", WV, 2, QWMAX, GS, MP), grid, block, s, a);
    case 3: return launch<&w4a16_skinny_lds_kernel<WV, 3, QWMAX, GS, MP>>(
        ktag("w4a16_skinny_lds_kernel", WV, 3, QWMAX, GS, MP), grid, block, s, a);
    default: return launch<&w4a16_skinny_lds_kernel<WV, 4, QWMAX, GS, MP>>(
        ktag("w4a16_skinny_lds_kernel", WV, 4, QWMAX, GS, MP), grid, block, s, a);
  }
}

template <int QWMAX, bool MP>
hipError_t launch_gs(const W4Args& a, hipStream_t s) {
  return a.group == 32   ? launch_lds<QWMAX, 4, MP>(a, s)
         : a.group == 64 ? launch_lds<QWMAX, 2, MP>(a, s)
                         : launch_lds<QWMAX, 1, MP>(a, s);
}

}  // namespace

int w4a16_skinny_lds_max_k() { return 32 * 4 * kLdsQuads; }

bool w4a16_skinny_lds_groups(const W4Args& a) {
  return a.K % 128 == 0 && (a.group & (a.group - 1)) == 0;  // 32, 64, 128, ...
}

hipError_t launch_w4a16_skinny_lds(const W4Args& a, hipStream_t s) {
  if (a.M <= 16) return a.K <= w4a16_skinny_lds_max_k() ? launch_gs<4, false>(a, s) : launch_gs<4, true>(a, s);
  return launch_gs<2, true>(a, s);
}

}  // namespace neso
