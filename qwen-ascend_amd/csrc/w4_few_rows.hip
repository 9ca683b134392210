// W4A16 MFMA for row tiles of a few rows (gfx950): the projections of a batch
// of decoding sequences or a short prompt, dense or by expert.
//
//   y[p, n] = bf16( sum_k x[p, k] * q[e_p, k, n] * S[e_p, k / gs, n] )
//
// A workgroup owns one row tile (up to ROWS rows of one expert) and WC column
// blocks of 16 F columns; for each block WK waves split K (contiguous runs of
// 32-k steps), every wave streaming its weights straight into registers in
// MFMA B-fragment order: lane (i16, kb) reads for each of its 8 k rows
// 32 s + 8 kb + i one int32 word, whose nibbles are the B fragments of its
// columns (F = 8: word i16, all eight; F = 4: word i16 % 8, nibbles 4 (i16 / 8)
// and the next three). The waves' partial tiles meet in LDS and are summed in
// wave order: no second launch and no partials in memory, the same bits every
// run. D steps of weights per wave are in flight.
//
// Exact fp16 operands. The tile's activation rows are converted once per
// workgroup into LDS: a' = a * 2^er with er per row such that max |a'| is in
// [2^13, 2^14), exact as in the tiled kernel, while the first weights are on
// their way. A nibble pair becomes fp16 1024 + u or 1024 + 16 u (u = q + 8) in
// place, without a shift, by one v_bitop3 (mask, flip of the nibble's top bit,
// exponent), and q = that - 1032 or / 16 - 72 by one packed fma, exact. A scale
// group's sums are scaled by S[g, n] in fp32; the result by 2^-er. Those sums stay
// below 2^29 |S|, so only a scale above 2^98 can take them out of the fp32 range
// while the result, 2^er smaller, is in it: an output whose sum is not finite is
// summed again from the inputs in 64 bits. No scale made from an int8 and an fp16
// base is near that, so the range costs one test per four outputs (48 rows, 2048 x
// 4096: 9.17 against 9.12 us), not a pass over the scales ahead of the weights. Where
// every output of that call is summed again it takes 225 us.
//
// Modes: 0 = y rows; 1 = SwiGLU act, the first half of the column blocks the gate
// and the second half the up columns of the same act columns; 2 = down projection with the routing weight,
// prod[perm[p], n] = bf16(bf16(y) * w[perm[p]]).
//
// What bounds it. By expert: the weight stream, 70 us for 324 MB of gate_up
// (2560 x 1280 g64, 23 tokens; 4.6 TB/s, the loads alone 66 us, the arithmetic
// on cached weights 49 us); the tiled kernel, whose workgroup runs one chain of
// 64-k chunks with two in flight, took 81.5 us and two more launches for the
// fp16 rows. Dense: the workgroup's own chain (launch, rows, weights, sums), 11
// us for 4.3 MB at 48 rows (2048 x 4096) against 30 us of the tiled kernel, whose
// 16 workgroups each ran all of K.
#include "qmoe_common.h"
#include "qmoe.h"
#include "w4_few_rows.h"

#include <algorithm>

namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_v __attribute__((ext_vector_type(4)));

constexpr int BK = 32;  // k per MFMA step

QMOE_DEV half2_t as_h2(uint32_t v) { return __builtin_bit_cast(half2_t, v); }
QMOE_DEV uint32_t h2_bits(half2_t v) { return __builtin_bit_cast(uint32_t, v); }

constexpr size_t few_rows_lds(int rows, int wc, int wk, int f, int K) {
  const size_t a = (size_t)rows * (2 * K + 16), r = (size_t)wk * rows * wc * 16 * f * 4;
  return (a > r ? a : r) + 3 * 4 * (size_t)rows;
}

template <int MODE, int ROWS, int F, int WC, int WK, int D>
__global__ __launch_bounds__(64 * WC * WK) void w4_few_rows_kernel(FewRowsArgs g, int n_ntiles) {
  constexpr int NW = WC * WK, LIVE = (ROWS + 15) / 16;
  constexpr int CB = 16 * F;                    // columns per column block
  constexpr int CT = WC * CB;                   // columns per workgroup
  constexpr int CA = CT / 2;                    // mode 1: act columns
  constexpr int kPieces = kFewRowsMaxK / 512;   // 16-byte pieces of a row per lane
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int K = g.K, N = g.N, nw = N >> 3;
  const int lda = 2 * K + 16;                   // bytes per fp16 row (16 more: rows in different banks)
  float* red = reinterpret_cast<float*>(lds);   // [WK][ROWS][CT], over the rows once they are used up
  const size_t row_data = max((size_t)ROWS * lda, (size_t)WK * ROWS * CT * 4);
  int* s_erow = reinterpret_cast<int*>(lds + row_data);             // row exponents
  int* s_orow = s_erow + ROWS;                                      // mode 2: output row
  float* s_wrow = reinterpret_cast<float*>(s_orow + ROWS);          // mode 2: routing weight

  // ---- tile of this block: XCD x takes row tiles x, x + 8, ... in table order,
  // each with its column tiles in a row
  // The table entry is read beside the count, not after it (one round trip less
  // ahead of everything else); past the count it is not used.
  int mt, nt, tiles_m, e = 0, row0 = 0, rows = 0;
  if (g.tile_expert != nullptr) {
    const int xi = (int)(blockIdx.x >> 3);
    nt = xi % n_ntiles;
    mt = 8 * (xi / n_ntiles) + (int)(blockIdx.x & 7);
    const int at = min(mt, g.mtiles_max - 1);
    tiles_m = min(g.tile_count[0], g.mtiles_max);
    e = g.tile_expert[at];
    row0 = g.tile_row0[at];
    rows = g.tile_rows[at];
    asm volatile("" : "+s"(e), "+s"(row0), "+s"(rows), "+s"(tiles_m));  // all loaded before the first is tested
    rows = min(ROWS, rows);
  } else {
    // dense: the row tiles of a column tile side by side on one XCD
    tiles_m = (g.R + ROWS - 1) / ROWS;
    const int b = xcd_remap(blockIdx.x, gridDim.x);
    mt = b % tiles_m;
    nt = b / tiles_m;
    row0 = mt * ROWS;
    rows = min(ROWS, g.R - row0);
  }
  if (mt >= tiles_m || nt >= n_ntiles) return;
  if (rows <= 0) return;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wc = wave % WC, wk = wave / WC;
  const int i16 = lane & 15, kb = lane >> 4;

  // ---- this lane's word and scales
  const int word_l = F == 8 ? i16 : (i16 & 7);           // word within the block
  const int col_l = F == 8 ? 8 * i16 : 8 * word_l + 4 * (i16 >> 3);  // its first column within the block
  int c0, cs;                                            // columns of the word, of the lane's first value
  bool ok;
  if (MODE == 1) {
    const int a = nt * CA + (wc % (WC / 2)) * CB + 8 * word_l;
    ok = a < g.MI;
    c0 = (ok ? a : 0) + (wc / (WC / 2)) * g.MI;
  } else {
    c0 = nt * CT + wc * CB + 8 * word_l;
    ok = c0 < N;
    if (!ok) c0 = 0;
  }
  cs = c0 + (F == 8 ? 0 : 4 * (i16 >> 3));
  const uint32_t* we = g.w + (size_t)e * K * nw;
  const int G = K / g.gs;
  const uint16_t* se = g.s + (size_t)e * G * N;
  constexpr int kRsrcWord3 = 0x00020000;
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void*)we, (short)0, K * nw * 4, kRsrcWord3);
  const __amdgpu_buffer_rsrc_t rsrc_s = __builtin_amdgcn_make_buffer_rsrc((void*)se, (short)0, G * N * 2, kRsrcWord3);
  const int boff = 4 * (8 * kb * nw + (c0 >> 3));

  // ---- this wave's run of steps; the load position's scale group is counted
  const int nsteps = K / BK, spg = g.gs / BK;
  const int per = (nsteps + WK - 1) / WK;
  const int s0 = min(nsteps, wk * per), s1 = min(nsteps, s0 + per);
  struct Step {
    uint32_t b[8];
    uint32_t s[F / 2];
  };
  // a wave without steps (s0 == nsteps: fewer steps than slices) loads the last
  // one, which it does not use: row K is past the last expert's weights
  const int l0 = min(s0, nsteps - 1), g0 = l0 / spg;
  int lq = l0, lrow = g0 * N * 2, lleft = spg - (l0 - g0 * spg), cleft = lleft;
  auto load_step = [&](Step& v) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      v.b[i] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rsrc_b, boff, (lq * BK + i) * nw * 4, 0);
    if constexpr (F == 8) {
      const uint4 sv = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_s, 2 * cs, lrow, 0));
      v.s[0] = sv.x; v.s[1] = sv.y; v.s[2] = sv.z; v.s[3] = sv.w;
    } else {
      const uint2 sv = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rsrc_s, 2 * cs, lrow, 0));
      v.s[0] = sv.x; v.s[1] = sv.y;
    }
    // a run's last step is loaded again past its end (not used)
    if (lq + 1 < s1) {
      ++lq;
      if (--lleft == 0) {
        lleft = spg;
        lrow += 2 * N;
      }
    }
  };

  // ---- activation rows to fp16 in LDS, one wave per row; the loads of a
  // wave's first row go out ahead of its first weights
  const int32_t* perm_lo = reinterpret_cast<const int32_t*>(g.perm);  // entries are < 2^31
  uint4 xv[kPieces];
  int prow = 0;
  auto load_row = [&](int r) {
    const int p = row0 + r;
    prow = MODE == 0 ? p : perm_lo[2 * (size_t)p];
    const uint16_t* xr = g.x + (size_t)(MODE == 1 ? prow / g.topk : p) * K;
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int c = lane * 8 + 512 * i;
      xv[i] = c < K ? *reinterpret_cast<const uint4*>(xr + c) : make_uint4(0u, 0u, 0u, 0u);
    }
  };
  auto convert_row = [&](int r) {
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const uint32_t vv[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w};
#pragma unroll
      for (int q = 0; q < 4; ++q) m = max(m, max(vv[q] & 0x7fffu, (vv[q] >> 16) & 0x7fffu));
    }
    m = wave_max_u32(m);
    const int ex = exp_to(m, 140);
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int c = lane * 8 + 512 * i;
      const uint32_t vv[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w};
      uint32_t h[4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        h[q] = pk_rtz(ldexpf(__uint_as_float(vv[q] << 16), ex), ldexpf(__uint_as_float(vv[q] & 0xffff0000u), ex));
      if (c < K) *reinterpret_cast<uint4*>(lds + (size_t)r * lda + 2 * c) = make_uint4(h[0], h[1], h[2], h[3]);
    }
    if (lane == 0) {
      s_erow[r] = ex;
      if (MODE == 2) {
        s_orow[r] = prow;
        s_wrow[r] = bf16_to_f32(g.wts[prow]);
      }
    }
  };
  Step ring[D];
  if (wave < rows) load_row(wave);
  asm volatile("" ::: "memory");
#pragma unroll
  for (int d = 0; d < D; ++d) load_step(ring[d]);
  asm volatile("" ::: "memory");
  if (wave < rows) convert_row(wave);
  for (int r = wave + NW; r < rows; r += NW) {
    load_row(r);
    convert_row(r);
  }
  // the rows are written; the weights stay in flight
  wait_vm_lgkm0<63>();
  asm volatile("" ::: "memory");
  barrier_no_fence();

  // ---- main loop
  const unsigned char* ap[LIVE];
#pragma unroll
  for (int t = 0; t < LIVE; ++t) ap[t] = lds + (size_t)min(16 * t + i16, rows - 1) * lda + 16 * kb;
  f32x4_v acc[LIVE][F], accg[LIVE][F];
#pragma unroll
  for (int t = 0; t < LIVE; ++t)
#pragma unroll
    for (int f = 0; f < F; ++f) acc[t][f] = accg[t][f] = f32x4_v{0.f, 0.f, 0.f, 0.f};
  // byte selectors: byte b of two words to the low bytes of a dword's halves
  const uint32_t sel0 = F == 8 ? 0x0c040c00u : (i16 >> 3) ? 0x0c060c02u : 0x0c040c00u;
  auto compute = [&](int q, const Step& v) {
    half8_t af[LIVE];
#pragma unroll
    for (int t = 0; t < LIVE; ++t) af[t] = *reinterpret_cast<const half8_t*>(ap[t] + q * (2 * BK));
#pragma unroll
    for (int b = 0; b < F / 2; ++b) {
      uint32_t ev[4], od[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const uint32_t t = __builtin_amdgcn_perm(v.b[2 * p + 1], v.b[2 * p], sel0 + 0x00010001u * (uint32_t)b);
        const half2_t me = as_h2(__builtin_amdgcn_bitop3_b32(t, 0x000f000fu, 0x64086408u, 0x6A));  // 1024 + u
        const half2_t mo = as_h2(__builtin_amdgcn_bitop3_b32(t, 0x00f000f0u, 0x64806480u, 0x6A));  // 1024 + 16 u
        const half2_t k1 = {(_Float16)-1032.0f, (_Float16)-1032.0f}, k2 = {(_Float16)0.0625f, (_Float16)0.0625f},
                      k3 = {(_Float16)-72.0f, (_Float16)-72.0f};
        ev[p] = h2_bits(me + k1);
        od[p] = h2_bits(__builtin_elementwise_fma(mo, k2, k3));
      }
      const half8_t be = __builtin_bit_cast(half8_t, make_uint4(ev[0], ev[1], ev[2], ev[3]));
      const half8_t bo = __builtin_bit_cast(half8_t, make_uint4(od[0], od[1], od[2], od[3]));
#pragma unroll
      for (int t = 0; t < LIVE; ++t) {
        accg[t][2 * b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[t], be, accg[t][2 * b], 0, 0, 0);
        accg[t][2 * b + 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[t], bo, accg[t][2 * b + 1], 0, 0, 0);
      }
    }
    if (--cleft == 0 || q + 1 == s1) {
      cleft = spg;
#pragma unroll
      for (int f = 0; f < F; ++f) {
        const float sc = __uint_as_float((f & 1) ? (v.s[f >> 1] & 0xffff0000u) : (v.s[f >> 1] << 16));
#pragma unroll
        for (int t = 0; t < LIVE; ++t) {
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[t][f][r] = __builtin_fmaf(accg[t][f][r], sc, acc[t][f][r]);
          accg[t][f] = f32x4_v{0.f, 0.f, 0.f, 0.f};
        }
      }
    }
  };
  for (int q = s0; q < s1; q += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (q + d < s1) compute(q + d, ring[d]);
      if (q + d + D < s1) load_step(ring[d]);
    }
  }
  __syncthreads();  // the rows are used up
  // lane holds, for each row tile, rows 4 kb + r of its F columns
#pragma unroll
  for (int t = 0; t < LIVE; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * t + 4 * kb + r;
      if (row < rows) {
        float* dst = red + ((size_t)wk * ROWS + row) * CT + wc * CB + col_l;
#pragma unroll
        for (int f = 0; f < F; f += 4)
          *reinterpret_cast<float4*>(dst + f) = make_float4(acc[t][f][r], acc[t][f + 1][r], acc[t][f + 2][r], acc[t][f + 3][r]);
      }
    }
  __syncthreads();

  // ---- sums over the waves in order, four columns per thread and item
  // Output columns col .. col + 3 of a row from the inputs, in 64 bits
  auto resum = [&](int row, int col, float (&o)[4]) {
    const int p = row0 + row;
    const uint16_t* xr = g.x + (size_t)(MODE == 1 ? perm_lo[2 * (size_t)p] / g.topk : p) * K;
    double v[4] = {0., 0., 0., 0.};
#pragma unroll 4
    for (int k = 0; k < K; ++k) {
      const uint32_t word = we[(size_t)k * nw + (col >> 3)] >> (4 * (col & 7));  // col is a multiple of 4
      const uint16_t* sr = se + (size_t)(k / g.gs) * N + col;
      const double xk = (double)bf16_to_f32(xr[k]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        v[j] += xk * (double)((int)(word << (28 - 4 * j)) >> 28) * (double)bf16_to_f32(sr[j]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = (float)v[j];
  };
  // tile columns c .. c + 3, which are columns col .. of the weights
  auto total = [&](int row, int c, int col, bool ok_col, int ex, float (&o)[4]) {
    float4 b[WK];
#pragma unroll
    for (int q = 0; q < WK; ++q) b[q] = *reinterpret_cast<const float4*>(red + ((size_t)q * ROWS + row) * CT + c);
    __builtin_amdgcn_sched_barrier(0);  // every read on its way before the first sum
    float4 a = b[0];
#pragma unroll
    for (int q = 1; q < WK; ++q) {
      a.x += b[q].x;
      a.y += b[q].y;
      a.z += b[q].z;
      a.w += b[q].w;
    }
    o[0] = ldexpf(a.x, -ex);
    o[1] = ldexpf(a.y, -ex);
    o[2] = ldexpf(a.z, -ex);
    o[3] = ldexpf(a.w, -ex);
    // left the fp32 range (not a padding column, nor a row that holds an infinity or NaN)
    const bool left = !(fabsf(a.x) + fabsf(a.y) + fabsf(a.z) + fabsf(a.w) < INFINITY);
    if (__builtin_expect(left, 0) && ok_col && ex != exp_to(0x7f80u, 140)) resum(row, col, o);
  };
  constexpr int C4 = (MODE == 1 ? CA : CT) / 4;
  for (int p = tid; p < rows * C4; p += 64 * NW) {
    const int row = p / C4, c = 4 * (p % C4);
    const int ex = s_erow[row], col = nt * (MODE == 1 ? CA : CT) + c;
    const bool in = col < (MODE == 1 ? g.MI : N);
    float v[4];
    total(row, c, col, in, ex, v);
    const uint32_t p01 = pk_bf16(v[0], v[1]), p23 = pk_bf16(v[2], v[3]);
    auto lo = [](uint32_t u) { return __uint_as_float(u << 16); };
    auto hi = [](uint32_t u) { return __uint_as_float(u & 0xffff0000u); };
    if (MODE == 1) {
      float u[4];
      total(row, CA + c, g.MI + col, in, ex, u);
      const uint32_t u01 = pk_bf16(u[0], u[1]), u23 = pk_bf16(u[2], u[3]);
      if (in)
        *reinterpret_cast<uint2*>(g.y + (size_t)(row0 + row) * g.ldy + col) =
            make_uint2(pk_bf16(silu_f32(lo(p01)) * lo(u01), silu_f32(hi(p01)) * hi(u01)),
                       pk_bf16(silu_f32(lo(p23)) * lo(u23), silu_f32(hi(p23)) * hi(u23)));
    } else {
      if (in) {
        if (MODE == 2) {
          const float wv = s_wrow[row];
          *reinterpret_cast<uint2*>(g.y + (size_t)s_orow[row] * g.ldy + col) =
              make_uint2(pk_bf16(lo(p01) * wv, hi(p01) * wv), pk_bf16(lo(p23) * wv, hi(p23) * wv));
        } else {
          *reinterpret_cast<uint2*>(g.y + (size_t)(row0 + row) * g.ldy + col) = make_uint2(p01, p23);
        }
      }
    }
  }
}

template <int MODE, int ROWS, int F, int WC, int WK, int D>
int go(const FewRowsArgs& a, hipStream_t st) {
  constexpr int kMaxLds = 160 * 1024;
  const size_t lds = few_rows_lds(ROWS, WC, WK, F, a.K);
  if (lds > kMaxLds) return QMOE_EINVAL;
  int dev = 0;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return (int)err;
  if (dev < 0 || dev >= 64) return QMOE_EINVAL;
  static bool attr_set[64] = {};
  if (!attr_set[dev]) {
    err = hipFuncSetAttribute((const void*)w4_few_rows_kernel<MODE, ROWS, F, WC, WK, D>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds);
    if (err != hipSuccess) return (int)err;
    attr_set[dev] = true;
  }
  const int n_ntiles = MODE == 1 ? host_ceil_div(a.MI, WC / 2 * 16 * F) : host_ceil_div(a.N, WC * 16 * F);
  const long tiles = a.tile_expert != nullptr ? 8L * host_ceil_div(a.mtiles_max, 8) : host_ceil_div(a.R, ROWS);
  const long blocks = (tiles * n_ntiles + 7) / 8 * 8;
  if (blocks <= 0) return QMOE_OK;
  if (blocks > 0x7fffffffL) return QMOE_EINVAL;
  hipLaunchKernelGGL((w4_few_rows_kernel<MODE, ROWS, F, WC, WK, D>), dim3((unsigned)blocks), dim3(64 * WC * WK), lds, st, a,
                     n_ntiles);
  return (int)hipGetLastError();
}

}  // namespace

bool w4_few_rows_ok(int K, int N, int gs) {
  return K >= 64 && K % 64 == 0 && K <= kFewRowsMaxK && N >= 32 && N % 32 == 0 && gs >= BK && gs % BK == 0 && K % gs == 0;
}

// Tiles of 12 rows: the fp16 rows of two workgroups fit a CU's LDS up to K = 3072
// (16-row tiles leave one from K = 2560 on), four K-slices of 256 columns. An
// act tile of 256 columns (128-byte row pieces of gate and of up, two K-slices)
// where the width is a multiple of it, else 128: 2048/512 128 tokens 199 against
// 206 us per block, 3072/768 393 against 413; 2560/640 23 tokens 166 against 143.
int launch_w4_few_rows(int mode, const FewRowsArgs& a, hipStream_t st) {
  if (mode == 0) return go<0, kFewRowsTile, 8, 2, 4, 2>(a, st);
  if (mode == 1)
    return a.MI % 256 == 0 ? go<1, kFewRowsTile, 8, 4, 2, 2>(a, st) : go<1, kFewRowsTile, 8, 2, 4, 3>(a, st);
  return go<2, kFewRowsTile, 4, 4, 2, 2>(a, st);
}

// Dense rows: 64-column tiles, K over 16 waves, while the workgroups fit the 256
// CUs at once; else 128-column ones (half the conversions of x per weight):
// 2048 x 4096 at 128 rows 12.3 against 18.0 us.
int launch_w4_few_rows_dense(const FewRowsArgs& a, hipStream_t st) {
  if ((long)host_ceil_div(a.R, 16) * host_ceil_div(a.N, 64) <= 256) return go<0, 16, 4, 1, 16, 2>(a, st);
  return go<0, 16, 8, 1, 16, 2>(a, st);
}
