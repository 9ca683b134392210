// Dense bf16 GEMM on MFMA for the shared expert and router projections of
// the prefill MoE block (fnx/engine.py:1786-1802 at more than four rows):
//
//   y[m, n] = bf16( sum_k a[m, k] * W[n, k] )   (F.linear, fp32 accumulation)
//
// a: bf16 rows of K (row m at a + m*lda), W: bf16 [N, K] row-major (the
// reference's Raw container), y: bf16 rows (row m at y + m*ldy).
//
// BM x BN output tiles per workgroup of 4 waves (2 x 2, each (BM/2) x (BN/2):
// TI x TJ v_mfma_f32_16x16x32_bf16 tiles). Both operands keep K contiguous,
// so a lane's MFMA fragment (8 consecutive k of one row of a, or of W) is one
// 16-byte piece: K runs in KC-wide chunks that stream straight into a ring of
// RING LDS slots by buffer-resource global->LDS DMA, RING - 1 chunks ahead,
// the 16-byte pieces of every row stored XOR-swizzled by row so the 16 rows a
// fragment read touches fall in different banks. One barrier per chunk.
// Workgroups that share rows of a run on one XCD. Outputs of a few tiles take a
// kernel of their own (below). SWIGLU (the fused shared-expert projection, W =
// [gate MI | up MI | rest]): the first 2 MI columns leave as the SwiGLU rows
// act = bf16(bf16(silu(g)) * u) of their bf16 results instead of y. Products of two bf16 are
// exact in fp32, so the result is the rounding of an fp32 accumulation of
// exact terms.
#include "qmoe_common.h"
#include "qmoe.h"

namespace {

typedef __bf16 bf16x8_v __attribute__((ext_vector_type(8)));
typedef float f32x4_v __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int BK = 32;  // k per MFMA step

template <int BM_, int BN_, int KC_, int RING_>
struct Bf16Tile {
  static constexpr int BM = BM_, BN = BN_, KC = KC_, RING = RING_;
  static constexpr int TI = BM / 32, TJ = BN / 32;
  static constexpr int NS = KC / BK;            // MFMA steps per chunk
  static constexpr int PPR = KC / 8;            // 16-byte pieces per row and chunk
  static constexpr int A_BYTES = BM * 2 * KC;
  static constexpr int B_BYTES = BN * 2 * KC;
  static constexpr int SLOT = A_BYTES + B_BYTES;
  static constexpr int AQ = A_BYTES / 1024 / 4;  // DMA instructions per wave and chunk (1 KB each)
  static constexpr int BQ = B_BYTES / 1024 / 4;
  static constexpr int IPC = AQ + BQ;
  static constexpr int LDS = RING * SLOT;
  static_assert(A_BYTES % 4096 == 0 && B_BYTES % 4096 == 0, "tile shape");
};

template <class T, bool SWIGLU>
__global__ __launch_bounds__(kThreads) void bf16_gemm_kernel(const uint16_t* __restrict__ a, long lda,
                                                             const uint16_t* __restrict__ w, uint16_t* __restrict__ y,
                                                             long ldy, int M, int K, int N, uint16_t* __restrict__ act,
                                                             int MI) {
  constexpr int BM = T::BM, BN = T::BN, KC = T::KC, RING = T::RING;
  constexpr int TI = T::TI, TJ = T::TJ, PPR = T::PPR;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int act_tiles = SWIGLU ? (MI + BN / 2 - 1) / (BN / 2) : 0;
  const int ntn = act_tiles + (N - (SWIGLU ? 2 * MI : 0) + BN - 1) / BN;
  const int ntiles = ((M + BM - 1) / BM) * ntn;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  if (tile >= ntiles) return;
  const int m0 = (tile / ntn) * BM, nt = tile % ntn;
  const bool sw = SWIGLU && nt < act_tiles;
  const int n0 = SWIGLU && !sw ? 2 * MI + (nt - act_tiles) * BN : nt * BN;
  // tile column c -> row of w (rows past the last re-read it, never stored). A
  // SwiGLU tile: columns c with c / 16 even are gate rows, odd the up rows of
  // the same act columns, so a lane holds both of an act column.
  auto wrow = [&](int c) {
    if (sw) return ((c >> 4) & 1) * MI + min(nt * (BN / 2) + 16 * (c >> 5) + (c & 15), MI - 1);
    return min(n0 + c, N - 1);
  };
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const int wm = wave >> 1, wn = wave & 1;
  const int i16 = lane & 15, kb = lane >> 4;
  // piece swizzle of row r: the 16 rows of a fragment read spread over the banks
  auto swz = [](int r) { return PPR == 4 ? ((r >> 2) & 3) : (r & 7); };

  // ---- DMA sources: instruction q of wave w covers rows (64 / PPR) (4q + w)
  // + lane / PPR of its operand; LDS piece lane % PPR of the row holds k-piece
  // (lane % PPR) ^ swz(row). Rows past M or N re-read the last one (never
  // stored). Buffer resources bound every access to its tensor.
  constexpr int kRsrcWord3 = 0x00020000;
  const __amdgpu_buffer_rsrc_t rsrc_a =
      __builtin_amdgcn_make_buffer_rsrc((void*)a, (short)0, (int)(((long)(M - 1) * lda + K) * 2), kRsrcWord3);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void*)w, (short)0, N * K * 2, kRsrcWord3);
  uint32_t aoff[T::AQ], boff[T::BQ];
#pragma unroll
  for (int q = 0; q < T::AQ; ++q) {
    const int r = (64 / PPR) * (4 * q + wave) + lane / PPR;
    aoff[q] = 2u * ((uint32_t)min(m0 + r, M - 1) * (uint32_t)lda + 8u * (uint32_t)((lane % PPR) ^ swz(r)));
  }
#pragma unroll
  for (int q = 0; q < T::BQ; ++q) {
    const int r = (64 / PPR) * (4 * q + wave) + lane / PPR;
    boff[q] = 2u * ((uint32_t)wrow(r) * (uint32_t)K + 8u * (uint32_t)((lane % PPR) ^ swz(r)));
  }
  auto issue_chunk = [&](int c) {
    unsigned char* base = lds + (c % RING) * T::SLOT;
    const int k0 = c * KC;
#pragma unroll
    for (int q = 0; q < T::AQ; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (__attribute__((address_space(3))) void*)(base + (4 * q + wave_u) * 1024),
                                               16, (int)aoff[q], k0 * 2, 0, 0);
#pragma unroll
    for (int q = 0; q < T::BQ; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc_b, (__attribute__((address_space(3))) void*)(base + T::A_BYTES + (4 * q + wave_u) * 1024), 16,
          (int)boff[q], k0 * 2, 0, 0);
  };

  f32x4_v acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = f32x4_v{0.f, 0.f, 0.f, 0.f};
  int arow[TI], brow[TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i) arow[i] = wm * (BM / 2) + 16 * i + i16;
#pragma unroll
  for (int j = 0; j < TJ; ++j) brow[j] = wn * (BN / 2) + 16 * j + i16;

  const int nch = K / KC;
#pragma unroll
  for (int c = 0; c < RING - 1; ++c)
    if (c < nch) issue_chunk(c);
  for (int c = 0; c < nch; ++c) {
    // chunk c has landed once only the later chunks in flight may be pending
    if (c + RING - 2 < nch) wait_vm_lgkm0<(RING - 2) * T::IPC>();
    else __builtin_amdgcn_s_waitcnt(0);
    // every wave is past chunk c - 1: its ring slot takes chunk c + RING - 1.
    // A barrier without a fence: the wait above has settled what it orders,
    // and __syncthreads' fence would also wait for the chunks prefetched ahead.
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (c + RING - 1 < nch) issue_chunk(c + RING - 1);
    const unsigned char* as = lds + (c % RING) * T::SLOT;
    const unsigned char* bs = as + T::A_BYTES;
#pragma unroll
    for (int st = 0; st < T::NS; ++st) {
      bf16x8_v bf[TJ];
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        const int r = brow[j];
        bf[j] = *reinterpret_cast<const bf16x8_v*>(bs + r * (2 * KC) + (((4 * st + kb) ^ swz(r)) << 4));
      }
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        const int r = arow[i];
        const bf16x8_v af = *reinterpret_cast<const bf16x8_v*>(as + r * (2 * KC) + (((4 * st + kb) ^ swz(r)) << 4));
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bf[j], acc[i][j], 0, 0, 0);
      }
    }
  }

  // lane holds column i16 of tile (i, j) for rows 4*kb + r
  if (sw) {
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; j += 2) {
        const int n = nt * (BN / 2) + 16 * ((wn * (BN / 2) + 16 * j) >> 5) + i16;
        if (n >= MI) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + wm * (BM / 2) + i * 16 + 4 * kb + r;
          if (m < M) act[(size_t)m * MI + n] = (uint16_t)swiglu_bf16_bits(f32_to_bf16(acc[i][j][r]), f32_to_bf16(acc[i][j + 1][r]));
        }
      }
    return;
  }
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      const int n = n0 + brow[j];
      if (n >= N) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm * (BM / 2) + i * 16 + 4 * kb + r;
        if (m < M) y[(size_t)m * ldy + n] = (uint16_t)f32_to_bf16(acc[i][j][r]);
      }
    }
}

struct Bf16Args {
  const uint16_t* x;
  long ldx;
  const uint16_t* w;
  uint16_t* y;
  long ldy;
  int M, K, N;
  uint16_t* act;  // SwiGLU form: act rows of the first 2 MI columns
  int MI;
};

template <bool SWIGLU>
long col_tiles(const Bf16Args& a, int bn) {
  return SWIGLU ? (long)host_ceil_div(a.MI, bn / 2) + host_ceil_div(a.N - 2 * a.MI, bn) : host_ceil_div(a.N, bn);
}

template <class T, bool SWIGLU>
int launch_bf16_gemm(const Bf16Args& a, hipStream_t stream) {
  int dev = 0;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return (int)err;
  if (dev < 0 || dev >= 64) return QMOE_EINVAL;
  static bool attr_set[64] = {};
  if (!attr_set[dev]) {
    err = hipFuncSetAttribute((const void*)bf16_gemm_kernel<T, SWIGLU>, hipFuncAttributeMaxDynamicSharedMemorySize, T::LDS);
    if (err != hipSuccess) return (int)err;
    attr_set[dev] = true;
  }
  const long tiles = (long)host_ceil_div(a.M, T::BM) * col_tiles<SWIGLU>(a, T::BN);
  const long blocks = (tiles + 7) / 8 * 8;  // whole XCD rounds (extra blocks exit)
  if (blocks > 0x7fffffffL) return QMOE_EINVAL;
  hipLaunchKernelGGL((bf16_gemm_kernel<T, SWIGLU>), dim3((unsigned)blocks), dim3(kThreads), T::LDS, stream, a.x, a.ldx, a.w,
                     a.y, a.ldy, a.M, a.K, a.N, a.act, a.MI);
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------- few tiles: K split over the waves
//
// 16 LIVE rows of a times 16 F columns per workgroup; the NW waves split K
// (contiguous runs of 32-k steps) and load both operands' fragments straight
// into registers (a fragment is one 16-byte piece per lane), U steps as one
// batch while the previous batch's MFMAs run. The waves' partial tiles meet in
// LDS and are summed in wave order: the same bits every run. SWIGLU: the tiles of
// the first 2 MI columns take 8 F gate columns, then their 8 F up columns.
//
// What bounds it: launch and first load (about 4 us) and the (LIVE + F) KB per
// step that a CU draws from L2 at some 27 bytes per clock. 2560 x 1793: 7.2 us
// at 5 rows (1.3 TB/s of cold weights) and 11.3 at 64, against 19.4 and 24.1 of
// the 64 x 64 LDS-ring tile, whose one chain of 32-k chunks ran on 29 CUs;
// 2048 x 512 at 200 rows 7.9 against 14.4.
template <int LIVE, int F, int NW, int U, bool SWIGLU>
__global__ __launch_bounds__(64 * NW) void bf16_skinny_kernel(Bf16Args g) {
  constexpr int BN = 16 * F, ROWS = 16 * LIVE, LDR = BN + 4;  // LDS row: the four k-blocks' rows in different banks
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  float* red = reinterpret_cast<float*>(lds);  // [NW][ROWS][LDR]
  const int M = g.M, K = g.K, N = g.N, MI = g.MI;
  const int nrg = (M + ROWS - 1) / ROWS;
  const int act_tiles = SWIGLU ? (MI + BN / 2 - 1) / (BN / 2) : 0;
  const int ntn = act_tiles + (N - (SWIGLU ? 2 * MI : 0) + BN - 1) / BN;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  if (tile >= nrg * ntn) return;
  const int m0 = (tile % nrg) * ROWS, nt = tile / nrg;
  const bool sw = SWIGLU && nt < act_tiles;
  const int n0 = SWIGLU && !sw ? 2 * MI + (nt - act_tiles) * BN : nt * BN;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i16 = lane & 15, kb = lane >> 4;
  // tile column c -> row of w (rows past the last re-read it, never stored)
  auto wrow = [&](int c) {
    if (sw) return (c / (BN / 2)) * MI + min(nt * (BN / 2) + c % (BN / 2), MI - 1);
    return min(n0 + c, N - 1);
  };
  constexpr int kRsrcWord3 = 0x00020000;
  const __amdgpu_buffer_rsrc_t rsrc_a =
      __builtin_amdgcn_make_buffer_rsrc((void*)g.x, (short)0, (int)(((long)(M - 1) * g.ldx + K) * 2), kRsrcWord3);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void*)g.w, (short)0, N * K * 2, kRsrcWord3);
  int aoff[LIVE], boff[F];
#pragma unroll
  for (int t = 0; t < LIVE; ++t) aoff[t] = (int)(2 * ((long)min(m0 + 16 * t + i16, M - 1) * g.ldx + 8 * kb));
#pragma unroll
  for (int f = 0; f < F; ++f) boff[f] = 2 * (wrow(16 * f + i16) * K + 8 * kb);
  const int nsteps = K / BK, per = (nsteps + NW - 1) / NW;
  const int s0 = min(nsteps, wave * per), s1 = min(nsteps, s0 + per);
  f32x4_v acc[LIVE][F];
#pragma unroll
  for (int t = 0; t < LIVE; ++t)
#pragma unroll
    for (int f = 0; f < F; ++f) acc[t][f] = f32x4_v{0.f, 0.f, 0.f, 0.f};
  struct Batch {
    bf16x8_v a[U][LIVE], b[U][F];
  };
  auto load = [&](int st, Batch& v) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int off = 2 * BK * min(st + u, s1 - 1);  // past the run's end its last step (not used)
#pragma unroll
      for (int f = 0; f < F; ++f)
        v.b[u][f] = __builtin_bit_cast(bf16x8_v, __builtin_amdgcn_raw_buffer_load_b128(rsrc_b, boff[f], off, 0));
#pragma unroll
      for (int t = 0; t < LIVE; ++t)
        v.a[u][t] = __builtin_bit_cast(bf16x8_v, __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, aoff[t], off, 0));
    }
  };
  auto mma = [&](int st, const Batch& v) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (st + u >= s1) break;
#pragma unroll
      for (int t = 0; t < LIVE; ++t)
#pragma unroll
        for (int f = 0; f < F; ++f)
          acc[t][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v.a[u][t], v.b[u][f], acc[t][f], 0, 0, 0);
    }
  };
  if (s0 < s1) {
    Batch v0, v1;
    load(s0, v0);
    for (int st = s0; st < s1; st += 2 * U) {
      if (st + U < s1) load(st + U, v1);
      mma(st, v0);
      if (st + 2 * U < s1) load(st + 2 * U, v0);
      if (st + U < s1) mma(st + U, v1);
    }
  }
  // lane holds column i16 of each fragment for rows 4 kb + r
#pragma unroll
  for (int t = 0; t < LIVE; ++t)
#pragma unroll
    for (int f = 0; f < F; ++f)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[((size_t)wave * ROWS + 16 * t + 4 * kb + r) * LDR + 16 * f + i16] = acc[t][f][r];
  __syncthreads();
  auto total = [&](int row, int c) {
    float v = red[row * LDR + c];
#pragma unroll
    for (int q = 1; q < NW; ++q) v += red[((size_t)q * ROWS + row) * LDR + c];
    return v;
  };
  const int rows = min(ROWS, M - m0);
  if (sw) {
    for (int p = tid; p < rows * (BN / 2); p += 64 * NW) {
      const int row = p / (BN / 2), c = p % (BN / 2), col = nt * (BN / 2) + c;
      const uint32_t gb = f32_to_bf16(total(row, c)), ub = f32_to_bf16(total(row, BN / 2 + c));
      if (col < MI) g.act[(size_t)(m0 + row) * MI + col] = (uint16_t)swiglu_bf16_bits(gb, ub);
    }
    return;
  }
  for (int p = tid; p < rows * BN; p += 64 * NW) {
    const int row = p / BN, c = p % BN;
    if (n0 + c < N) g.y[(size_t)(m0 + row) * g.ldy + n0 + c] = (uint16_t)f32_to_bf16(total(row, c));
  }
}

template <int LIVE, int F, int NW, int U, bool SWIGLU>
int launch_bf16_skinny(const Bf16Args& a, hipStream_t stream) {
  constexpr int kLds = NW * 16 * LIVE * (16 * F + 4) * 4;
  static_assert(kLds <= 160 * 1024, "LDS of a CU");
  int dev = 0;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return (int)err;
  if (dev < 0 || dev >= 64) return QMOE_EINVAL;
  static bool attr_set[64] = {};
  auto* kern = bf16_skinny_kernel<LIVE, F, NW, U, SWIGLU>;
  if (!attr_set[dev]) {
    err = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (err != hipSuccess) return (int)err;
    attr_set[dev] = true;
  }
  const long blocks = (host_ceil_div(a.M, 16 * LIVE) * col_tiles<SWIGLU>(a, 16 * F) + 7) / 8 * 8;  // whole XCD rounds
  if (blocks > 0x7fffffffL) return QMOE_EINVAL;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(64 * NW), kLds, stream, a);
  return (int)hipGetLastError();
}

// The skinny kernel where a tile of at most four fragments (LIVE + F) covers
// the output in one round of the 256 CUs; false where none does.
// Eight waves with longer batches for a long K (2560 x 1793 at 48 rows 11.0
// against 11.5 us with 16), 16 for a short one (640 x 2560 4.4 against 5.0).
template <bool SWIGLU>
bool launch_bf16_few_tiles(const Bf16Args& a, hipStream_t st, int* rc) {
  auto fits = [&](int live, int f) { return host_ceil_div(a.M, 16 * live) * col_tiles<SWIGLU>(a, 16 * f) <= 256; };
  const bool long_k = a.K >= 1536;
#define QMOE_SKINNY(L_, F_, U8_, U16_)                                                 \
  if (fits(L_, F_)) {                                                                  \
    *rc = long_k ? launch_bf16_skinny<L_, F_, 8, U8_, SWIGLU>(a, st)                   \
                 : launch_bf16_skinny<L_, F_, 16, U16_, SWIGLU>(a, st);                \
    return true;                                                                       \
  }
  QMOE_SKINNY(1, 1, 4, 2) QMOE_SKINNY(1, 2, 4, 2) QMOE_SKINNY(2, 1, 4, 2) QMOE_SKINNY(2, 2, 2, 2)
  QMOE_SKINNY(3, 1, 2, 2)
#undef QMOE_SKINNY
  return false;
}

template <bool SWIGLU>
int run_bf16_gemm(const Bf16Args& a, hipStream_t st) {
  int rc = QMOE_OK;
  if (launch_bf16_few_tiles<SWIGLU>(a, st, &rc)) return rc;
  // 64 x 64 tiles while each has a CU of its own: 128-k chunks in three slots
  // (2560 x 1793 at 200 rows 13.7 us against 20.3 with 32-k chunks in four, 14.3
  // with 64-k ones; K split over two rings per workgroup: no gain, 13.5).
  if ((long)host_ceil_div(a.M, 64) * col_tiles<SWIGLU>(a, 64) <= 256) {
    if (a.K % 128 == 0) return launch_bf16_gemm<Bf16Tile<64, 64, 128, 3>, SWIGLU>(a, st);
    if (a.K % 64 == 0) return launch_bf16_gemm<Bf16Tile<64, 64, 64, 4>, SWIGLU>(a, st);
    return launch_bf16_gemm<Bf16Tile<64, 64, 32, 4>, SWIGLU>(a, st);
  }
  // 128 x 128 tiles where they give every CU two workgroups. 64-k chunks,
  // double-buffered at 128 x 128, where K allows (4096 x 3072 x 2048: 650 -> 980
  // TFLOP/s against 32-k chunks in a 4-slot ring: half the barriers and waits
  // per MFMA)
  if ((long)host_ceil_div(a.M, 128) * col_tiles<SWIGLU>(a, 128) >= 512)
    return a.K % 64 == 0 ? launch_bf16_gemm<Bf16Tile<128, 128, 64, 2>, SWIGLU>(a, st)
                         : launch_bf16_gemm<Bf16Tile<128, 128, 32, 4>, SWIGLU>(a, st);
  // 128 x 64 tiles where they give every CU one, and with fewer where they run
  // 64-k chunks of a K of 512 or more; else 64 x 64 tiles, two or more per CU. us from
  // cold operands, 128 x 64 against 64 x 64: 400 x 768 x 3072 9.9 / 10.8, 512 x 640 x 2560
  // 9.2 / 11.3, 1200 x 1536 x 1500 15.5 / 19.9, 130 x 512 x 6000 8.2 / 8.2; but 768 x 320
  // x 1500 6.3 / 5.9, 130 x 320 x 6000 6.9 / 6.5, and with 32-k chunks 640 x 672 x 2048 11.1 /
  // 9.9, 768 x 1632 x 1500 19.3 / 15.4.
  const bool full = (long)host_ceil_div(a.M, 128) * col_tiles<SWIGLU>(a, 64) >= 256;
  if (a.K % 64 == 0 && (full || a.K >= 512)) return launch_bf16_gemm<Bf16Tile<128, 64, 64, 3>, SWIGLU>(a, st);
  return full ? launch_bf16_gemm<Bf16Tile<128, 64, 32, 4>, SWIGLU>(a, st)
              : launch_bf16_gemm<Bf16Tile<64, 64, 32, 4>, SWIGLU>(a, st);
}

bool bf16_gemm_ok(const void* x, long ldx, const void* w, long ldy, int M, int K, int N) {
  return M >= 1 && N >= 1 && K >= BK && K % BK == 0 && ldx >= K && ldx % 8 == 0 && ldy >= N && ((uintptr_t)x & 15) == 0 &&
         ((uintptr_t)w & 15) == 0 && ((long)(M - 1) * ldx + K) * 2 < 0x80000000L && (long)N * K * 2 < 0x80000000L;
}

}  // namespace

extern "C" {

int qmoe_bf16_gemm(const void* x, long ldx, const void* w, void* y, long ldy, int M, int K, int N, void* stream) {
  if (!bf16_gemm_ok(x, ldx, w, ldy, M, K, N)) return QMOE_EINVAL;
  return run_bf16_gemm<false>({(const uint16_t*)x, ldx, (const uint16_t*)w, (uint16_t*)y, ldy, M, K, N, nullptr, 0},
                              (hipStream_t)stream);
}

int qmoe_bf16_gemm_swiglu(const void* x, long ldx, const void* w, void* y, long ldy, void* act, int M, int K, int N,
                          int MI, void* stream) {
  if (!bf16_gemm_ok(x, ldx, w, ldy, M, K, N) || MI < 1 || N <= 2 * MI) return QMOE_EINVAL;
  return run_bf16_gemm<true>({(const uint16_t*)x, ldx, (const uint16_t*)w, (uint16_t*)y, ldy, M, K, N, (uint16_t*)act, MI},
                             (hipStream_t)stream);
}

}  // extern "C"
