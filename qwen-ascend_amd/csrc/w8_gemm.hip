// W8A16 per-group GEMM: the int8 form of npu_weight_quant_batchmatmul used
// by the reference's dense projections (DenseW8, fnx/engine.py:297-384).
//
//   y[m, n] = bf16( sum_k x[m, k] * q[k, n] * S[k / gs, n] ),  fp32 accumulation
//
// q int8 [K, N] (row k holds the N columns), S bf16 [K/gs, N], x bf16 [M, K].
//
// One row, and up to four where the MFMA forms do not take the shape: split-K
// GEMV. A workgroup owns 256 columns (16 chunks of 16 bytes)
// and a K-slice of 16 L rows: thread (row-lane r = tid/16, chunk tid%16)
// loads its L rows of 16 columns at once (L = 4, 8 or 16, the most that
// keeps >= 512 workgroups in the grid and a run inside one scale group). A byte is read as offset binary u = q + 128
// (one xor per word) and converted by v_cvt_f32_ubyte; x * u is exact in
// fp32, and the accumulator starts at -128 * sum(x) so it ends at
// sum(x * q). A thread's 4 rows lie in one scale group, so it applies S once.
// Row-lanes are summed in LDS in row-lane order, the K-slices by the last
// workgroup to arrive, in slice order: deterministic run to run.
//
// Few rows or few tiles: bf16 MFMA (16x16x32), K split over a workgroup's
// waves, weights streamed into registers.
// Else: the same MFMA on 128 x 128 output tiles (128 x 64 for groups that are
// not whole 64-k chunks), the operands streaming through an LDS ring of chunks. int8 values are exact in bf16, so the MFMA sums
// x * q exactly per product with fp32 accumulation; after each scale group
// the group's partial sums are scaled by S[g, n] and added to the output
// accumulators.
#include "qmoe_common.h"
#include "qmoe.h"

namespace {

constexpr int kThreads = 256;
constexpr int kChunks = 16;                  // 16-byte chunks per tile row (256 columns)
constexpr int kTileCols = kChunks * 16;      // 256
constexpr int kRowLanes = kThreads / kChunks;  // 16
constexpr int kMaxL = 16;                    // largest rows per thread
constexpr int kRedStride = 17;               // LDS floats per (row-lane, chunk): 16 + 1 pad

template <int MR, int kL>
__global__ __launch_bounds__(kThreads) void w8a16_gemv_kernel(const uint16_t* __restrict__ x,
                                                              const int8_t* __restrict__ w,
                                                              const uint16_t* __restrict__ s,
                                                              uint16_t* __restrict__ y, int M, int K, int N, int gs,
                                                              float* __restrict__ part, int* __restrict__ counters) {
  __shared__ float red[kRowLanes * kChunks * kRedStride];
  __shared__ float res[MR][kTileCols];
  const int tile = blockIdx.x, slice = blockIdx.y, nslices = gridDim.y;
  const int tid = threadIdx.x;
  const int cc = tid % kChunks, r = tid / kChunks;
  const int col0 = tile * kTileCols + cc * 16;
  constexpr int kSlice = kRowLanes * kL;
  const int kr = slice * kSlice + r * kL;
  const bool active = col0 < N && kr < K;

  float acc[MR][16];
  if (active) {
    uint4 wv[kL];
#pragma unroll
    for (int i = 0; i < kL; ++i) wv[i] = load_nt16(w + (size_t)(kr + i) * N + col0);
    const uint4* sp = reinterpret_cast<const uint4*>(s + (size_t)(kr / gs) * N + col0);
    const uint4 s0 = sp[0], s1 = sp[1];
    float xv[MR][kL], sx[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      sx[m] = 0.f;
#pragma unroll
      for (int i = 0; i < kL; ++i) {
        xv[m][i] = m < M ? bf16_to_f32(x[(size_t)m * K + kr + i]) : 0.f;
        sx[m] += xv[m][i];
      }
#pragma unroll
      for (int c = 0; c < 16; ++c) acc[m][c] = -128.f * sx[m];
    }
#pragma unroll
    for (int i = 0; i < kL; ++i) {
      const uint32_t wd[4] = {wv[i].x ^ 0x80808080u, wv[i].y ^ 0x80808080u, wv[i].z ^ 0x80808080u,
                              wv[i].w ^ 0x80808080u};
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        const float u = (float)((wd[c >> 2] >> (8 * (c & 3))) & 0xffu);
#pragma unroll
        for (int m = 0; m < MR; ++m) acc[m][c] = __builtin_fmaf(xv[m][i], u, acc[m][c]);
      }
    }
    const uint32_t sw[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const float sc = bf16_to_f32((c & 1) ? (sw[c >> 1] >> 16) : (sw[c >> 1] & 0xffffu));
#pragma unroll
      for (int m = 0; m < MR; ++m) acc[m][c] *= sc;
    }
  } else {
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
      for (int c = 0; c < 16; ++c) acc[m][c] = 0.f;
  }

  // row-lane sums in LDS, one x row at a time; column tid of the tile
#pragma unroll
  for (int m = 0; m < MR; ++m) {
    float* dst = red + (r * kChunks + cc) * kRedStride;
#pragma unroll
    for (int c = 0; c < 16; ++c) dst[c] = acc[m][c];
    __syncthreads();
    const float* src = red + (tid / 16) * kRedStride + (tid & 15);
    float sum = 0.f;
#pragma unroll
    for (int rr = 0; rr < kRowLanes; ++rr) sum += src[rr * kChunks * kRedStride];
    res[m][tid] = sum;
    __syncthreads();
  }

  const int col = tile * kTileCols + tid;
  if (nslices == 1) {
    if (col < N)
      for (int m = 0; m < M; ++m) y[(size_t)m * N + col] = (uint16_t)f32_to_bf16(res[m][tid]);
    return;
  }
  float* mypart = part + (size_t)slice * MR * N;
  if (col < N)
    for (int m = 0; m < M; ++m) store_agent(&mypart[(size_t)m * N + col], res[m][tid]);
  if (!arrive_last(counters + tile, nslices)) return;
  if (col >= N) return;
  for (int m = 0; m < M; ++m) {
    const float sum = sum_agent_ordered(&part[(size_t)m * N + col], (size_t)MR * N, nslices);
    y[(size_t)m * N + col] = (uint16_t)f32_to_bf16(sum);
  }
}

// ---------------------------------------------------------------- many tiles, other groups: LDS ring
//
// bf16 MFMA 16x16x32 on 128 x 64 output tiles per workgroup of 4 waves (2 x 2,
// each 64 x 32: 4 x 2 MFMA tiles). K runs in 32-k chunks (one MFMA step) that
// stream into a ring of four LDS slots by
// buffer-resource global->LDS DMA, three chunks ahead: the x rows (16-byte
// pieces of a row stored XOR-swizzled by row, so the 16 rows a fragment
// read touches fall in different banks), the raw int8 weight rows [32][64]
// (row k in row slot k ^ ((k / 4) % 4), so the four rows a
// conversion read touches fall in different banks) and the bf16 scale row of
// the chunk's group. One chunk ahead of the MFMAs
// every thread converts a 4 k x 2 block of that chunk's weights to bf16
// (exact: |q| <= 128 has at most 8 significant bits) into one of two
// transposed buffers [column][k] (rows padded by 4 elements), so a lane's B
// fragment (8 consecutive k of one column) is two 8-byte reads; one barrier
// per chunk orders it all. Every LDS layout here keeps the lanes of one
// access in different banks. The MFMAs of one scale
// group sum into group accumulators; at the group's end those are scaled by
// S[g, n] with one fp32 fma into the output accumulators and cleared.

typedef __bf16 bf16x8_v __attribute__((ext_vector_type(8)));
typedef float f32x4_v __attribute__((ext_vector_type(4)));

constexpr int kBK = 32;                     // k per MFMA step

// four bf16 results as one 8-byte store (y rows may start at any element)
typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));
QMOE_DEV void store_bf16x4(uint16_t* p, uint32_t lo, uint32_t hi) { *reinterpret_cast<u32x2_a2*>(p) = u32x2_a2{lo, hi}; }

QMOE_DEV uint32_t i8_to_bf16_bits(uint32_t word, int byte) {
  return __float_as_uint((float)(int)(int8_t)(word >> (8 * byte))) >> 16;
}

// An 8-byte LDS write the compiler does not track. It cannot tell which LDS
// bytes an in-flight global->LDS DMA writes, so before an ordinary LDS store
// it would wait for every outstanding DMA (the chunks prefetched ahead too);
// used only for the converted weights, which no DMA touches.
QMOE_DEV void lds_write8_untracked(void* p, uint32_t lo, uint32_t hi) {
  const unsigned a = (unsigned)(size_t)(__attribute__((address_space(3))) char*)p;
  asm volatile("ds_write_b64 %0, %1" ::"v"(a), "v"(make_uint2(lo, hi)) : "memory");
}

// An 8-byte LDS read the compiler does not track (an ordinary one would wait for
// the DMAs in flight); waits for its own result.
QMOE_DEV uint2 lds_read8_untracked(const void* p) {
  const unsigned a = (unsigned)(size_t)(__attribute__((address_space(3))) const char*)p;
  uint2 v;
  asm volatile("ds_read_b64 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(a) : "memory");
  return v;
}

// The two weight fragments of a chunk (16 columns apart), each read from the
// converted rows as two 8-byte halves, in one
// block that waits for its own reads. An ordinary LDS load here would make
// the compiler wait for every global->LDS DMA in flight (the chunk just issued
// included), since it cannot tell which LDS bytes a DMA writes; no DMA writes
// the converted buffers.
QMOE_DEV void lds_read_frags2(const void* p0, const void* p1, uint4& f0, uint4& f1) {
  auto a = [](const void* p) { return (unsigned)(size_t)(__attribute__((address_space(3))) const char*)p; };
  asm volatile(
      "ds_read2_b64 %0, %2 offset1:1\n\t"
      "ds_read2_b64 %1, %3 offset1:1\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(f0), "=&v"(f1)
      : "v"(a(p0)), "v"(a(p1))
      : "memory");
}

template <int V>
struct W8C {
  static constexpr int value = V;
};

struct W8Ring {
  static constexpr int BM = 128, BN = 64, KC = kBK, RING = 4;
  static constexpr int TI = BM / 32, TJ = BN / 32;      // MFMA tiles per wave
  static constexpr int PPR = KC / 8;                    // 16-byte pieces per x row and chunk
  static constexpr int A_BYTES = BM * 2 * KC;           // x rows of one chunk
  static constexpr int B_BYTES = KC * BN;               // raw int8 weight rows of one chunk
  static constexpr int S_BYTES = BN * 2;                // bf16 scale row of the chunk's group
  static constexpr int SLOT = A_BYTES + B_BYTES + S_BYTES;
  static constexpr int AQ = A_BYTES / 1024 / 4;         // A DMA instructions per wave and chunk
  static constexpr int BQ = B_BYTES / 1024;             // B DMA instructions per chunk (waves past them repeat the last one)
  static constexpr int IPC = AQ + 1 + 1;                // DMA instructions per wave and chunk: x, weights, scales
  static constexpr int CG = kThreads / (KC / 4);        // converting threads' column groups (k-row groups of 4)
  static constexpr int CPT = BN / CG;                   // weight columns per converting thread
  static constexpr int RPS = 256 / BN;                  // raw weight rows per sweep of the 64 LDS banks
  static constexpr int LDK = KC + 4;                    // bf16 per row of the converted weights (8-byte aligned)
  static constexpr int CONV = 2 * BN * LDK * 2;         // two converted weight buffers
  static constexpr int LDS = RING * SLOT + CONV;
  static_assert(CPT == 2 && BQ <= 4, "a converting thread reads two bytes per row, a wave at most 1 KB of weights");
};

__global__ __launch_bounds__(kThreads) void w8a16_mfma_kernel(const uint16_t* __restrict__ x,
                                                              const int8_t* __restrict__ w,
                                                              const uint16_t* __restrict__ s,
                                                              uint16_t* __restrict__ y, int M, int K, int N, int gs) {
  using T = W8Ring;
  constexpr int BM = T::BM, BN = T::BN, KC = T::KC, RING = T::RING;
  constexpr int TI = T::TI, TJ = T::TJ, CPT = T::CPT, PPR = T::PPR, LDK = T::LDK;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  uint16_t* sbc = reinterpret_cast<uint16_t*>(lds + RING * T::SLOT);  // [2][BN][LDK]
  const int ntn = (N + BN - 1) / BN;
  const int ntiles = ((M + BM - 1) / BM) * ntn;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  if (tile >= ntiles) return;
  const int m0 = (tile / ntn) * BM, n0 = (tile % ntn) * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const int wm = wave >> 1, wn = wave & 1;
  const int i16 = lane & 15, kb = lane >> 4;
  // piece swizzle of x row r: the 16 rows of a fragment read spread over the banks
  auto swz = [](int r) { return (r >> 2) & 3; };

  // ---- DMA sources. A instruction q of wave w: rows (64 / PPR) (4q + w) +
  // lane / PPR, LDS piece lane % PPR of the row holding k-piece
  // (lane % PPR) ^ swz(row). B: wave w takes 1 KB of the raw [KC][BN] chunk,
  // lane l at byte 16 l. Scales: lane l < BN / 32 of wave w fetches 8 columns
  // at w BN / 4 + 8 l of the chunk's group row. Buffer resources bound every
  // access to its tensor; the per-lane offsets are fixed and a wave-uniform
  // offset advances per chunk.
  constexpr int kRsrcWord3 = 0x00020000;
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void*)x, (short)0, M * K * 2, kRsrcWord3);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void*)w, (short)0, K * N, kRsrcWord3);
  const __amdgpu_buffer_rsrc_t rsrc_s =
      __builtin_amdgcn_make_buffer_rsrc((void*)s, (short)0, (K / gs) * N * 2, kRsrcWord3);
  uint32_t aoff[T::AQ];
#pragma unroll
  for (int q = 0; q < T::AQ; ++q) {
    const int r = (64 / PPR) * (4 * q + wave) + lane / PPR;
    const int piece = (lane % PPR) ^ swz(r);
    aoff[q] = 2u * ((uint32_t)min(m0 + r, M - 1) * (uint32_t)K + 8u * (uint32_t)piece);
  }
  // raw weight row k sits in LDS row slot k ^ ((k / 4) % RPS) (an involution):
  // the four rows a converting thread reads at once are then in different banks
  auto row_slot = [](int k) { return k ^ ((k >> 2) & (T::RPS - 1)); };
  const int bblock = min(wave_u, T::BQ - 1), bbyte = 1024 * bblock + 16 * lane;
  const uint32_t boff = (uint32_t)row_slot(bbyte / BN) * (uint32_t)N + (uint32_t)(n0 + bbyte % BN);
  const uint32_t soff = 2u * (uint32_t)(n0 + wave * (BN / 4) + 8 * (lane & (BN / 32 - 1)));
  auto issue_chunk = [&](int c, int slot) {
    unsigned char* base = lds + slot * T::SLOT;
    const int k0 = c * KC;
#pragma unroll
    for (int q = 0; q < T::AQ; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (__attribute__((address_space(3))) void*)(base + (4 * q + wave_u) * 1024),
                                               16, (int)aoff[q], k0 * 2, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rsrc_b, (__attribute__((address_space(3))) void*)(base + T::A_BYTES + bblock * 1024), 16, (int)boff, k0 * N, 0, 0);
    if (lane < BN / 32)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_s,
                                               (__attribute__((address_space(3))) void*)(base + T::A_BYTES + T::B_BYTES + wave_u * (BN / 2)),
                                               16, (int)soff, (k0 / gs) * N * 2, 0, 0);
  };
  // ---- conversion of chunk c's raw weights into converted buffer c % 2:
  // thread t takes k rows 4 (t / CG) .. + 3 of columns CPT (t % CG) .. + CPT - 1
  // (row 4 kg + r from its slot)
  const int kg = tid / T::CG, cg = tid % T::CG;
  int rawoff[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) rawoff[r] = row_slot(4 * kg + r) * BN + CPT * cg;
  // the raw weight bytes a thread converts (convert_load), then their bf16
  // rows written to converted buffer buf (convert_store)
  auto convert_load = [&](int slot, uint32_t (&rw)[4]) {
    const unsigned char* raw = lds + slot * T::SLOT + T::A_BYTES;
#pragma unroll
    for (int r = 0; r < 4; ++r) rw[r] = (uint32_t)*reinterpret_cast<const uint16_t*>(raw + rawoff[r]);
  };
  auto convert_store = [&](int buf, const uint32_t (&rw)[4]) {
    uint16_t* dst = sbc + buf * BN * LDK + (CPT * cg) * LDK + 4 * kg;
#pragma unroll
    for (int cc = 0; cc < CPT; ++cc) {
      const uint32_t lo = i8_to_bf16_bits(rw[0], cc) | (i8_to_bf16_bits(rw[1], cc) << 16);
      const uint32_t hi = i8_to_bf16_bits(rw[2], cc) | (i8_to_bf16_bits(rw[3], cc) << 16);
      lds_write8_untracked(dst + cc * LDK, lo, hi);
    }
  };

  f32x4_v acc[TI][TJ], accg[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = accg[i][j] = f32x4_v{0.f, 0.f, 0.f, 0.f};
  int col[TJ];
#pragma unroll
  for (int j = 0; j < TJ; ++j) col[j] = n0 + wn * (BN / 2) + j * 16 + i16;
  // A fragment rows of this lane (tile i: row wm BM/2 + 16 i + i16)
  int arow[TI];
#pragma unroll
  for (int i = 0; i < TI; ++i) arow[i] = wm * (BM / 2) + 16 * i + i16;

  const int nch = K / KC, cpg = gs / KC;
  // ---- prologue: chunks 0 .. RING - 2 in flight, chunk 0 converted
#pragma unroll
  for (int c = 0; c < RING - 1; ++c)
    if (c < nch) issue_chunk(c, c);
  if (nch >= RING - 1) wait_vm_lgkm0<(RING - 2) * T::IPC>();
  else __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  {
    uint32_t rw[4];
    convert_load(0, rw);
    convert_store(0, rw);
  }

  // one chunk: ring slot SL = c % RING and converted buffer BU = c % 2 are
  // compile-time constants (the loop below is unrolled over RING chunks), so
  // every LDS address is an immediate offset; FIRST: c starts a
  // scale group, whose first MFMAs take a zero accumulator instead of the
  // group sums being cleared after each group
  auto chunk = [&](auto sl_c, auto bu_c, auto first_c, int c) {
    constexpr int SL = decltype(sl_c)::value, BU = decltype(bu_c)::value;
    constexpr bool FIRST = decltype(first_c)::value != 0;
    // chunk c + 1 has landed once only the later chunks in flight may be
    // pending; this chunk's converted rows (LDS stores) are complete
    if (c + 1 < nch) {
      if (c + RING - 2 < nch) wait_vm_lgkm0<(RING - 3) * T::IPC>();
      else __builtin_amdgcn_s_waitcnt(0);
    } else {
      wait_vm_lgkm0<63>();
    }
    // every wave is past chunk c - 1: its ring slot and converted buffer are
    // free. No fence: it would also wait for the chunks prefetched ahead.
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (c + RING - 1 < nch) issue_chunk(c + RING - 1, (SL + RING - 1) % RING);
    // Every LDS read of the chunk goes out together: the raw bytes of chunk
    // c + 1 to convert, the weight and activation fragments and, at
    // the end of a scale group, the group's scale row.
    const bool convert_next = c + 1 < nch;
    const bool group_end = (c + 1) % cpg == 0;
    uint32_t rw[4];
    if (convert_next) convert_load((SL + 1) % RING, rw);
    const unsigned char* as = lds + SL * T::SLOT;
    bf16x8_v bf[TJ], af[TI];
#pragma unroll
    for (int i = 0; i < TI; ++i) {
      const int r = arow[i];
      af[i] = *reinterpret_cast<const bf16x8_v*>(as + r * (2 * KC) + ((kb ^ swz(r)) << 4));
    }
    {
      // weight fragments (converted rows are 8-byte aligned)
      static_assert(TJ == 2, "two weight fragments per wave");
      const uint16_t* bs = sbc + BU * BN * LDK + (wn * (BN / 2) + i16) * LDK + kb * 8;
      uint4 f0, f1;
      lds_read_frags2(bs, bs + 16 * LDK, f0, f1);
      bf[0] = __builtin_bit_cast(bf16x8_v, f0);
      bf[1] = __builtin_bit_cast(bf16x8_v, f1);
    }
    float sc[TJ];
    if (group_end) {
      // the group's scale row came with this chunk
      const uint16_t* srow = reinterpret_cast<const uint16_t*>(as + T::A_BYTES + T::B_BYTES);
#pragma unroll
      for (int j = 0; j < TJ; ++j) sc[j] = col[j] < N ? bf16_to_f32(srow[wn * (BN / 2) + j * 16 + i16]) : 0.f;
    }
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j)
        accg[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bf[j], FIRST ? f32x4_v{0.f, 0.f, 0.f, 0.f} : accg[i][j],
                                                             0, 0, 0);
    if (convert_next) convert_store(1 - BU, rw);
    if (group_end) {
      // end of scale group: acc += S[g, col] * group sums
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[i][j][r] = __builtin_fmaf(accg[i][j][r], sc[j], acc[i][j][r]);
    }
  };
  auto chunk_at = [&](auto sl_c, auto bu_c, int c) {
    if (c % cpg == 0) chunk(sl_c, bu_c, W8C<1>{}, c);
    else chunk(sl_c, bu_c, W8C<0>{}, c);
  };
  static_assert(RING % 2 == 0, "ring slot and converted buffer repeat together");
  auto unrolled = [&](auto self, auto j_c, int c) {
    constexpr int J = decltype(j_c)::value;
    if constexpr (J < RING) {
      if (c + J < nch) {
        chunk_at(W8C<J>{}, W8C<J % 2>{}, c + J);
        self(self, W8C<J + 1>{}, c);
      }
    }
  };
  for (int c = 0; c < nch; c += RING) unrolled(unrolled, W8C<0>{}, c);
  // D layout: lane holds column i16 of tile (i, j) for rows 4 kb .. 4 kb + 3
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      if (col[j] >= N) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm * (BM / 2) + i * 16 + 4 * kb + r;
        if (row < M) y[(size_t)row * N + col[j]] = (uint16_t)f32_to_bf16(acc[i][j][r]);
      }
    }
}

// ---------------------------------------------------------------- few tiles: K split over the waves
//
// 16 LIVE rows of x (LIVE MFMA row tiles) times 16 F columns per workgroup. The
// NW waves split K (contiguous runs of 32-k steps) and stream their weights
// straight into registers in MFMA B-fragment order: lane (i16, kb) reads, for
// each of its 8 k rows 32 s + 8 kb + i, one 4-byte word, and a byte position of
// the eight words is the B fragment of that column. F = 4: word i16, all four
// columns (64-byte row pieces); F = 2: word i16 % 8, columns 2 (i16 / 8) and
// the next (32-byte pieces, the words read twice from the L1). int8 -> bf16
// (exact) is one conversion per value and one v_perm per pair; a scale group's
// MFMA sums are scaled by S[g, n] in fp32 as in the tiled kernel. U steps are
// loaded as one batch while the previous batch is computed. The waves' partial
// tiles meet in LDS and are summed in wave order: no second launch, counters
// or partials in memory, and the same bits every run.
//
// What bounds it: not HBM (2048 x 8192 at 7 rows: 7.9 us for 17 MB) but the
// workgroup's own chain: launch and first load about 4 us, then ~66 VALU and 10
// load instructions per step and wave, four waves per SIMD. So the grid takes
// few rows and columns per workgroup while it still fits the CUs at once.
// Against the 64 x 64 tiles (one chain over all of K per workgroup) it replaces
// here: 33.5 -> 7.9 us at 7 rows, 33.9 -> 13.2 at 64 (2048 x 8192), 34.0 -> 7.3
// at 7 rows, 34.1 -> 13.7 at 512 (2048 x 2048). Nontemporal weight loads lose
// (11.6 us): the two halves of a 128-byte line are read by two workgroups of one
// XCD and the second then misses.
template <int LIVE, int NW, int U, int F>
__global__ __launch_bounds__(64 * NW) void w8a16_skinny_kernel(const uint16_t* __restrict__ x,
                                                               const int8_t* __restrict__ w,
                                                               const uint16_t* __restrict__ s,
                                                               uint16_t* __restrict__ y, int M, int K, int N, int gs) {
  constexpr int BN = 16 * F, ROWS = 16 * LIVE;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  float* red = reinterpret_cast<float*>(lds);  // [NW][ROWS][BN]
  const int nrg = (M + ROWS - 1) / ROWS;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  if (tile >= nrg * ((N + BN - 1) / BN)) return;
  const int m0 = (tile % nrg) * ROWS, n0 = (tile / nrg) * BN;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i16 = lane & 15, kb = lane >> 4;
  const int nsteps = K / kBK, spg = gs / kBK;  // steps per scale group
  const int per = (nsteps + NW - 1) / NW;
  const int s0 = min(nsteps, wave * per), s1 = min(nsteps, s0 + per);
  // columns past N read column 0 (never stored), rows past M the last row
  const int cl = F == 4 ? 4 * i16 : 4 * (i16 & 7);  // the lane's word: tile columns cl .. cl + 3
  const int lc = F == 4 ? cl : cl + 2 * (i16 >> 3);  // its first column: lc .. lc + F - 1
  const int c0 = n0 + cl < N ? n0 + cl : 0;
  // buffer resources: per-lane offsets fixed for the whole loop, a scalar
  // offset per step, every access bounded by its tensor
  constexpr int kRsrcWord3 = 0x00020000;
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void*)x, (short)0, M * K * 2, kRsrcWord3);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void*)w, (short)0, K * N, kRsrcWord3);
  const __amdgpu_buffer_rsrc_t rsrc_s =
      __builtin_amdgcn_make_buffer_rsrc((void*)s, (short)0, (K / gs) * N * 2, kRsrcWord3);
  const int boff = 8 * kb * N + c0;
  const int sh = 16 * (i16 >> 3);  // F = 2: this lane's half of the word
  int aoff[LIVE];
#pragma unroll
  for (int t = 0; t < LIVE; ++t) aoff[t] = 2 * (min(m0 + 16 * t + i16, M - 1) * K + 8 * kb);

  f32x4_v acc[LIVE][F], accg[LIVE][F];
#pragma unroll
  for (int t = 0; t < LIVE; ++t)
#pragma unroll
    for (int f = 0; f < F; ++f) acc[t][f] = accg[t][f] = f32x4_v{0.f, 0.f, 0.f, 0.f};

  struct Block {
    uint32_t b[U][8];
    uint4 a[U][LIVE];
    uint2 sc[U];
  };
  // the load position: a step, its scale group's row and the group's steps
  // left (counted, not divided); steps past the wave's last re-read it (their
  // results are not used)
  int lq = s0, lrow = 0, lleft = 0, cleft = 0;
  auto load_block = [&](Block& v) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        v.b[u][i] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rsrc_b, boff, (lq * kBK + i) * N, 0);
#pragma unroll
      for (int t = 0; t < LIVE; ++t)
        v.a[u][t] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, aoff[t], lq * kBK * 2, 0));
      v.sc[u] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rsrc_s, 2 * c0, lrow, 0));
      if (lq + 1 < s1) {
        ++lq;
        if (--lleft == 0) {
          lleft = spg;
          lrow += 2 * N;
        }
      }
    }
  };
  auto compute = [&](int st, const Block& v) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = st + u;
      if (q >= s1) break;
      uint32_t b[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) b[i] = F == 4 ? v.b[u][i] : v.b[u][i] >> sh;
#pragma unroll
      for (int f = 0; f < F; ++f) {
        uint32_t p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float lo = (float)(int)(int8_t)(b[2 * i] >> (8 * f));
          const float hi = (float)(int)(int8_t)(b[2 * i + 1] >> (8 * f));
          p[i] = __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
        }
        const bf16x8_v bf = __builtin_bit_cast(bf16x8_v, make_uint4(p[0], p[1], p[2], p[3]));
#pragma unroll
        for (int t = 0; t < LIVE; ++t)
          accg[t][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_v, v.a[u][t]), bf, accg[t][f], 0, 0, 0);
      }
      if (--cleft == 0 || q + 1 == s1) {
        cleft = spg;
        const uint32_t s01 = (F == 4 || i16 < 8) ? v.sc[u].x : v.sc[u].y;
        const float sc[4] = {bf16_to_f32(s01 & 0xffffu), bf16_to_f32(s01 >> 16), bf16_to_f32(v.sc[u].y & 0xffffu),
                             bf16_to_f32(v.sc[u].y >> 16)};
#pragma unroll
        for (int t = 0; t < LIVE; ++t)
#pragma unroll
          for (int f = 0; f < F; ++f) {
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[t][f][r] = __builtin_fmaf(accg[t][f][r], sc[f], acc[t][f][r]);
            accg[t][f] = f32x4_v{0.f, 0.f, 0.f, 0.f};
          }
      }
    }
  };
  if (s0 < s1) {
    const int g0 = s0 / spg;
    lrow = g0 * N * 2;
    lleft = cleft = spg - (s0 - g0 * spg);
    Block v0, v1;
    load_block(v0);
    for (int st = s0; st < s1; st += 2 * U) {
      if (st + U < s1) load_block(v1);
      compute(st, v0);
      if (st + 2 * U < s1) load_block(v0);
      if (st + U < s1) compute(st + U, v1);
    }
  }
  // lane holds, for each row tile, rows 4 kb + r of its F columns
#pragma unroll
  for (int t = 0; t < LIVE; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float* dst = red + ((size_t)wave * ROWS + 16 * t + 4 * kb + r) * BN + lc;
      if constexpr (F == 4) *reinterpret_cast<float4*>(dst) = make_float4(acc[t][0][r], acc[t][1][r], acc[t][2][r], acc[t][3][r]);
      else *reinterpret_cast<float2*>(dst) = make_float2(acc[t][0][r], acc[t][1][r]);
    }
  __syncthreads();
  for (int p = tid; p < min(ROWS, M - m0) * BN / 4; p += 64 * NW) {
    const int row = p / (BN / 4), c = 4 * (p % (BN / 4));
    float4 a = *reinterpret_cast<const float4*>(red + row * BN + c);
#pragma unroll
    for (int q = 1; q < NW; ++q) {
      const float4 b = *reinterpret_cast<const float4*>(red + ((size_t)q * ROWS + row) * BN + c);
      a.x += b.x;
      a.y += b.y;
      a.z += b.z;
      a.w += b.w;
    }
    if (n0 + c < N)
      store_bf16x4(y + (size_t)(m0 + row) * N + n0 + c, f32_to_bf16(a.x) | (f32_to_bf16(a.y) << 16),
                   f32_to_bf16(a.z) | (f32_to_bf16(a.w) << 16));
  }
}

template <int LIVE, int NW, int U, int F>
int launch_w8_skinny(const void* x, const void* w, const void* scale, void* y, int M, int K, int N, int gs,
                     hipStream_t stream) {
  constexpr int kLds = NW * 16 * LIVE * 16 * F * 4;
  int dev = 0;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return (int)err;
  if (dev < 0 || dev >= 64) return QMOE_EINVAL;
  static bool attr_set[64] = {};
  if (!attr_set[dev]) {
    err = hipFuncSetAttribute((const void*)w8a16_skinny_kernel<LIVE, NW, U, F>, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (err != hipSuccess) return (int)err;
    attr_set[dev] = true;
  }
  const long tiles = (long)host_ceil_div(M, 16 * LIVE) * host_ceil_div(N, 16 * F);
  const long blocks = (tiles + 7) / 8 * 8;  // whole XCD rounds (extra blocks exit)
  if (blocks > 0x7fffffffL) return QMOE_EINVAL;
  hipLaunchKernelGGL((w8a16_skinny_kernel<LIVE, NW, U, F>), dim3((unsigned)blocks), dim3(64 * NW), kLds, stream,
                     (const uint16_t*)x, (const int8_t*)w, (const uint16_t*)scale, (uint16_t*)y, M, K, N, gs);
  return (int)hipGetLastError();
}

bool w8_mfma_ok(const void* x, const void* w, int M, int K, int N, int gs) {
  return M >= 1 && K >= kBK && K % kBK == 0 && N >= 16 && N % 16 == 0 && gs >= kBK && gs % kBK == 0 && K % gs == 0 &&
         ((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0 && (long)M * K * 2 < 0x80000000L &&
         (long)K * N < 0x80000000L;
}

// The skinny kernel's tile: the fewest row tiles per workgroup whose grid
// still runs at once (a workgroup's 8 or 16 waves take a CU), 32-column tiles
// where those fit the 256 CUs as well.
// Few rows and many workgroups win because each workgroup's conversions and x
// reads, not HBM, set its time: at K = 2048 one, two, three and four row tiles
// take 7.9, 10.0, 11.6 and 13.2 us with 32 columns, 8.3, 10.6, 11.8 and 13.7
// with 64, whatever N is (2048 or 8192).
int launch_w8_few_tiles(const void* x, const void* w, const void* scale, void* y, int M, int K, int N, int gs,
                        hipStream_t st) {
  constexpr long kCus = 256;
  auto groups = [&](int live) { return (long)host_ceil_div(M, 16 * live); };
  int live = 1;
  while (live < 4 && groups(live) * host_ceil_div(N, 64) > kCus) ++live;
  live = host_ceil_div(M, 16 * (int)groups(live));  // no emptier than needed
  if (groups(live) * host_ceil_div(N, 32) <= kCus) {
    if (live == 1) return launch_w8_skinny<1, 16, 1, 2>(x, w, scale, y, M, K, N, gs, st);
    if (live == 2) return launch_w8_skinny<2, 16, 2, 2>(x, w, scale, y, M, K, N, gs, st);
    if (live == 3) return launch_w8_skinny<3, 8, 2, 2>(x, w, scale, y, M, K, N, gs, st);
    return launch_w8_skinny<4, 8, 2, 2>(x, w, scale, y, M, K, N, gs, st);
  }
  if (live == 1) return launch_w8_skinny<1, 16, 2, 4>(x, w, scale, y, M, K, N, gs, st);
  if (live == 2) return launch_w8_skinny<2, 16, 1, 4>(x, w, scale, y, M, K, N, gs, st);
  if (live == 3) return launch_w8_skinny<3, 8, 1, 4>(x, w, scale, y, M, K, N, gs, st);
  return launch_w8_skinny<4, 8, 1, 4>(x, w, scale, y, M, K, N, gs, st);
}

// ---------------------------------------------------------------- many tiles, 64-k groups: conversion in registers
//
// 128 x 128 output tiles, 4 waves (2 x 2) of 64 x 64: 4 x 4 MFMA tiles each. K
// runs in 64-k chunks (x rows and raw int8 weight rows, with the bf16 scale row
// of the chunk's group) through a ring of three LDS slots by buffer-resource
// global->LDS DMA, two chunks ahead; one barrier per chunk. A lane reads, for
// each of its 8 k rows of a step, the 4 bytes of its columns 4 i16 .. 4 i16 + 3,
// and makes the four B fragments of the step itself: one conversion per value
// and one v_perm per pair (int8 is exact in bf16), between the MFMAs of the
// fragment before. So the weights are neither written back to LDS nor read a
// second time, and no conversion stands in the chunk's chain.
// LDS: x row r holds k-piece p at p ^ (r & 7); weight row r sits at r ^ 1 for
// odd r / 8 and its words at w ^ 16 for odd r / 16, so the four 16-word pieces a
// wave reads at once lie in different banks.
//
// What bounds it: VALU and MFMA issue. With one wave per SIMD a chunk costs the
// wave about 100 conversion and 32 scaling operations at 5 cycles each beside 512
// cycles of MFMA; issued in blocks rather than behind the MFMAs, with the seven
// DMA instructions together (350 cycles) and the chunk's LDS reads ahead of it
// (415), it took 2130. 2048 x 8192 at 512 rows 39.1 -> 24.5 us (700 TFLOP/s), at
// 1024 73.0 -> 40.6 (847), 4096 x 4096 at 4096 rows 273 -> 176 (781), against 128
// x 64 tiles that converted through LDS. A deeper ring changes nothing (4 and 6
// slots: 31.2 and 31.9 us where 3 took 30.6).
struct W8Reg {
  static constexpr int BM = 128, BN = 128, KC = 64, RING = 3;
  static constexpr int A_BYTES = BM * KC * 2, B_BYTES = KC * BN, S_BYTES = 1024;  // scales: one DMA instruction, 256 bytes used
  static constexpr int SLOT = A_BYTES + B_BYTES + S_BYTES;
  static constexpr int IPC = 4 + 2 + 1;  // DMA instructions per wave and chunk: x, weights, scales
  static constexpr int LDS = RING * SLOT;
};

template <int KS, int CPG>
__global__ __launch_bounds__(kThreads * KS, 2) void w8a16_reg_kernel(const uint16_t* __restrict__ x,
                                                                const int8_t* __restrict__ w,
                                                                const uint16_t* __restrict__ s,
                                                                uint16_t* __restrict__ y, int M, int K, int N, int gs) {
  using T = W8Reg;
  constexpr int RING = T::RING;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int ntn = (N + T::BN - 1) / T::BN;
  const int ntiles = ((M + T::BM - 1) / T::BM) * ntn;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  if (tile >= ntiles) return;
  const int nrt = ntiles / ntn;  // row tiles of a column tile side by side on one XCD: its weights come through one L2
  const int m0 = (tile % nrt) * T::BM, n0 = (tile / nrt) * T::BN;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6) & 3);
  const int ks = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / kThreads);
  unsigned char* ring = lds + ks * T::LDS;
  const int wm = wave >> 1, wn = wave & 1;
  const int i16 = lane & 15, kb = lane >> 4;

  constexpr int kRsrcWord3 = 0x00020000;
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void*)x, (short)0, M * K * 2, kRsrcWord3);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void*)w, (short)0, K * N, kRsrcWord3);
  const __amdgpu_buffer_rsrc_t rsrc_s =
      __builtin_amdgcn_make_buffer_rsrc((void*)s, (short)0, (K / gs) * N * 2, kRsrcWord3);
  // this wave group's run of chunks: whole scale groups of cpg chunks, the same number for each
  const int cpg = CPG != 0 ? CPG : gs / T::KC;
  const int nch = K / T::KC / KS, c0 = ks * nch;
  uint32_t aoff[4], boff[2];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = 8 * (4 * q + wave) + (lane >> 3);
    aoff[q] = 2u * ((uint32_t)min(m0 + r, M - 1) * (uint32_t)K + 8u * (uint32_t)((lane & 7) ^ (r & 7)));
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int b = 4 * q + wave;  // 8 weight rows
    boff[q] = (uint32_t)(8 * b + ((lane >> 3) ^ (b & 1))) * (uint32_t)N +
              (uint32_t)(n0 + 16 * ((lane & 7) ^ (4 * ((b >> 1) & 1))));
  }
  // scales: every wave writes the same row; lanes past it read beyond the
  // resource's extent, which gives zeros and no traffic
  const uint32_t soff = lane < 16 ? 2u * (uint32_t)(n0 + 8 * lane) : 0x80000000u;
  // DMA instruction j of a chunk: 0, 1 weights, 2 .. 5 x, 6 scales
  // (srow: byte offset of the scale row of the chunk's group)
  auto issue_one = [&](int j, int c, int slot, int srow) {
    unsigned char* base = ring + slot * T::SLOT;
    const int k0 = (c0 + c) * T::KC;
    if (j < 2) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc_b, (__attribute__((address_space(3))) void*)(base + T::A_BYTES + (4 * j + wave) * 1024), 16, (int)boff[j],
          k0 * N, 0, 0);
    } else if (j < 6) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc_a, (__attribute__((address_space(3))) void*)(base + (4 * (j - 2) + wave) * 1024), 16, (int)aoff[j - 2],
          k0 * 2, 0, 0);
    } else {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_s, (__attribute__((address_space(3))) void*)(base + T::A_BYTES + T::B_BYTES),
                                               16, (int)soff, srow, 0, 0);
    }
  };

  f32x4_v acc[4][4], accg[4][4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int f = 0; f < 4; ++f) acc[t][f] = f32x4_v{0.f, 0.f, 0.f, 0.f};
  // this lane's LDS offsets: x row i16 of row tile 0 (its pieces by step), its
  // word of even and odd weight rows
  const int arow = (wm * 64 + i16) * 128;
  const int bword = 4 * ((16 * wn + i16) ^ (16 * (kb >> 1))) + 8 * kb * 128;
  const int beven = T::A_BYTES + bword + (kb & 1) * 128, bodd = T::A_BYTES + bword - (kb & 1) * 128;

#pragma unroll
  for (int c = 0; c < RING - 1; ++c)
    {
      const int cc = min(c, nch - 1);
#pragma unroll
      for (int j = 0; j < T::IPC; ++j) issue_one(j, cc, c, (c0 + cc) * T::KC / gs * N * 2);
    }
  // the current ring slot; the chunk DMA'd next (the run's last one again past
  // its end, into a slot that is not read any more), its scale row and its
  // group's chunks left, counted
  int slot = 0, inext = min(RING - 1, nch - 1);
  int irow = (c0 + inext) * T::KC / gs * N * 2, ileft = cpg - (c0 + inext) % cpg;
  // one chunk; FIRST / LAST: it starts / ends a run of group sums
  auto chunk = [&](auto first_c, auto last_c) {
    constexpr bool FIRST = decltype(first_c)::value != 0, LAST = decltype(last_c)::value != 0;
    wait_vm_lgkm0<(RING - 2) * T::IPC>();
    // every wave is past the chunk before: its slot takes the chunk RING - 1 ahead
    barrier_no_fence();
    const unsigned char* base = ring + slot * T::SLOT;
    uint32_t bw[2][8];
    bf16x8_v af[2][4];
    auto read_words = [&](int st) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        bw[st][i] = *reinterpret_cast<const uint32_t*>(base + ((i & 1) ? bodd : beven) + (32 * st + i) * 128);
    };
    auto read_x = [&](int st, int t) {
      af[st][t] = *reinterpret_cast<const bf16x8_v*>(base + arow + t * 16 * 128 + (((4 * st + kb) ^ (i16 & 7)) << 4));
    };
    // pair i of fragment n (step n / 4, column n % 4)
    auto pair = [&](int n, int i) -> uint32_t {
      const float lo = (float)(int)(int8_t)(bw[n >> 2][2 * i] >> (8 * (n & 3)));
      const float hi = (float)(int)(int8_t)(bw[n >> 2][2 * i + 1] >> (8 * (n & 3)));
      return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
    };
    read_words(0);
#pragma unroll
    for (int t = 0; t < 4; ++t) read_x(0, t);
    __builtin_amdgcn_sched_barrier(0);
    uint32_t cur[4], nxt[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) cur[i] = pair(0, i);
    __builtin_amdgcn_sched_barrier(0);
    // Behind each MFMA, in its shadow: a pair of the next fragment (three VALU
    // operations), step 1's reads behind step 0's first fragment, one DMA
    // instruction of the chunk to come per fragment (issued together they held
    // the wave for 350 cycles) and, in a group's last chunk, the scaled sums of
    // the columns that are complete. sched_barrier keeps this order.
    uint2 sv{};
    float sc = 0.f;
    auto scaled = [&](int f, int t) {
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[t][f][r] = __builtin_fmaf(accg[t][f][r], sc, acc[t][f][r]);
    };
    auto scale_of = [&](int f) {
      const uint32_t v = f < 2 ? sv.x : sv.y;
      return __uint_as_float((f & 1) ? (v & 0xffff0000u) : (v << 16));
    };
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      const bf16x8_v b = __builtin_bit_cast(bf16x8_v, make_uint4(cur[0], cur[1], cur[2], cur[3]));
      if (LAST && n >= 5) sc = scale_of(n - 5);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        accg[t][n & 3] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            af[n >> 2][t], b, (FIRST && n < 4) ? f32x4_v{0.f, 0.f, 0.f, 0.f} : accg[t][n & 3], 0, 0, 0);
        if (n < 7) nxt[t] = pair(n + 1, t);
        if (n == 0 && t == 0) read_words(1);
        if (n == 0 && t > 1) {
          read_x(1, 2 * t - 4);
          read_x(1, 2 * t - 3);
        }
        if (n < 7 && t == 3) issue_one(n, inext, slot == 0 ? RING - 1 : slot - 1, irow);
        if (LAST && n >= 5) scaled(n - 5, t);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (LAST && n == 3) sv = lds_read8_untracked(base + T::A_BYTES + T::B_BYTES + 2 * (64 * wn + 4 * i16));
#pragma unroll
      for (int i = 0; i < 4; ++i) cur[i] = nxt[i];
    }
    if (LAST) {
      sc = scale_of(3);
#pragma unroll
      for (int t = 0; t < 4; ++t) scaled(3, t);
    }
  };
  auto next_chunk = [&]() {
    slot = slot + 1 == RING ? 0 : slot + 1;
    if (inext + 1 < nch) {
      ++inext;
      if (--ileft == 0) {
        ileft = cpg;
        irow += 2 * N;
      }
    }
  };
  for (int c = 0; c < nch; c += cpg) {
    if constexpr (CPG == 1) {
      chunk(W8C<1>{}, W8C<1>{});
      next_chunk();
    } else {
      chunk(W8C<1>{}, W8C<0>{});
      next_chunk();
      if constexpr (CPG == 0) {
        for (int i = 2; i < cpg; ++i) {
          chunk(W8C<0>{}, W8C<0>{});
          next_chunk();
        }
      }
      chunk(W8C<0>{}, W8C<1>{});
      next_chunk();
    }
  }
  __builtin_amdgcn_s_waitcnt(0);  // the DMA past the end
  if constexpr (KS > 1) {
    // the second group's tile through LDS
    float4* part = reinterpret_cast<float4*>(lds);  // [4][4][256 threads]
    const int gt = threadIdx.x % kThreads;
    __syncthreads();
    if (ks > 0) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int f = 0; f < 4; ++f)
          part[(4 * t + f) * kThreads + gt] = make_float4(acc[t][f][0], acc[t][f][1], acc[t][f][2], acc[t][f][3]);
    }
    __syncthreads();
    if (ks > 0) return;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const float4 v = part[(4 * t + f) * kThreads + gt];
        acc[t][f] += f32x4_v{v.x, v.y, v.z, v.w};
      }
  }
  // lane holds columns 4 i16 .. + 3 for rows 4 kb .. + 3 of each row tile
  const int col = n0 + 64 * wn + 4 * i16;
  if (col >= N) return;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = m0 + 64 * wm + 16 * t + 4 * kb + r;
      if (row < M)
        store_bf16x4(y + (size_t)row * N + col, pk_bf16(acc[t][0][r], acc[t][1][r]), pk_bf16(acc[t][2][r], acc[t][3][r]));
    }
}

template <int KS, int CPG>
int launch_w8_reg(const void* x, const void* w, const void* scale, void* y, int M, int K, int N, int gs, hipStream_t st) {
  int dev = 0;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return (int)err;
  if (dev < 0 || dev >= 64) return QMOE_EINVAL;
  static bool attr_set[64] = {};
  if (!attr_set[dev]) {
    err = hipFuncSetAttribute((const void*)w8a16_reg_kernel<KS, CPG>, hipFuncAttributeMaxDynamicSharedMemorySize, KS * W8Reg::LDS);
    if (err != hipSuccess) return (int)err;
    attr_set[dev] = true;
  }
  const long blocks = ((long)host_ceil_div(M, W8Reg::BM) * host_ceil_div(N, W8Reg::BN) + 7) / 8 * 8;
  if (blocks > 0x7fffffffL) return QMOE_EINVAL;
  hipLaunchKernelGGL((w8a16_reg_kernel<KS, CPG>), dim3((unsigned)blocks), dim3(kThreads * KS), KS * W8Reg::LDS, st, (const uint16_t*)x,
                     (const int8_t*)w, (const uint16_t*)scale, (uint16_t*)y, M, K, N, gs);
  return (int)hipGetLastError();
}

int launch_w8_mfma(const void* x, const void* w, const void* scale, void* y, int M, int K, int N, int gs,
                   hipStream_t stream) {
  using T = W8Ring;
  int dev = 0;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return (int)err;
  if (dev < 0 || dev >= 64) return QMOE_EINVAL;
  static bool attr_set[64] = {};
  if (!attr_set[dev]) {
    err = hipFuncSetAttribute((const void*)w8a16_mfma_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, T::LDS);
    if (err != hipSuccess) return (int)err;
    attr_set[dev] = true;
  }
  const long tiles = (long)((M + T::BM - 1) / T::BM) * ((N + T::BN - 1) / T::BN);
  const long blocks = (tiles + 7) / 8 * 8;  // whole XCD rounds (extra blocks exit)
  if (blocks > 0x7fffffffL) return QMOE_EINVAL;
  hipLaunchKernelGGL(w8a16_mfma_kernel, dim3((unsigned)blocks), dim3(kThreads), T::LDS, stream,
                     (const uint16_t*)x, (const int8_t*)w, (const uint16_t*)scale, (uint16_t*)y, M, K, N, gs);
  return (int)hipGetLastError();
}

}  // namespace

extern "C" {

// Rows per thread for a shape: the largest L in {16, 8, 4} (up to kMaxL)
// that divides gs and still leaves >= 256 workgroups, one per CU (or is 4).
// With the weights read nontemporally the longer rows won: 2048 x 8192
// took 9.0 us with L = 16 (256 workgroups) against 9.9 with L = 8 (512).
static int w8_rows_per_thread(int K, int N, int gs) {
  for (int L = kMaxL; L > 4; L >>= 1)
    if (gs % L == 0 && (long)host_ceil_div(N, kTileCols) * host_ceil_div(K, kRowLanes * L) >= 256) return L;
  return 4;
}

size_t qmoe_w8a16_gemv_workspace(int M, int K, int N) {
  (void)M;
  return (size_t)host_ceil_div(K, kRowLanes * 4) * 4 * (size_t)N * sizeof(float);
}

int qmoe_w8a16_gemv_counters(int N) { return host_ceil_div(N, kTileCols); }

int qmoe_w8a16_gemv(const void* x, const void* w, const void* scale, void* y, int M, int K, int N, int group_size,
                    void* workspace, size_t workspace_bytes, void* counters, void* stream) {
  if (M < 1 || M > 4 || K < 4 || (K % 4) || N < 16 || (N % 16) || group_size < 4 || (group_size % 4) ||
      (K % group_size) || host_ceil_div(N, kTileCols) >= QMOE_DECODE_MAILBOX_BASE - 1)
    return QMOE_EINVAL;
  const int L = w8_rows_per_thread(K, N, group_size);
  const int nslices = host_ceil_div(K, kRowLanes * L);
  if (nslices > 1 && workspace_bytes < qmoe_w8a16_gemv_workspace(M, K, N)) return QMOE_EWORKSPACE;
  // Two to four rows: the skinny MFMA kernel where it takes the shape (its waves
  // share K, so it needs no second reduction through memory): 8.3 against 11.7
  // to 16.5 us (2048 x 8192), 10.5 against 19.2 (three rows, 4096 x 512). One
  // row stays here: from cold weights 9.0 us against 9.75 (2048 x 8192).
  if (M > 1 && w8_mfma_ok(x, w, M, K, N, group_size))
    return launch_w8_few_tiles(x, w, scale, y, M, K, N, group_size, (hipStream_t)stream);
  dim3 grid(host_ceil_div(N, kTileCols), nslices);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(kThreads), 0, (hipStream_t)stream, (const uint16_t*)x, (const int8_t*)w,
                       (const uint16_t*)scale, (uint16_t*)y, M, K, N, group_size, (float*)workspace,
                       (int*)counters);
  };
#define QMOE_W8_L(L_)                                                   \
  if (L == L_) {                                                        \
    if (M == 1) go(w8a16_gemv_kernel<1, L_>);                           \
    else if (M == 2) go(w8a16_gemv_kernel<2, L_>);                      \
    else go(w8a16_gemv_kernel<4, L_>);                                  \
    return (int)hipGetLastError();                                      \
  }
  QMOE_W8_L(16) QMOE_W8_L(8) QMOE_W8_L(4)
#undef QMOE_W8_L
  return QMOE_EINVAL;
}

int qmoe_w8a16_gemm_mfma(const void* x, const void* w, const void* scale, void* y, int M, int K, int N,
                         int group_size, void* stream) {
  if (!w8_mfma_ok(x, w, M, K, N, group_size)) return QMOE_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  // Groups of whole 64-k chunks: 128 x 128 tiles from 128 of them on. At 2048 x
  // 8192 they take 23.1 us for 256 rows and the skinny kernel 29.4 from cold
  // weights; with 64 tiles 22.4 against 15.2 (512 rows, 2048 x 2048). Up to one
  // tile per CU K is split over two groups of waves where both get whole scale
  // groups (4096 x 4096 at 512 rows 42.5 against 53.4 us); beyond, two workgroups
  // share a CU instead (2048 x 8192 at 1024 rows 40.6 against 45.8).
  const long tiles = (long)host_ceil_div(M, 128) * host_ceil_div(N, 128);
  if (group_size % 64 == 0) {
    if (tiles < 128) return launch_w8_few_tiles(x, w, scale, y, M, K, N, group_size, st);
    auto go = [&](auto ks) {
      constexpr int KS = decltype(ks)::value;
      if (group_size == 64) return launch_w8_reg<KS, 1>(x, w, scale, y, M, K, N, group_size, st);
      if (group_size == 128) return launch_w8_reg<KS, 2>(x, w, scale, y, M, K, N, group_size, st);
      return launch_w8_reg<KS, 0>(x, w, scale, y, M, K, N, group_size, st);
    };
    return tiles <= 256 && K / group_size % 2 == 0 ? go(W8C<2>{}) : go(W8C<1>{});
  }
  // other groups: 128 x 64 tiles of 32-k chunks above 256 rows where they give
  // every CU a workgroup
  if (M <= 256 || (long)host_ceil_div(M, 128) * host_ceil_div(N, 64) < 256)
    return launch_w8_few_tiles(x, w, scale, y, M, K, N, group_size, st);
  return launch_w8_mfma(x, w, scale, y, M, K, N, group_size, st);
}

}  // extern "C"
