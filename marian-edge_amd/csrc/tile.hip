// tile.hip — LDS-tiled int8 MFMA GEMM for many rows (v_mfma_i32_32x32x32_i8).
//
// Operands and epilogue are those of gemm.hip: activations A[M, K] and weights
// W[N, K], both K-contiguous, exact i32 accumulators, y = acc * (1/(a_m w_n)) +
// b_n with optional ReLU, i32 copy and statically quantized copy.
#include "device_common.h"
#include "kernels.h"
#include <algorithm>
#include <type_traits>

namespace mh {
namespace {

typedef int v16i __attribute__((ext_vector_type(16)));

// ---------------------------------------------------------------------------
// One workgroup of WM x WN waves per BM x BN output tile, each wave a grid of
// 32x32 MFMA blocks.  K moves in 128-byte chunks: registers hold the next PF
// chunks (requested that far ahead, across tile boundaries too: a workgroup
// walks several tiles, so the next tile's first chunks arrive while this
// tile's results are dequantized and stored), LDS two, one barrier per chunk.
//
// LDS rows are 128 bytes, the 16-byte piece p of row r at slot p ^ (r % 8), so
// that both the stores (eight lanes per row) and the MFMA operand reads (32
// rows, one piece each) touch every bank equally.
//
// Lane l of an output block holds column l % 32 and rows 8(r/4) + 4(l/32) +
// r%4 (register r): a store instruction writes two whole 128-byte lines
// straight from the accumulators, with no pass through LDS.
//
// Tile order: workgroups reach the 8 XCDs round-robin; each XCD takes a
// contiguous range of tiles.  Wide outputs go in groups of kTileGroup row
// tiles (row tile fastest), so a weight tile reaches an XCD's L2 once per
// group; narrow ones column tile fastest, so activations are shared.
//
// What bounds it (4096 x 32000, K = 512, 256x128 tiles, one workgroup per CU):
// 134 us against 236 us for the 64x64 tiles it replaces, which divided in the
// epilogue and staged every result through LDS.  The epilogue with its stores
// alone takes 105 us (5.0 TB/s of output), the K loop alone under 90 us; the
// rest is what the two do not overlap.  At 1459 x 512 (K = 512) a tile's
// memory round trip and the dispatch are 5.1 us (6.3 before).
// ---------------------------------------------------------------------------
constexpr int kTileKC = 128;     // bytes of K per chunk
constexpr int kTileGroup = 8;    // row tiles per group
constexpr int kTileWideN = 32;   // column tiles above which tiles go in groups

// Output rows [0, rows) of a tile as a raw buffer: stores at or past its end
// are dropped.
constexpr int kRawBufferWord3 = 0x00020000;  // gfx9 raw buffer: 32-bit data format, no swizzle
constexpr int kNt = 2;                       // non-temporal: the outputs are not read again here
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rows(const void* p, int64_t elem0, int64_t ld, int rows,
                                                            int size) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)p + elem0 * size), (short)0, (int)(rows * ld * size),
                                           kRawBufferWord3);
}

// One output (fp32, the int32 accumulators or the int8 codes) of one wave's
// blocks of a tile: rows row0 + 32 i, columns ncol.  r: the tile's output rows,
// whose range ends with the last one, so that rows past M are dropped; a lane
// past N starts past the range.  A pass per output keeps one running offset per
// column block: with all outputs' offsets and branches in one loop the 128x128
// tile spilled 85 registers (4096 x 2304, K = 512, fp32 and int32: 57.2 us, now 22.7).
enum TileOut { TO_F32, TO_I32, TO_Q };
template <TileOut OUT, int AUX, bool RELU, int MB, int NB>
__device__ __forceinline__ void tile_pass(__amdgpu_buffer_rsrc_t r, int64_t ld, const GemmArgs& g,
                                          const v16i (&acc)[MB][NB], const float* sm, const float (&wm)[NB],
                                          const float (&bi)[NB], bool ok, uint32_t row0, const int (&ncol)[NB],
                                          float qmult, int rows, bool& bad) {
  constexpr uint32_t size = OUT == TO_Q ? 1 : 4;
  const uint32_t ldb = (uint32_t)ld * size;
  uint32_t off[NB];
#pragma unroll
  for (int k = 0; k < NB; ++k) off[k] = ncol[k] < g.N ? row0 * ldb + (uint32_t)ncol[k] * size : 0x80000000u;
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float inv[4][NB];
      if constexpr (OUT != TO_I32) {
        const float4 a4 = *(const float4*)(sm + i * 32 + 8 * q);
        const float av[4] = {a4.x, a4.y, a4.z, a4.w};
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int k = 0; k < NB; ++k) inv[t][k] = recip_exact(av[t] * wm[k]);
        if (!ok) {  // a multiplier outside recip_exact's range: the IEEE quotient
#pragma unroll
          for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int k = 0; k < NB; ++k) inv[t][k] = dequant_scale(av[t], wm[k]);
        }
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int k = 0; k < NB; ++k) {
          const int32_t iv = acc[i][k][4 * q + t];
          if constexpr (OUT == TO_I32) {
            __builtin_amdgcn_raw_buffer_store_b32((uint32_t)iv, r, off[k], 0, AUX);
          } else {
            float y = dequant_apply(iv, inv[t][k], bi[k]);
            if (RELU) y = y > 0.0f ? y : 0.0f;
            if constexpr (OUT == TO_F32) {
              __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y), r, off[k], 0, AUX);
            } else {
              __builtin_amdgcn_raw_buffer_store_b8((uint8_t)(int8_t)quantize_one(y, qmult), r, off[k], 0, AUX);
              bad |= ncol[k] < g.N && (int)row0 + i * 32 + 8 * q + t < rows && !isfinite(y);
            }
          }
          off[k] += (t == 3 ? 5u : 1u) * ldb;  // rows 0-3, 8-11, 16-19, 24-27 of each block
        }
    }
}

// Dequantizes and stores one wave's blocks of a tile at (m0, n0): rows wr +
// 32 i, columns wc + 32 k.  sAm: the tile's row multipliers in LDS; ok: this
// lane's share of them has exponents in recip_exact's range.
// stream: the fp32 and int32 stores are non-temporal.
template <int BM, int MB, int NB, bool RELU, bool EXTRA, bool WIDE>
__device__ __forceinline__ void tile_store(const GemmArgs& g, const Epilogue& e, const v16i (&acc)[MB][NB],
                                           const float* sAm, const float (&wm)[NB], const float (&bi)[NB], bool ok,
                                           int m0, int n0, int wr, int wc, bool stream) {
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
#pragma unroll
  for (int k = 0; k < NB; ++k) ok &= recip_factor(wm[k]);
  ok = __all(ok);
  const float* sm = sAm + wr + 4 * half;
  const int rows = min(BM, g.M - m0);
  const uint32_t row0 = (uint32_t)(wr + 4 * half);
  bool bad = false;
  int ncol[NB];
#pragma unroll
  for (int k = 0; k < NB; ++k) ncol[k] = n0 + wc + k * 32 + (lane & 31);
  if constexpr (WIDE) {  // row strides past the buffer offsets
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t m = m0 + (int64_t)row0 + i * 32 + 8 * (r >> 2) + (r & 3);
        const float am = sm[i * 32 + 8 * (r >> 2) + (r & 3)];
#pragma unroll
        for (int k = 0; k < NB; ++k) {
          const int32_t iv = acc[i][k][r];
          float y = dequant(iv, am, wm[k], bi[k]);
          if (RELU) y = y > 0.0f ? y : 0.0f;
          if (m < g.M && ncol[k] < g.N) {
            if (e.out) e.out[m * e.ldo + ncol[k]] = y;
            if (e.out_i32) e.out_i32[m * e.ldi + ncol[k]] = iv;
            if (e.out_q) e.out_q[m * e.ldq + ncol[k]] = (int8_t)quantize_one(y, e.qmult);
            bad |= !isfinite(y);
          }
        }
      }
  } else {
    auto pass = [&](auto out, const void* p, int64_t ld) {
      const __amdgpu_buffer_rsrc_t r = tile_rows(p, m0 * ld, ld, rows, 4);
      if (stream)
        tile_pass<out(), kNt, RELU>(r, ld, g, acc, sm, wm, bi, ok, row0, ncol, 0.0f, rows, bad);
      else
        tile_pass<out(), 0, RELU>(r, ld, g, acc, sm, wm, bi, ok, row0, ncol, 0.0f, rows, bad);
    };
    if (!EXTRA || e.out) pass(std::integral_constant<TileOut, TO_F32>(), e.out, e.ldo);
    if constexpr (EXTRA) {
      if (e.out_i32) pass(std::integral_constant<TileOut, TO_I32>(), e.out_i32, e.ldi);
      if (e.out_q)
        tile_pass<TO_Q, 0, RELU>(tile_rows(e.out_q, (int64_t)m0 * e.ldq, e.ldq, rows, 1), e.ldq, g, acc, sm, wm, bi, ok,
                                 row0, ncol, e.qmult, rows, bad);
    }
  }
  if constexpr (EXTRA) {
    if (e.out_q) {
      if (n0 == 0 && tid < rows) e.out_qa[m0 + tid] = e.qmult;
      if (__any(bad) && lane == 0 && g.err) *g.err = 1;  // quantizing rejects non-finite input
    }
  }
}

template <int BM, int BN, int WM, int WN, int PF, bool RELU, bool EXTRA, bool WIDE>
__global__ __launch_bounds__(WM * WN * 64) __attribute__((amdgpu_waves_per_eu(BM > 128 ? 2 : WM * WN / 2)))
void k_gemm_tile(GemmArgs g, Epilogue e, int tiles_n, int tiles, int stream) {
  constexpr int NT = WM * WN * 64;
  constexpr int MB = BM / WM / 32, NB = BN / WN / 32;  // 32x32 blocks per wave
  constexpr int AP = BM * 8 / NT, BP = BN * 8 / NT;    // 16-byte pieces per thread and chunk
  static_assert(AP * NT == BM * 8 && BP * NT == BN * 8 && PF % 2 == 0, "whole pieces, even ring");
  static_assert(NT >= BM, "a thread per row multiplier");
  __shared__ __attribute__((aligned(16))) int8_t sA[2][BM * kTileKC];
  __shared__ __attribute__((aligned(16))) int8_t sB[2][BN * kTileKC];
  __shared__ float sAm[2][BM];
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave / WN * (BM / WM), wc = wave % WN * (BN / WN);  // the wave's corner
  const int M = g.M, N = g.N, K = g.K;

  // This workgroup's tiles: lo + slot, + per_xcd, ... below hi.
  const int xcd = blockIdx.x & 7, per_xcd = (gridDim.x + 7) >> 3;
  const int hi = (int)((int64_t)(xcd + 1) * tiles >> 3);
  const int first = (int)((int64_t)xcd * tiles >> 3) + (blockIdx.x >> 3);
  if (first >= hi) return;  // the whole workgroup
  auto corner = [&](int tile, int& m0, int& n0) {
    if (tiles_n > kTileWideN) {
      const int tiles_m = (M + BM - 1) / BM;
      const int grp = tile / (kTileGroup * tiles_n), first_m = grp * kTileGroup;
      const int gm = min(kTileGroup, tiles_m - first_m), in_g = tile - grp * kTileGroup * tiles_n;
      m0 = (first_m + in_g % gm) * BM;
      n0 = in_g / gm * BN;
    } else {
      m0 = tile / tiles_n * BM;
      n0 = tile % tiles_n * BN;
    }
  };

  // The loader runs PF chunks ahead and is branch-free: past a tile's last
  // chunk it goes on with the next tile (the last tile again at the end), rows
  // past M or N reload the last one (their results are not stored) and pieces
  // past K reload the row's last piece; A's are zeroed at the LDS store.  A
  // tile counts a multiple of PF chunks, so a chunk's registers and LDS buffer
  // are fixed at compile time.
  const int nslot = (K + kTileKC * PF - 1) / (kTileKC * PF) * PF;
  v4i ra[PF][AP], rb[PF][BP];
  const int8_t *pa[AP], *pb[BP];
  const int kp = (tid & 7) * 16;  // this thread's piece of each chunk
  auto point = [&](int m0, int n0) {
#pragma unroll
    for (int i = 0; i < AP; ++i) pa[i] = g.A + (int64_t)min(m0 + ((tid + i * NT) >> 3), M - 1) * g.lda;
#pragma unroll
    for (int i = 0; i < BP; ++i) pb[i] = g.W + (int64_t)min(n0 + ((tid + i * NT) >> 3), N - 1) * K;
  };
  auto gload = [&](int c, v4i (&xa)[AP], v4i (&xb)[BP]) {
    const int col = min(c * kTileKC + kp, K - 16);
#pragma unroll
    for (int i = 0; i < AP; ++i) xa[i] = *(const v4i*)(pa[i] + col);
#pragma unroll
    for (int i = 0; i < BP; ++i) xb[i] = *(const v4i*)(pb[i] + col);
  };
  int m0, n0;
  corner(first, m0, n0);
  point(m0, n0);
#pragma unroll
  for (int u = 0; u < PF; ++u) gload(u, ra[u], rb[u]);

  int tpar = 0;
  for (int tile = first; tile < hi; tile += per_xcd, tpar ^= 1) {
    int m1 = m0, n1 = n0;  // the next tile's corner
    v16i acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int k = 0; k < NB; ++k)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][k][r] = 0;
    // The tile's row multipliers (into LDS with its chunks) and this lane's
    // column operands: both arrive under the products.
    const float am = g.a[min(m0 + min(tid, BM - 1), M - 1)];
    float wm[NB], bi[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int n = min(n0 + wc + k * 32 + (lane & 31), N - 1);
      wm[k] = g.wmult[n];
      bi[k] = g.bias[n];
    }
    for (int c0 = 0; c0 < nslot; c0 += PF) {
      int cl = c0 + PF;  // the chunks to request
      if (cl == nslot) {
        if (tile + per_xcd < hi) corner(tile + per_xcd, m1, n1);
        point(m1, n1);
        cl = 0;
        if (tid < BM) sAm[tpar][tid] = am;
      }
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        const bool in_k = (c0 + u) * kTileKC + kp < K;
#pragma unroll
        for (int i = 0; i < AP; ++i) {
          const int c = tid + i * NT, row = c >> 3;
          *(v4i*)(sA[u & 1] + row * kTileKC + (((c & 7) ^ (row & 7)) << 4)) = keep_or_zero(ra[u][i], in_k);
        }
#pragma unroll
        for (int i = 0; i < BP; ++i) {
          const int c = tid + i * NT, row = c >> 3;
          *(v4i*)(sB[u & 1] + row * kTileKC + (((c & 7) ^ (row & 7)) << 4)) = rb[u][i];
        }
        gload(cl + u, ra[u], rb[u]);
        wg_lds_barrier();
        const int8_t* la = sA[u & 1] + (wr + (lane & 31)) * kTileKC;
        const int8_t* lb = sB[u & 1] + (wc + (lane & 31)) * kTileKC;
#pragma unroll
        for (int ks = 0; ks < kTileKC / 32; ++ks) {
          const int at = ((2 * ks + half) ^ (lane & 7)) << 4;
          v4i fa[MB], fb[NB];
#pragma unroll
          for (int i = 0; i < MB; ++i) fa[i] = *(const v4i*)(la + i * 32 * kTileKC + at);
#pragma unroll
          for (int k = 0; k < NB; ++k) fb[k] = *(const v4i*)(lb + k * 32 * kTileKC + at);
#pragma unroll
          for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int k = 0; k < NB; ++k)
              acc[i][k] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i], fb[k], acc[i][k], 0, 0, 0);
        }
      }
    }
    bool ok = true;
#pragma unroll
    for (int i = 0; i < BM; i += 64) ok &= recip_factor(sAm[tpar][i + lane]);
    tile_store<BM, MB, NB, RELU, EXTRA, WIDE>(g, e, acc, sAm[tpar], wm, bi, ok, m0, n0, wr, wc, stream);
    m0 = m1;
    n0 = n1;
  }
}

// ---------------------------------------------------------------------------
// The same product from fp32 rows: a workgroup quantizes its 64 rows itself
// (row multiplier 127 / max|x|, or the static one in g.act) into LDS for the
// whole K (at most 512), then streams the weights past them, so the layer is
// one launch.  Each row is quantized once per column tile, which costs less
// than the launch and the pass over memory it replaces while the shape is at
// most one round of workgroups (gemm_f32_supported).  A serial chain of one
// tile bounds it: the rows' round trip, 1.3 us of quantizing (39 instructions
// a row and wave: a row on 16 lanes needs four lane moves for its maximum and
// shares one division, against 90 with a row per wave), the K loop, the
// stores.  1459 x 512, K = 512: 10.0 us a call in two launches, 7.4 in one.
// ---------------------------------------------------------------------------
constexpr int kF32MaxK = 512;
constexpr int kF32Rows = 64;

template <int BN, int WM, int WN, bool RELU, bool EXTRA>
__global__ __launch_bounds__(WM * WN * 64) void k_gemm_tile_f32(GemmArgs g, Epilogue e, int tiles_n, int tiles) {
  constexpr int BM = kF32Rows, NW = WM * WN, NT = NW * 64;
  constexpr int MB = BM / WM / 32, NB = BN / WN / 32, BP = BN * 8 / NT, PF = 2;
  __shared__ __attribute__((aligned(16))) int8_t sA[BM * kF32MaxK];  // [128-byte chunk][row][piece ^ row % 8]
  __shared__ __attribute__((aligned(16))) int8_t sB[2][BN * kTileKC];
  __shared__ float sAm[BM];
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave / WN * (BM / WM), wc = wave % WN * (BN / WN);
  const int M = g.M, N = g.N, K = g.K;
  const int xcd = blockIdx.x & 7;
  const int tile = (int)((int64_t)xcd * tiles >> 3) + (blockIdx.x >> 3);
  if (tile >= (int)((int64_t)(xcd + 1) * tiles >> 3)) return;  // the whole workgroup
  const int m0 = tile / tiles_n * BM, n0 = tile % tiles_n * BN;
  const int nslot = (K + 2 * kTileKC - 1) / (2 * kTileKC) * 2;  // 2 or 4 chunks

  const int8_t* pb[BP];
  v4i rb[PF][BP];
  const int kp = (tid & 7) * 16;
  auto gload = [&](int c, v4i (&xb)[BP]) {
    const int col = min(c * kTileKC + kp, K - 16);
#pragma unroll
    for (int i = 0; i < BP; ++i) xb[i] = *(const v4i*)(pb[i] + col);
  };
#pragma unroll
  for (int i = 0; i < BP; ++i) pb[i] = g.W + (int64_t)min(n0 + ((tid + i * NT) >> 3), N - 1) * K;

  // ---- the rows: a wave takes four at a time, 16 lanes each; lane l of them
  // holds columns 4l + 64j ----
  constexpr int RW = BM / NW, G = RW / 4;  // rows per wave, groups of four
  const int kj = K >> 6;                   // live j
  const int c4 = 4 * (lane & 15);
  float4 v[G][8];
#pragma unroll
  for (int t = 0; t < G; ++t) {
    const float* xr = g.Af + (int64_t)min(m0 + wave * RW + 4 * t + (lane >> 4), M - 1) * g.ldaf + c4;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[t][j] = *(const float4*)(xr + 64 * min(j, kj - 1));  // past K: the last again
  }
#pragma unroll
  for (int u = 0; u < PF; ++u) gload(u, rb[u]);  // the first weights arrive under the quantization
  bool bad = false;
#pragma unroll
  for (int t = 0; t < G; ++t) {
    const int row = wave * RW + 4 * t + (lane >> 4);
    float mx = 0.0f;
    bool nan = false;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float4 x = v[t][j];
      mx = fmaxf(fmaxf(mx, fmaxf(fabsf(x.x), fabsf(x.y))), fmaxf(fabsf(x.z), fabsf(x.w)));
      nan |= __builtin_isunordered(x.x, x.y) || __builtin_isunordered(x.z, x.w);
    }
    bad |= (nan || !(mx < INFINITY)) && m0 + row < M;
    mx = fmaxf(mx, __int_as_float(dpp_mov<0xB1>(__float_as_int(mx))));   // over the row's 16 lanes
    mx = fmaxf(mx, __int_as_float(dpp_mov<0x4E>(__float_as_int(mx))));
    mx = fmaxf(mx, __int_as_float(dpp_mov<0x124>(__float_as_int(mx))));
    mx = fmaxf(mx, __int_as_float(dpp_mov<0x128>(__float_as_int(mx))));
    const float a = g.act > 0.0f ? g.act : row_multiplier(mx);
    if ((lane & 15) == 0) sAm[row] = a;
    int8_t* ar = sA + row * kTileKC + (c4 & 15);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int c = c4 + 64 * j;
      if (j < 2 * nslot)  // uniform; a last chunk past K holds zeros
        *(uint32_t*)(ar + (j >> 1) * (BM * kTileKC) + ((((c >> 4) & 7) ^ (row & 7)) << 4)) =
            j < kj ? quantize_pack4(v[t][j], a) : 0u;
    }
  }
  if (__any(bad) && lane == 0 && g.err) *g.err = 1;

  // ---- the weights past them ----
  v16i acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int k = 0; k < NB; ++k)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][k][r] = 0;
  float wm[NB], bi[NB];
#pragma unroll
  for (int k = 0; k < NB; ++k) {
    const int n = min(n0 + wc + k * 32 + (lane & 31), N - 1);
    wm[k] = g.wmult[n];
    bi[k] = g.bias[n];
  }
  for (int c0 = 0; c0 < nslot; c0 += PF) {
#pragma unroll
    for (int u = 0; u < PF; ++u) {
#pragma unroll
      for (int i = 0; i < BP; ++i) {
        const int c = tid + i * NT, row = c >> 3;
        *(v4i*)(sB[u & 1] + row * kTileKC + (((c & 7) ^ (row & 7)) << 4)) = rb[u][i];
      }
      gload(c0 + PF + u, rb[u]);  // past K: the last pieces again, unused
      wg_lds_barrier();
      const int8_t* la = sA + (c0 + u) * (BM * kTileKC) + (wr + (lane & 31)) * kTileKC;
      const int8_t* lb = sB[u & 1] + (wc + (lane & 31)) * kTileKC;
#pragma unroll
      for (int ks = 0; ks < kTileKC / 32; ++ks) {
        const int at = ((2 * ks + half) ^ (lane & 7)) << 4;
        v4i fa[MB], fb[NB];
#pragma unroll
        for (int i = 0; i < MB; ++i) fa[i] = *(const v4i*)(la + i * 32 * kTileKC + at);
#pragma unroll
        for (int k = 0; k < NB; ++k) fb[k] = *(const v4i*)(lb + k * 32 * kTileKC + at);
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int k = 0; k < NB; ++k)
            acc[i][k] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i], fb[k], acc[i][k], 0, 0, 0);
      }
    }
  }
  tile_store<BM, MB, NB, RELU, EXTRA, false>(g, e, acc, sAm, wm, bi, recip_factor(sAm[lane]), m0, n0, wr, wc, true);
}

// Whether the outputs are stored past the caches.  Rows of whole 64-byte pieces
// are (16384 x 2304, K = 512: 41.1 us, 60.2 through the caches).  In other rows a
// store instruction ends inside a piece at either end, and streaming the parts
// costs more than leaving them to the caches to join, once the outputs exceed
// the L2s and as long as the last cache holds them beside the operands, or the
// products are few (us; streamed | not, before this kernel): 2200 x 2300, K 512
// 11.1 | 12.1, 13.3; 8192 x 2300, K 256 32.2 | 22.1, 26.7; 3000 x 8300, K 512 54.5 |
// 36.0, 46.7; 16384 x 1500, K 512 40.3 | 44.0, 44.7; 16384 x 1000, K 2048 54.0 | 59.6.
// With both outputs streaming never paid (4096 x 8300, K 512 153 | 99, 114).
bool tile_streams(const GemmArgs& g, const Epilogue& e) {
  const bool whole = ((e.out ? (uintptr_t)e.out | 4 * e.ldo : 0) | (e.out_i32 ? (uintptr_t)e.out_i32 | 4 * e.ldi : 0)) % 64 == 0;
  if (e.out && e.out_i32) return whole;
  const int64_t mb = (int64_t)g.M * g.N * 4 / 1000000;
  return whole || mb < 26 || (g.K > 256 && mb > (g.K > 512 ? 60 : (g.N > kTileWideN * 128 ? 128 : 88)));
}

template <int BM, int BN, int WM, int WN, int PF, bool WIDE = false>
hipError_t launch_tile(const GemmArgs& g, const Epilogue& e, int max_wgs, hipStream_t s) {
  const int64_t tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN, tiles = tiles_m * tiles_n;
  if (tiles > (int64_t)INT32_MAX / 2) return hipErrorInvalidValue;
  const int grid = (int)std::min<int64_t>((tiles + 7) / 8 * 8, max_wgs);
  const bool extra = WIDE || e.out_i32 || e.out_q || !e.out;
  auto kern = e.relu ? (extra ? k_gemm_tile<BM, BN, WM, WN, PF, true, true, WIDE> : k_gemm_tile<BM, BN, WM, WN, PF, true, WIDE, WIDE>)
                     : (extra ? k_gemm_tile<BM, BN, WM, WN, PF, false, true, WIDE> : k_gemm_tile<BM, BN, WM, WN, PF, false, WIDE, WIDE>);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(WM * WN * 64), 0, s, g, e, (int)tiles_n, (int)tiles,
                     (int)tile_streams(g, e));
  return hipGetLastError();
}

template <int BN, int WM, int WN>
hipError_t launch_tile_f32(const GemmArgs& g, const Epilogue& e, hipStream_t s) {
  const int64_t tiles_n = (g.N + BN - 1) / BN, tiles = (g.M + kF32Rows - 1) / kF32Rows * tiles_n;
  if (tiles > (1 << 30)) return hipErrorInvalidValue;
  const bool extra = e.out_i32 || e.out_q || !e.out;
  auto kern = e.relu ? (extra ? k_gemm_tile_f32<BN, WM, WN, true, true> : k_gemm_tile_f32<BN, WM, WN, true, false>)
                     : (extra ? k_gemm_tile_f32<BN, WM, WN, false, true> : k_gemm_tile_f32<BN, WM, WN, false, false>);
  hipLaunchKernelGGL(kern, dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(WM * WN * 64), 0, s, g, e, (int)tiles_n, (int)tiles);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_gemm_tile(const GemmArgs& g, const Epilogue& e, hipStream_t s) {
  if (g.K <= 0 || g.K % 64 || g.N <= 0 || g.M_dev || g.lda % 16) return hipErrorInvalidValue;
  if (e.out_q && (!e.out_qa || e.ldq < g.N || !(e.qmult > 0.0f) || !(e.qmult < __builtin_huge_valf())))
    return hipErrorInvalidValue;
  if (g.M <= 0) return hipSuccess;
  // Buffer offsets of a tile's rows stay below 2^30 (a lane past N starts at
  // 2^31, above every range); longer rows take 64-bit addresses.
  if (std::max(std::max(e.out ? e.ldo : 0, e.out_i32 ? e.ldi : 0), e.out_q ? e.ldq : 0) >= (1 << 20))
    return launch_tile<64, 64, 2, 2, 2, true>(g, e, 1024, s);
  // By the tiles a shape gives 256 CUs (kernel times in us, this kernel's
  // sizes in the order 64x64 / 128x128 / 256x128):
  //   below 224 128x128 tiles, one tile's latency decides and small tiles win:
  //     1459 x 512 (K 512) 5.1 / 6.9 / 9.3, 4096 x 512 (K 2048) 12.0 / 14.1 / 19.8;
  //   above, larger tiles read less per output: 7405 x 512 (K 2048) 17.8 / 14.4 /
  //     19.3, 1000 x 32000 44.9 / 34.0 / 36.9;
  //   past one round of 128x128 tiles their outputs count without the padding:
  //     12000 x 300 (K 2048; 282 tiles, 220 without) 20.0 / 24.4;
  //   from 2048 256x128 tiles (eight a CU) the largest: 4096 x 32000 175 / 157 / 134.
  // Both outputs make a barely started third round of 128x128 tiles (two a CU)
  // long, and 64x64 tiles win while their sums are short (us a call, 64x64 /
  // 128x128, the kernel before in brackets): 5504 x 1536 (K 512; 516 tiles) 17.3 /
  // 22.5 (20.5), 5600 x 2048 (704) 20.5 / 23.7 (24.1), 8000 x 2048 (K 640; 1008)
  // 34.1 / 33.8 (36.1), 5544 x 1536 (K 1024; 528) 22.5 / 26.6 (25.5), 11464 x 1000
  // (720) 32.0 / 28.9 (37.6), 16640 x 512 (K 2048; 520) 40.5 / 40.2 (42.2).
  // Where they go through the caches (rows that are not whole 64-byte pieces), the
  // largest tiles win as soon as the last cache cannot hold them, 256 MB or 2048
  // 128x128 tiles (128x128 / 256x128): 16384 x 2300 (K 512) 92.7 / 70.5 (108), 15072 x
  // 2500 (K 1024) 120 / 94.3 (114), 37680 x 1000 (K 640) 113 / 91.1 (89.9).
  const auto tiles = [&](int64_t bm, int64_t bn) { return ((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn); };
  if (tiles(256, 128) >= 2048) return launch_tile<256, 128, 4, 2, 2>(g, e, 256, s);
  if (e.out && e.out_i32 && tiles(128, 128) > 512 && tiles(128, 128) <= (g.K <= 640 ? 768 : 640) && g.K <= 1024)
    return launch_tile<64, 64, 2, 2, 2>(g, e, 1024, s);
  if (e.out && e.out_i32 && !tile_streams(g, e) && tiles(128, 128) >= 2048)
    return launch_tile<256, 128, 4, 2, 2>(g, e, 256, s);
  const bool one_round = tiles(128, 128) >= 224 && tiles(128, 128) <= 256;
  if (one_round || (int64_t)g.M * g.N >= 224 * 128 * 128) return launch_tile<128, 128, 2, 4, 2>(g, e, 1 << 30, s);
  return launch_tile<64, 64, 2, 2, 2>(g, e, 1024, s);
}

static int64_t f32_tiles(const GemmArgs& g, int bn) {
  return (int64_t)((g.M + kF32Rows - 1) / kF32Rows) * ((g.N + bn - 1) / bn);
}

bool gemm_f32_supported(const GemmArgs& g, const Epilogue& e) {
  const int64_t ld = std::max(std::max(e.out ? e.ldo : 0, e.out_i32 ? e.ldi : 0), e.out_q ? e.ldq : 0);
  // More than a round of 256-column tiles is faster quantized first, as one
  // pass: 2500 x 2048 (320 tiles) 15.4 us a call against 12.7 in two launches,
  // 7405 x 512 (232) 8.9 against 12.6.
  return g.Af && g.K <= kF32MaxK && g.ldaf % 4 == 0 && (uintptr_t)g.Af % 16 == 0 && ld < (1 << 20) &&
         f32_tiles(g, 256) <= 256;
}

hipError_t launch_gemm_f32(const GemmArgs& g, const Epilogue& e, hipStream_t s) {
  if (g.K <= 0 || g.K % 64 || g.N <= 0 || g.M_dev || !gemm_f32_supported(g, e)) return hipErrorInvalidValue;
  if (g.M <= 0) return hipSuccess;
  // One round of workgroups either way: 128 columns a tile while that fits the
  // 256 CUs (1459 x 512: 7.9 us, 8.5 with 256 columns), else 256 columns on 16
  // waves (1459 x 2048: 9.8 us, 11.0 with 128).
  return f32_tiles(g, 128) <= 256 ? launch_tile_f32<128, 2, 4>(g, e, s) : launch_tile_f32<256, 2, 8>(g, e, s);
}

}  // namespace mh
