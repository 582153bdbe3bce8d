// attnseq.hip — self-attention of packed sequences (ATT_SEQ): one workgroup of
// four waves per 64 (or 16) query rows of a (sequence, head), K and V staged in
// LDS in 64-key chunks, the products of both contractions from the matrix cores.
//
// The reference order (k_attention's, bit for bit): a score is a DH-term dot
// in dimension order from -0.0, each product and each sum rounded on its own;
// max, the C library's expf, the denominator folded in key order from 0.0,
// p = e * (1 / sum), and out_d = sum_k v_k[d] p_k in key order from 0.0.
//
// What bounds it and why this shape.  Separate roundings make every term a
// multiply and an add, and with lane = key each term also takes a lane's K (or
// V) value from LDS: the kernel this one replaced was bound by LDS reads.  Here
// one v_mfma_f32_16x16x1_4b_f32 with a +0.0 C operand forms the 16 x 64
// products of one dimension (scores) or one key (PV): each is a * b + 0 rounded
// once, the IEEE product (denormals included; compared with the host's on 16 M
// products of all kinds of operands), except that a product of -0.0 becomes
// +0.0.  That reaches no output: a zero score's sign leaves its exponential as
// it is, and a PV sum starts from +0.0, which either zero leaves unchanged.  A
// wave then holds 16 queries x 64 keys (scores) or 16 queries x DH dimensions
// (PV) in 16 registers, and LDS serves one 16-byte read per lane and operand
// for 64 sums per lane.  The bound is the issue of products and sums: 1024 terms
// cost a SIMD 64-68 cycles with three or four waves (108 with one; the 16 adds
// alone 36, the product alone 47, 32 separate multiplies and adds 68-91).
//
// Short sequences share a workgroup: with at most 32 (16) keys, two (four)
// heads' keys fill the 64 staged rows and each head takes two (one) waves.
// Score blocks past the last key are skipped in steps of 32 keys.
//
// A workgroup finds its (sequence, query tile, head) itself from the lengths
// (find_unit), the longest first; no tile list is built by a launch of its own.
// With more than kSeqFindMax sequences the lookup would cost more than the
// workgroups that find nothing to do, and the grid covers (sequence, head) x
// query tiles.
//
// Few rows leave most of the chip idle, and a unit then takes as long as one
// wave's steps: there a wave takes 4 queries (v_mfma_f32_4x4x1_16b_f32, 4 sums a
// step), a workgroup 16, and the grid covers (sequence, head) x query tiles.
//
// Measured (before -> now, us): 256 sentences, lengths lognormal(3.2, 0.6), 8
// heads of 64, fp32 (7405 rows): 59.6 -> 36; 48 segments of 96-256 rows, bf16
// (8800 rows): 196 -> 96; 54 sentences (1390 rows) 14.9 -> 11.9; one of 15 rows
// 7.6 -> 5.2; 24 sequences of 257-512 rows (9569; one wave per (row, head)
// before) 851 -> 216.
#include "device_common.h"
#include "kernels.h"

#include <algorithm>

namespace mh {
namespace {

// Four floats (bytes) of an output row, which only has its element's alignment.
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32u __attribute__((aligned(1)));

constexpr int kSeqWaves = 4;                   // waves per workgroup
// (row, head) pairs up to which a wave takes 4 queries instead of 16, by the
// scores a wave holds (sweep of 8 heads, us with 4 | 16 queries: sentences, 2867
// rows 20.1 | 22.6, 4393 24.8 | 24.6; segments of 96-256, 2241 rows 33.5 | 40.6,
// 3528 54.1 | 50.7, 4315 56.4 | 51.7; 257-512 keys, 1697 rows 58.2 | 70.2, 2388
// 75.7 | 80.6, 3073 85.8 | 78.1).
constexpr int64_t kSeqFewRows256 = 32768, kSeqFewRows512 = 20480;
// Workgroups up to which that holds, and workgroups per sequence past them:
// max_keys may be far above the lengths, and each 4096 that find nothing cost
// 1.6 us; with 16 queries the lengths decide, but finding a unit costs more the
// more sequences there are (us with 4 | 16: 300 of 8 rows, 9600 workgroups 15.2 |
// 14.9, 19200 19.0 | 14.9, 38400 27.1 | 15.0; 500 of 4 rows, 32000 25.6 | 21.1;
// 1024 of 4 rows, 8192 25.2 | 44.4, 32768 35.0 | 44.6, 131072 76.2 | 44.7; 128
// sentences, 16384 27.4 | 28.8).
constexpr int64_t kSeqFewGroups = 16384, kSeqFewGroupsPer = 48;
constexpr int kSeqFindMax = 1024;              // sequences up to which a workgroup finds its unit itself
constexpr int kSeqRow = kHeadDim + 4;          // padded LDS row (floats), 16-byte aligned

__constant__ uint64_t kSeqExp2Tab[32] = {MH_EXP2_TABLE_32};

// n rows of ld elements from p on, of which the last holds `width` elements, as
// a raw buffer resource: a load at or past its end returns zeros (the hardware
// range check on the VGPR offset), so one lane offset serves every row block
// and rows past the last need no mask.  It needs width <= ld and every offset
// below 2^32 bytes (seq_buffer_rows).
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
constexpr int kRawBufferWord3 = 0x00020000;  // gfx9 raw buffer: 32-bit data format, no swizzle
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_of(const T* p, int n, int64_t ld, int width) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)(uint32_t)(((n - 1) * ld + width) * sizeof(T)),
                                           kRawBufferWord3);
}
__device__ __forceinline__ u32x4 load4(__amdgpu_buffer_rsrc_t r, uint32_t off, float) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
}
__device__ __forceinline__ u32x2 load4(__amdgpu_buffer_rsrc_t r, uint32_t off, uint16_t) {
  return __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
}
__device__ __forceinline__ u32x4 floats4(u32x4 w) { return w; }
__device__ __forceinline__ u32x4 floats4(u32x2 w) {
  return u32x4{w.x << 16, w.x & 0xFFFF0000u, w.y << 16, w.y & 0xFFFF0000u};
}
__device__ __forceinline__ float load1(__amdgpu_buffer_rsrc_t r, uint32_t off, float) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
__device__ __forceinline__ float load1(__amdgpu_buffer_rsrc_t r, uint32_t off, uint16_t) {
  return bf16_to_f32(__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0));
}
// The same through a pointer with its element's alignment (general strides).
typedef u32x4 u32x4u __attribute__((aligned(4)));
typedef u32x2 u32x2u __attribute__((aligned(2)));
__device__ __forceinline__ u32x4 load4(const float* p) { return *(const u32x4u*)p; }
__device__ __forceinline__ u32x2 load4(const uint16_t* p) { return *(const u32x2u*)p; }
__device__ __forceinline__ float load1(const float* p) { return *p; }
__device__ __forceinline__ float load1(const uint16_t* p) { return bf16_to_f32(*p); }

// A wave's tile of QW queries x 64 keys (or dimensions): register 4b + r of
// lane l holds column l % QW and row 4 (64 / QW) b + 4 (l / QW) + r.
template <int QW>
using Tile = float __attribute__((ext_vector_type(QW)));

// Products of the lanes' values: row value a is lane row's, column value b
// lane l's is column l % QW's.
template <int QW>
__device__ __forceinline__ Tile<QW> products(float a, float b) {
  static_assert(QW == 16 || QW == 4, "matrix shapes");
  if constexpr (QW == 16)
    return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, Tile<16>{0}, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, Tile<4>{0}, 0, 0, 0);
}

// acc += p in the first N registers; the fence keeps each step's adds behind
// the next step's products, which run on the matrix cores meanwhile.
template <int N, int QW>
__device__ __forceinline__ void add_products(Tile<QW>& acc, const Tile<QW>& p) {
#pragma unroll
  for (int i = 0; i < N; ++i) acc[i] = acc[i] + p[i];
  __builtin_amdgcn_sched_barrier(0);
}

// Scores of one 64-key chunk (its first N registers) from -0.0 in dimension
// order: kr is the lane's key row, qr the row of query l % QW.
template <int N, int QW, int DH>
__device__ __forceinline__ Tile<QW> chunk_scores(const float* kr, const float* qr) {
  Tile<QW> acc;
#pragma unroll
  for (int i = 0; i < QW; ++i) acc[i] = -0.0f;
  float4 ka = *(const float4*)kr, qa = *(const float4*)qr;
  Tile<QW> p0 = products<QW>(ka.x, qa.x), p1;
#pragma unroll 1
  for (int i = 0; i < DH; i += 8) {
    const float4 kb = *(const float4*)(kr + i + 4), qb = *(const float4*)(qr + i + 4);
    p1 = products<QW>(ka.y, qa.y);
    add_products<N>(acc, p0);
    p0 = products<QW>(ka.z, qa.z);
    add_products<N>(acc, p1);
    p1 = products<QW>(ka.w, qa.w);
    add_products<N>(acc, p0);
    p0 = products<QW>(kb.x, qb.x);
    add_products<N>(acc, p1);
    const int nx = min(i + 8, DH - 4);  // past the end: re-read and unused
    ka = *(const float4*)(kr + nx);
    qa = *(const float4*)(qr + nx);
    p1 = products<QW>(kb.y, qb.y);
    add_products<N>(acc, p0);
    p0 = products<QW>(kb.z, qb.z);
    add_products<N>(acc, p1);
    p1 = products<QW>(kb.w, qb.w);
    add_products<N>(acc, p0);
    p0 = products<QW>(ka.x, qa.x);
    add_products<N>(acc, p1);
  }
  return acc;
}

// o += v_k p_k over n8 batches of 8 keys: vr is this lane's dimension of key
// 0's staged row, pr the probabilities of query l % QW.
template <int N, int QW>
__device__ __forceinline__ void chunk_pv(Tile<QW>& o, const float* vr, const float* pr, int n8) {
  float va[4], vb[4];
  float4 pa = *(const float4*)pr, pb;
#pragma unroll
  for (int i = 0; i < 4; ++i) va[i] = vr[i * kSeqRow];
  Tile<QW> p0 = products<QW>(va[0], pa.x), p1;
#pragma unroll 1
  for (int k = 0; k < n8; ++k) {
    const float* v8 = vr + 8 * k * kSeqRow;
    pb = *(const float4*)(pr + 8 * k + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) vb[i] = v8[(4 + i) * kSeqRow];
    p1 = products<QW>(va[1], pa.y);
    add_products<N>(o, p0);
    p0 = products<QW>(va[2], pa.z);
    add_products<N>(o, p1);
    p1 = products<QW>(va[3], pa.w);
    add_products<N>(o, p0);
    p0 = products<QW>(vb[0], pb.x);
    add_products<N>(o, p1);
    const int nx = k + 1 < n8 ? 8 * (k + 1) : 8 * k;  // past the end: re-read and unused
    pa = *(const float4*)(pr + nx);
#pragma unroll
    for (int i = 0; i < 4; ++i) va[i] = vr[(nx + i) * kSeqRow];
    p1 = products<QW>(vb[1], pb.y);
    add_products<N>(o, p0);
    p0 = products<QW>(vb[2], pb.z);
    add_products<N>(o, p1);
    p1 = products<QW>(vb[3], pb.w);
    add_products<N>(o, p0);
    p0 = products<QW>(va[0], pa.x);
    add_products<N>(o, p1);
  }
}

// The work units: a (sequence, 64 queries, head), or a sequence of at most 32
// (16) keys with two (four) of its heads.  Sequences fall into classes of equal
// units: class 0 up to 16 rows, 1 up to 32, k >= 2 up to 64 (k - 1).
__device__ __forceinline__ int seq_class(int L) { return L <= 32 ? (L > 16) : 1 + (L + 63) / 64; }
__device__ __forceinline__ int class_units(int k, int heads) {
  return k == 0 ? (heads + 3) / 4 : (k == 1 ? (heads + 1) / 2 : heads * (k - 1));
}

// Unit u of the n sequences in cu, longest classes first (so that no long
// unit starts last); false past the last unit.  Every wave finds it alone:
// the lanes hold 64 sequences' classes, ballots count and select.
template <int NCLS>
__device__ __forceinline__ bool find_unit(const uint32_t* cu, int n, int heads, int u, int lane, int& sq, int& qt,
                                          int& h0) {
  constexpr int B = 4;  // 64-sequence blocks requested together
  int cnt[NCLS] = {};
  int cls[B];
  auto load = [&](int s0) {
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const int s = s0 + 64 * j + lane, sc = min(s, n - 1);
      const int L = (int)(cu[sc + 1] - cu[sc]);
      cls[j] = s < n && L > 0 ? min(seq_class(L), NCLS - 1) : -1;
    }
  };
  for (int s0 = 0; s0 < n; s0 += 64 * B) {
    load(s0);
#pragma unroll
    for (int j = 0; j < B; ++j)
#pragma unroll
      for (int k = 0; k < NCLS; ++k) cnt[k] += __popcll(__ballot(cls[j] == k));
  }
  int want = -1;
#pragma unroll
  for (int k = NCLS - 1; k >= 0; --k) {
    const int units = cnt[k] * class_units(k, heads);
    if (want < 0) {
      if (u < units)
        want = k;
      else
        u -= units;
    }
  }
  if (want < 0) return false;
  const int per = class_units(want, heads);
  int ord = u / per;  // the class's ord-th sequence
  const int rem = u - ord * per;
  qt = want < 2 ? 0 : rem / heads;
  h0 = want == 0 ? 4 * rem : (want == 1 ? 2 * rem : rem - qt * heads);
  for (int s0 = 0; s0 < n; s0 += 64 * B) {
    if (n > 64 * B) load(s0);
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const uint64_t m = __ballot(cls[j] == want);
      const int c = __popcll(m);
      if (ord >= 0 && ord < c) {
        const int before = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
        const uint64_t hit = __ballot(cls[j] == want && before == ord);
        sq = s0 + 64 * j + __ffsll((unsigned long long)hit) - 1;
      }
      ord -= c;
    }
    if (ord < 0) break;
  }
  return true;
}

// Rows q0, q0 + 1, ... of a sequence, past the query tiles of the launch: one
// query per wave, lane = key or dimension, every operand straight from memory,
// the arithmetic in the order above.  Only a sequence longer than max_keys said
// comes here (the host does not know the lengths), so that its rows are written
// all the same.
template <int CH, typename T, int DH>
__device__ __forceinline__ void rest_of_sequence(const AttnArgs& a, int64_t key0, int L, int Lc, int h, int q0, int w,
                                                 int lane, float* sE, const uint64_t* sTab) {
  const T* kh = (const T*)a.k + key0 * a.ldkv + h * DH;
  const T* vh = (const T*)a.v + key0 * a.ldkv + h * DH + min(lane, DH - 1);
  bool bad = false;
#pragma unroll 1
  for (int64_t r = q0 + w; r < L; r += kSeqWaves) {
    const T* qr = (const T*)a.q + (key0 + r) * a.ldq + h * DH;
    float mx = -INFINITY;
#pragma unroll 1
    for (int c = 0; c < CH && 64 * c < Lc; ++c) {
      const T* kr = kh + min(64 * c + lane, Lc - 1) * a.ldkv;
      float dot = -0.0f;
#pragma unroll 1
      for (int i = 0; i < DH; ++i) dot = dot + load1(qr + i) * load1(kr + i);
      const float sc = 64 * c + lane < Lc ? dot * (1.0f / sqrtf((float)DH)) : -INFINITY;
      sE[64 * c + lane] = sc;
      mx = fmaxf(mx, sc);
    }
    mx = wave_max(mx);
#pragma unroll 1
    for (int c = 0; c < CH && 64 * c < Lc; ++c) sE[64 * c + lane] = ref_expf(sE[64 * c + lane] - mx, sTab);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's LDS writes land
    __builtin_amdgcn_wave_barrier();
    float sum = 0.0f, o = 0.0f;
#pragma unroll 1
    for (int k = 0; k < Lc; ++k) sum = sum + sE[k];
    const float inv = 1.0f / sum;
#pragma unroll 1
    for (int k = 0; k < Lc; ++k) o = o + load1(vh + k * a.ldkv) * (sE[k] * inv);
    __builtin_amdgcn_wave_barrier();
    if (lane < DH) {
      a.out[(key0 + r) * a.ldo + h * DH + lane] = o;
      if (a.qout) a.qout[(key0 + r) * a.ldqout + h * DH + lane] = (int8_t)quantize_one(o, a.qmult);
      bad |= !isfinite(o);
    }
    if (a.qout && h == 0 && lane == 0) a.qa[key0 + r] = a.qmult;
  }
  if (__any(bad) && lane == 0 && a.err) *a.err = 1;
}

// CH: 64-key chunks whose scores the registers hold (4: 256 keys; 8: 512 keys).
// QW: queries per wave.
// GEN: rows by 64-bit addresses, for the strides and alignments that
// seq_buffer_rows refuses (any stride, overlapping rows, odd bf16 addresses).
template <int CH, int QW, typename T, int DH, bool GEN>
__global__ __launch_bounds__(64 * kSeqWaves, QW == 4 ? 4 : (CH <= 4 ? 3 : 2)) void k_attn_seq(AttnArgs a) {
  static_assert(DH == 64 || DH == 48, "head widths");
  static_assert(64 * CH <= 64 * kSeqRow / kSeqWaves, "a wave's part of the stage holds a query's scores");
  constexpr int W = kSeqWaves, TQ = W * QW;  // queries per workgroup
  constexpr int G = 64 / QW;                 // lane groups of a tile
  constexpr int NB = QW / 4;                 // tile blocks of 4 G rows
  constexpr int NP = 16 / W;                 // staged 16-byte pieces per thread
  __shared__ __attribute__((aligned(16))) float stage[64 * kSeqRow];                  // K, then V rows
  __shared__ __attribute__((aligned(16))) float sPall[TQ * kSeqRow];  // queries, then probabilities
  __shared__ uint64_t sTab[32];
  const int tid = threadIdx.x, lane = tid & 63;
  int sq, qt, h0, tiles;  // tiles: query tiles of the launch
  if (QW == 16 && a.n_seqs <= kSeqFindMax) {
    if (!find_unit<CH + 2>(a.cu, a.n_seqs, a.heads, blockIdx.x, lane, sq, qt, h0)) return;
    sq = __builtin_amdgcn_readfirstlane(sq);
    qt = __builtin_amdgcn_readfirstlane(qt);
    h0 = __builtin_amdgcn_readfirstlane(h0);
    tiles = CH;  // the last class's
  } else if constexpr (QW == 4) {
    // Workgroups go round the 8 XCDs and their 32 CUs in order: a sequence's heads
    // lie on different XCDs, and high query tiles, which only long sequences have,
    // go first.  A sequence's tiles are heads * n_seqs workgroups apart, so the one
    // 256 / gcd(heads * n_seqs, 256) on would come to the first's CU: each such
    // group of tiles starts one sequence on (32 sequences, 775 rows, 8 heads:
    // 22.5 us without, 10.1 with).
    h0 = blockIdx.x;
    tiles = gridDim.z;
    qt = tiles - 1 - blockIdx.z;
    sq = (blockIdx.y + (blockIdx.z >> (8 - __builtin_ctz(a.heads * a.n_seqs | 256)))) % a.n_seqs;
  } else {
    // Every sequence's heads lie on different XCDs; the heads go slowest, or
    // whole XCDs would idle where short sequences' heads exit (below).
    sq = blockIdx.x % a.n_seqs;
    h0 = blockIdx.x / a.n_seqs;
    tiles = gridDim.y;
    qt = tiles - 1 - blockIdx.y;  // high query tiles first
  }
  const int64_t key0 = a.cu[sq];
  const int L = (int)(a.cu[sq + 1] - key0);
  // Heads per workgroup, staged rows per head, query tiles (waves) per head.
  const int hpw = QW == 4 || L > 32 ? 1 : (L > 16 ? 2 : 4);
  const int sp = 64 / hpw, tph = W / hpw;
  if (qt * TQ >= L || h0 % hpw) return;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Waves without queries rotate with the workgroup, so they do not all fall on one SIMD.
  const int role = (w + blockIdx.x) % W;
  const int sub = role / tph, h = h0 + sub;
  const int ql = lane % QW, g = lane / QW;
  const int Lc = min(L, 64 * CH);  // a longer range is cut to its first keys (and flagged)
  const int nch = (Lc + 63) >> 6;
  // A unit's time grows with its chunks, and with few rows the longest units
  // decide the call: they issue first (112 sentences 21.2 -> 19.9 us, 8 segments
  // 30.3 -> 28.3; 6 segments and where the chip is full within 1%).
  if (nch >= 4)
    __builtin_amdgcn_s_setprio(3);
  else if (nch == 3)
    __builtin_amdgcn_s_setprio(2);
  else if (nch == 2)
    __builtin_amdgcn_s_setprio(1);
  float* sP = sPall + w * QW * kSeqRow;
  const float* prow = sP + ql * kSeqRow;
  const float scale = 1.0f / sqrtf((float)DH);
  const T* kp = (const T*)a.k;
  const T* vp = (const T*)a.v;
  const T* qp = (const T*)a.q;
  if (tid < 32) sTab[tid] = kSeqExp2Tab[tid];
  if (L > Lc && tid == 0 && a.err) *a.err = 2;

  // Staged rows: thread t moves four values (t % 16) of rows t / 16 + 4 W i:
  // row hs * sp + key holds that key of head h0 + hs; keys past the last are zero.
  decltype(load4(__amdgpu_buffer_rsrc_t(), 0, T())) pre[NP];  // converted when published
  uint32_t off[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int row = (tid >> 4) + 4 * W * i, hs = row / sp;
    off[i] = ((uint32_t)(row - hs * sp) * (uint32_t)a.ldkv + hs * DH + min((tid & 15) * 4, DH - 4)) * sizeof(T);
  }
  const int nh = min(hpw, a.heads - h0);
  auto request = [&](const T* src, int c) {
    if constexpr (GEN) {
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int row = (tid >> 4) + 4 * W * i, hs = row / sp, key = 64 * c + row - hs * sp;
        pre[i] = {};
        if (key < Lc && hs < nh)
          pre[i] = load4(src + (key0 + key) * a.ldkv + (h0 + hs) * DH + min((tid & 15) * 4, DH - 4));
      }
      return;
    }
    const __amdgpu_buffer_rsrc_t r =
        rows_of(src + (key0 + 64 * c) * a.ldkv + (int64_t)h0 * DH, min(Lc - 64 * c, sp), a.ldkv, nh * DH);
#pragma unroll
    for (int i = 0; i < NP; ++i) pre[i] = load4(r, off[i], T());
  };
  auto publish = [&]() {
#pragma unroll
    for (int i = 0; i < NP; ++i) *(u32x4*)(stage + ((tid >> 4) + 4 * W * i) * kSeqRow + (tid & 15) * 4) = floats4(pre[i]);
  };

  const int qw = qt * TQ + (role % tph) * QW;  // this wave's first query
  const int nq = min(L - qw, QW);
  const bool live = nq > 0 && h < a.heads;  // uniform per wave
  request(kp, 0);
  if (live) {
    float qv[QW];
    if constexpr (GEN) {
#pragma unroll
      for (int i = 0; i < QW; ++i) {
        qv[i] = 0.0f;
        if (i < nq) qv[i] = load1(qp + (key0 + qw + i) * a.ldq + h * DH + min(lane, DH - 1));
      }
    } else {
      const __amdgpu_buffer_rsrc_t r = rows_of(qp + (key0 + qw) * a.ldq + h * DH, nq, a.ldq, DH);
#pragma unroll
      for (int i = 0; i < QW; ++i)
        qv[i] = load1(r, ((uint32_t)i * (uint32_t)a.ldq + min(lane, DH - 1)) * (uint32_t)sizeof(T), T());
    }
#pragma unroll
    for (int i = 0; i < QW; ++i) sP[i * kSeqRow + lane] = qv[i];
  }

  // ---- scores: rows are the chunk's keys ----
  Tile<QW> sc[CH];
  float mx = -INFINITY;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    if (c < nch) {
      __syncthreads();  // the staged rows have been read
      publish();
      __syncthreads();
      if (c + 1 < nch)
        request(kp, c + 1);
      else
        request(vp, 0);
      if (live) {
        const int left = Lc - 64 * c;  // keys of the chunk
        const float* kr = stage + (sub * sp + (lane & (sp - 1))) * kSeqRow;
        sc[c] = QW == 4 || left > 32 ? chunk_scores<QW, QW, DH>(kr, prow) : chunk_scores<QW / 2, QW, DH>(kr, prow);
#pragma unroll
        for (int i = 0; i < QW; ++i) {
          sc[c][i] = 4 * G * (i >> 2) + 4 * g + (i & 3) < left ? sc[c][i] * scale : -INFINITY;
          mx = fmaxf(mx, sc[c][i]);
        }
      }
    }
  }

  // ---- softmax: max, exponentials (scores are never above their maximum; the -inf past the last key
  // gives 0, or NaN where a NaN or infinite row has made the denominator NaN anyway), the denominator
  // folded in key order by every lane of a query ----
  float inv = 0.0f;
  if (live) {
    if constexpr (QW == 4) {
      mx = fmaxf(mx, xor_lane_f<4>(mx));
      mx = fmaxf(mx, xor_lane_f<8>(mx));
    }
    mx = fmaxf(mx, xor_lane_f<16>(mx));
    mx = fmaxf(mx, xor_lane_f<32>(mx));
    float sum = 0.0f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      if (c < nch) {
        const int left = Lc - 64 * c;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          if (4 * G * b < left) {
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[c][4 * b + r] = ref_expf_nonpos(sc[c][4 * b + r] - mx, sTab);
            *(float4*)(sP + ql * kSeqRow + 4 * G * b + 4 * g) =
                make_float4(sc[c][4 * b], sc[c][4 * b + 1], sc[c][4 * b + 2], sc[c][4 * b + 3]);
          }
          __builtin_amdgcn_sched_barrier(0);  // few exponentials in flight: their doubles are registers
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's LDS writes land
        __builtin_amdgcn_wave_barrier();
        sum = seq_fold_lds_upto<4>((const float4*)prow, min((left + 15) >> 4, 4), sum);
        __builtin_amdgcn_wave_barrier();
      }
    }
    inv = 1.0f / sum;
  }

  // ---- PV: rows are the dimensions ----
  Tile<QW> o = {0};
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    if (c < nch) {
      const int left = Lc - 64 * c;
      __syncthreads();  // the staged rows have been read
      publish();
      if (live) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
          if (4 * G * b < left)
            *(float4*)(sP + ql * kSeqRow + 4 * G * b + 4 * g) =
                make_float4(sc[c][4 * b] * inv, sc[c][4 * b + 1] * inv, sc[c][4 * b + 2] * inv,
                            sc[c][4 * b + 3] * inv);
      }
      __syncthreads();
      if (c + 1 < nch) request(vp, c + 1);
      if (live)
        chunk_pv<QW == 4 ? 4 : DH / 4, QW>(o, stage + sub * sp * kSeqRow + min(lane, DH - 1), prow,
                          __builtin_amdgcn_readfirstlane(min((left + 7) >> 3, 8)));
    }
  }

  if (live) {
    bool bad = false;
    const int64_t row = key0 + qw + ql;
    if (ql < nq) {
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int dim = 4 * G * b + 4 * g, col = h * DH + dim;
        if (dim >= DH) continue;
        const f4u v = {o[4 * b], o[4 * b + 1], o[4 * b + 2], o[4 * b + 3]};
        *(f4u*)(a.out + row * a.ldo + col) = v;
        if (a.qout) {  // static multiplier of the next layer (elementwise)
          uint32_t pk = 0;
#pragma unroll
          for (int r = 0; r < 4; ++r) pk |= (uint32_t)(quantize_one(v[r], a.qmult) & 0xFF) << (8 * r);
          *(u32u*)(a.qout + row * a.ldqout + col) = pk;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) bad |= !isfinite(v[r]);
      }
      if (a.qout && h == 0 && g == 0) a.qa[row] = a.qmult;
    }
    if (__any(bad) && lane == 0 && a.err) *a.err = 1;
  }
  if (L > tiles * TQ && qt == tiles - 1) {  // the whole workgroup
    __syncthreads();  // the staged rows have been read
    rest_of_sequence<CH, T, DH>(a, key0, L, Lc, h0, tiles * TQ, w, lane, stage + w * (64 * kSeqRow / W), sTab);
  }
}

template <int CH, int QW, typename T, bool GEN>
void launch_dh(const AttnArgs& a, dim3 grid, hipStream_t s) {
  if (a.head_dim == 48)
    hipLaunchKernelGGL((k_attn_seq<CH, QW, T, 48, GEN>), grid, dim3(64 * kSeqWaves), 0, s, a);
  else
    hipLaunchKernelGGL((k_attn_seq<CH, QW, T, 64, GEN>), grid, dim3(64 * kSeqWaves), 0, s, a);
}
template <int CH, int QW, bool GEN = false>
void launch_t(const AttnArgs& a, dim3 grid, hipStream_t s) {
  if (a.bf16)
    launch_dh<CH, QW, uint16_t, GEN>(a, grid, s);
  else
    launch_dh<CH, QW, float, GEN>(a, grid, s);
}

// Whether the rows fit the kernel's raw buffers: 64 key rows (16 query rows)
// within 32-bit offsets, no row reaching into the next (a row past the range's
// end has to lie past it in every head), 4-byte aligned four-element loads.
bool seq_buffer_rows(const AttnArgs& a) {
  const int64_t d = (int64_t)a.heads * a.head_dim, size = a.bf16 ? 2 : 4, top = int64_t(1) << 32;
  return a.ldq >= d && a.ldkv >= d && a.ldkv < top / (64 * size) && a.ldq < top / (16 * size) &&
         ((uintptr_t)a.k | (uintptr_t)a.v) % 4 == 0;
}

}  // namespace

// One wave per (row, head) is faster where few long rows leave even the 4-query
// units' eight chunks unhidden: 424 rows of 257-512 keys with 1 head 18.0 | 26.9 us
// here, with 2 20.4 | 26.9, with 3 (1284 pairs) 24.5 | 26.8, with 4 (1712) 27.9 | 26.7.
// The average length tells such calls from short sequences under a max_keys
// far above them.  That kernel addresses all keys of a range by 32 bits.
bool attention_seq_wins(const AttnArgs& a) {
  return a.max_keys <= 256 || (int64_t)a.rows * a.heads > 1536 || a.rows <= 128 * (int64_t)a.n_seqs ||
         !seq_buffer_rows(a) || a.ldkv >= (int64_t(1) << 32) / (kSeqMaxKeys * 4);
}

hipError_t launch_attention_seq(const AttnArgs& a, hipStream_t s) {
  if (a.mode != ATT_SEQ || a.n_seqs <= 0 || a.max_keys <= 0 || a.max_keys > kSeqMaxKeys || !a.cu ||
      (int64_t)a.n_seqs * a.heads > 0x7fffffff || (int64_t)a.rows * a.heads > 0x7fffffff)
    return hipErrorInvalidValue;
  const bool gen = !seq_buffer_rows(a);
  const int64_t groups = (int64_t)a.n_seqs * a.heads * ((a.max_keys + 4 * kSeqWaves - 1) / (4 * kSeqWaves));
  const bool few = !gen && (int64_t)a.rows * a.heads <= (a.max_keys <= 256 ? kSeqFewRows256 : kSeqFewRows512) &&
                   groups <= std::max(kSeqFewGroups, kSeqFewGroupsPer * a.n_seqs);
  const int tq = kSeqWaves * (few ? 4 : 16);
  // Units: at most heads / 4 + 7 / 256 heads L of a sequence of L rows (equal at 65 rows).
  const int64_t units = (int64_t)a.n_seqs * ((a.heads + 3) / 4) + ((int64_t)a.rows * a.heads * 7 + 255) / 256;
  const uint32_t tiles = (a.max_keys + tq - 1) / tq;
  const dim3 grid = few                         ? dim3(a.heads, a.n_seqs, tiles)
                    : a.n_seqs <= kSeqFindMax ? dim3((uint32_t)units)
                                                : dim3(a.n_seqs * a.heads, tiles);
  if (gen)
    launch_t<8, 16, true>(a, grid, s);
  else if (a.max_keys <= 256)
    few ? launch_t<4, 4>(a, grid, s) : launch_t<4, 16>(a, grid, s);
  else
    few ? launch_t<8, 4>(a, grid, s) : launch_t<8, 16>(a, grid, s);
  return hipGetLastError();
}

}  // namespace mh
