// Gated DeltaNet chunked prefill as a fused scan: the chunk output is computed
// beside the state recurrence, and long sequences are cut into segments.
//
// Semantics and chunk algebra as in gdn_prefill.hip (chunk = 64 tokens, G the
// chunk-local cumsum of the log decay, T = (I + A)^-1, S the k-last state):
//   v_new = T diag(beta) (V - e^G K S),   o = scale (e^G Q S + P v_new),
//   S    <- e^{G_last} S + K^T (e^{G_last - G} v_new),
//   P     = mask_{j<=i}(e^{G_i - G_j} q_i . k_j).
// Two launches (three when a sequence is cut):
//   1. scan_intra_kernel, per (chunk, v-head): T' = T diag(beta) (split bf16),
//      P (bf16) and the per-token decay factors, 19 KB, as MFMA fragments.
//   2. scan_chain_kernel, per (sequence, v-head, 32 state columns): the
//      recurrence over the chunks, and the output.
//
// What bounds it: the recurrence is a serial chain of three products per
// chunk, K S, T' y and K^T D, and the operand-form pipeline spreads one
// 16-column state tile over the four waves of a workgroup, which exchange the
// state, the right-hand side and v_new through LDS at every step; its step
// then waits on those exchanges, and every 16 columns load all operands anew.
// Here one wave owns a 16-column tile for all 128 k.  The rows of the state
// tiles and of the K and T' operands are numbered so that a product's result
// tile is, lane by lane, the next product's operand: the chain needs no
// exchange at all, and the operands are staged in LDS once for all of a
// workgroup's waves.  Two helper waves beside the two chain waves stage K, V
// and Q a chunk ahead and compute the output from the bf16 state and v_new
// that the chain waves publish, so the output costs no launch, no second read
// of Q and K, and no round trip of the chunk-start states (48 KB per chunk and
// head).  A step takes 1.4 us for 32 columns alone on a CU (~80 matrix and
// ~330 vector instructions per chain wave), two workgroups fit a CU.
// Workgroups of four or eight chain waves, or of 32 columns per wave, were
// slower (1.8, 3.4 and 3.1 us a step).
//
// Measured against the operand-form pipeline (us per call, states given):
// 64x256 161 -> 93, 16x1024 135 -> 74, 8x2048 133 -> 79, 2x4096 94 -> 70,
// 4x8192 252 -> 187, 1x8192 110 -> 81, 1x512 27 -> 24; 1x1024 31 -> 35.
#include "gdn_chunk.h"
#include "gdn_device.h"
#include "gdn_host.h"

namespace gdn {

// Record of one (chunk, v-head), left by scan_intra_kernel: T' and P as MFMA
// fragments, then the per-token vectors e^{G_i} and e^{G_last - G_i} (f32).
// Fragment x of T' is 1 KB of bf16 hi parts and 1 KB of lo parts, fragment x
// of P is 1 KB; x = 0..5 names the 16-row tile and 32-column step (r, jj), jj
// <= r / 2: (0,0) (1,0) (2,0) (2,1) (3,0) (3,1).
constexpr int kRecT = 0, kRecP = 6 * 2048, kRecVec = kRecP + 6 * 1024;
constexpr int kRecBytes = kRecVec + 2 * kChunk * 4;
constexpr size_t kRecStride = static_cast<size_t>(kChunk) * kDK * 4;  // its slot in the w region

constexpr int kScanIntraLds = kChunk * kStrideK * 2 + 10 * kABlk * 4 + 2 * kChunk * 4;

__device__ __forceinline__ void scan_intra(
    char *smem, char *rec, int h, int start, int len, const uint16_t *__restrict__ q,
    const uint16_t *__restrict__ k, const float *__restrict__ A_log,
    const uint16_t *__restrict__ a, const float *__restrict__ dt_bias,
    const uint16_t *__restrict__ b, const Heads &H) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4, kg = g * 8;
  const int hq = h / H.ratio;
  constexpr int kStrideF = 68;  // f32 stride of the T scratch (16-byte rows)
  uint16_t *const sK = reinterpret_cast<uint16_t *>(smem);              // [64][136]
  float *const sA = reinterpret_cast<float *>(sK + kChunk * kStrideK);  // 10 blocks
  float *const sBeta = sA + 10 * kABlk, *const sG = sBeta + kChunk;
  static_assert(kChunk * kStrideF * 4 <= kChunk * kStrideK * 2, "T must fit in the K tile");
  float *const sT = reinterpret_cast<float *>(sK);

  u32x4 qf[4];  // this wave's 16 rows of Q, k-steps 0..3 (B operand of P^T)
  {
    const uint32_t rstride = static_cast<uint32_t>(H.qk) * (kDK * 2);
    const size_t base = (static_cast<size_t>(start) * H.qk + hq) * kDK;
    const auto rk = buf_rsrc(k + base, static_cast<uint32_t>(len) * rstride);
    const auto rq = buf_rsrc(q + base, static_cast<uint32_t>(len) * rstride);
    u32x4 kv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = tid + 256 * i;
      kv[i] = buf_load16(rk, static_cast<uint32_t>(idx >> 4) * rstride + (idx & 15) * 16);
    }
    if (wave == 0) {
      float gl, be;
      chunk_gates(lane, start, len, h, H, A_log, a, dt_bias, b, gl, be);
      float G = gl;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const float y = __shfl_up(G, off);
        if (lane >= off) G += y;
      }
      sG[lane] = G;
      sBeta[lane] = be;
      const float G_last = __shfl(G, 63);
      float *vec = reinterpret_cast<float *>(rec + kRecVec);
      vec[lane] = expf(G);
      vec[kChunk + lane] = expf(G_last - G);
    }
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
      qf[kk] = buf_load16(rq, static_cast<uint32_t>(16 * wave + r16) * rstride + (32 * kk + kg) * 2);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = tid + 256 * i;
      *reinterpret_cast<u32x4 *>(&sK[(idx >> 4) * kStrideK + (idx & 15) * 8]) = kv[i];
    }
  }
  __syncthreads();

  build_A(sK, sA, sG, sBeta, len, wave, lane);

  // P = mask_{j<=i}(e^{G_i - G_j} q_i . k_j), rows i = 16 wave + r16, as the
  // transposed product K Q^T: with the K rows of tile (jj, t) permuted so that
  // its row 4 g + r is token 32 jj + 8 g + 4 t + r, the two tiles t = 0, 1 hold
  // 8 consecutive j of one row i per lane, the fragment the chain kernel reads.
#pragma unroll
  for (int jj = 0; jj < 2; ++jj) {
    if (jj > (wave >> 1)) break;
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int row = 32 * jj + 8 * (r16 >> 2) + 4 * t + (r16 & 3);
        const u32x4 kf = *reinterpret_cast<const u32x4 *>(&sK[row * kStrideK + 32 * kk + kg]);
        acc[t] = mfma_bf16(kf, qf[kk], acc[t]);
      }
    const int i = 16 * wave + r16;
    const float Gi = sG[i];
    u32x4 pf;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int j0 = 32 * jj + kg + 4 * t;
      const f32x4 Gj = *reinterpret_cast<const f32x4 *>(&sG[j0]);
      float p[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float d = __builtin_amdgcn_exp2f(fminf(Gi - Gj[r], 0.f) * 1.44269504088896341f);
        p[r] = j0 + r <= i ? d * acc[t][r] : 0.f;
      }
      pf[2 * t] = pk_bf16(p[0], p[1]);
      pf[2 * t + 1] = pk_bf16(p[2], p[3]);
    }
    const int x = wave < 2 ? wave : 2 * wave - 2 + jj;
    *reinterpret_cast<u32x4 *>(rec + kRecP + x * 1024 + lane * 16) = pf;
  }
  __syncthreads();
  diag_inverse(sA, wave, lane);
  __syncthreads();

  // Block column j = wave of T = (I + A)^-1, scaled by beta of its columns:
  // T' = T diag(beta).
  f32x4 Tc[4];
  t_column(sA, wave, g, r16, Tc);
  const float be = sBeta[16 * wave + r16];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      sT[(16 * i + 4 * g + r) * kStrideF + 16 * wave + r16] = Tc[i][r] * be;
  __syncthreads();

  // T' as split A operand fragments: tile (ii, t) = wave, row r16 of the tile
  // is token 32 ii + 8 (r16 / 4) + 4 t + r16 % 4.
  const int row = 32 * (wave >> 1) + 8 * (r16 >> 2) + 4 * (wave & 1) + (r16 & 3);
#pragma unroll
  for (int jj = 0; jj < 2; ++jj) {
    if (jj > (wave >> 1)) break;
    const f32x4 x0 = *reinterpret_cast<const f32x4 *>(&sT[row * kStrideF + 32 * jj + kg]);
    const f32x4 x1 = *reinterpret_cast<const f32x4 *>(&sT[row * kStrideF + 32 * jj + kg + 4]);
    const float x8[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
    u32x4 hi, lo;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t h2, l2;
      split2_rne(x8[2 * e], x8[2 * e + 1], h2, l2);
      hi[e] = h2;
      lo[e] = l2;
    }
    const int x = wave < 2 ? wave : 2 * wave - 2 + jj;
    char *dst = rec + kRecT + x * 2048 + lane * 16;
    *reinterpret_cast<u32x4 *>(dst) = hi;
    *reinterpret_cast<u32x4 *>(dst + 1024) = lo;
  }
}

__global__ __launch_bounds__(256) void scan_intra_kernel(
    const uint16_t *__restrict__ q, const uint16_t *__restrict__ k,
    const float *__restrict__ A_log, const uint16_t *__restrict__ a,
    const float *__restrict__ dt_bias, const uint16_t *__restrict__ b,
    const int4 *__restrict__ chunks, OneSeq one, int nt_max, Heads H, SelfIndex si,
    char *__restrict__ ws_rec) {
  constexpr int kLds = kScanIntraLds > kSelfIndexLds ? kScanIntraLds : kSelfIndexLds;
  __shared__ __align__(16) char smem[kLds];
  const int id = blockIdx.x;
  int c = 0, h = 0;
  const bool unit = chunk_head_of(id, nt_max, H, c, h);
  int4 ch;
  if (si.cu != nullptr) {
    if (!unit && id != 0) return;
    const SelfIndexed x = self_index(smem, si, nt_max, H.v);
    ch = self_chunk(smem, si.N, c, x.nt);
    __syncthreads();  // the LDS arrays are dead: the unit's tiles take their place
    if (!unit) return;
  } else {
    if (one.cu != nullptr && id == 0 && threadIdx.x < 64) {
      if (threadIdx.x == 0)
        si.status[0] = cu_status_bits(raw_cu(one.cu, one.cu64, 0), raw_cu(one.cu, one.cu64, 1), one.T);
      if (si.max_more > 0) {
        int bos, eos;
        one_seq_bounds(one, bos, eos);
        const int n = threadIdx.x == 0 ? (eos - bos + kChunk - 1) / kChunk : 0;
        const int len = segment_length(n, si.max_more, H.v);
        if (threadIdx.x == 0) si.offsets[si.N + 2] = len;
      }
    }
    if (!unit) return;
    ch = chunk_info(chunks, c, one);
  }
  if (ch.x < 0) return;
  scan_intra(smem, ws_rec + (static_cast<size_t>(c) * H.v + h) * kRecStride, h, ch.y, ch.z, q, k,
             A_log, a, dt_bias, b, H);
}

// ---------------------------------------------------------------------------
// the recurrence and the output
// ---------------------------------------------------------------------------
struct ScanArgs {
  const uint16_t *q, *k, *v;
  const float *state;
  float *new_state;
  uint16_t *out;
  const void *cu;
  int cu64, N, T;
  const int *offsets;  // first chunk of each sequence (nullptr: one sequence)
  const char *rec;
  char *seg;           // segment maps (SegSlot)
  const int *seg_len;  // chunks of a segment, 0 if the sequences are not cut (nullptr: 0)
  int out_units;       // first launch: units of the first segments' output
  int out_grid;        // and the workgroups that take them (fewer: each loops)
  Heads H;
  float scale;
};

constexpr int kScanThreads = 256;
static_assert(kMinSegment >= 4, "a segment's map takes four of its chunks' slots (SegSlot)");
constexpr int kOutCols = 32, kMapCols = 64;  // state columns of a workgroup
constexpr int kLKBytes = kChunk * kDK * 2;   // K or Q rows of one chunk
constexpr int kLEBytes = 2 * kChunk * 4;     // its per-token vectors
// LDS maps (bytes).  K, V and the vectors are double-buffered by chunk parity;
// Q, the published state and v_new are handed over within a chunk.  OutLds: a
// workgroup of two chain waves and two helpers; MapLds: four chain waves.
struct OutLds {
  static constexpr int K = 0;
  static constexpr int V = 2 * kLKBytes, VRow = kOutCols * 2, VBytes = kChunk * VRow;
  static constexpr int E = V + 2 * VBytes;
  static constexpr int Q = E + 2 * kLEBytes;
  static constexpr int S = Q + kLKBytes;  // chunk-start state, bf16: 4 KB per column tile
  static constexpr int N = S + 2 * 4096;  // v_new, bf16: 2 KB per column tile
  static constexpr int kBytes = N + 2 * 2048;
  static constexpr bool kPublish = true;
  static constexpr int kTiles = 2;
  // 16-byte unit u of a V row, placed so that the transposing reads of four
  // rows touch distinct banks
  __device__ static int vunit(int, int u) { return u; }
};
struct MapLds {
  static constexpr int K = 0;
  static constexpr int V = 2 * kLKBytes, VRow = kMapCols * 2, VBytes = kChunk * VRow;
  static constexpr int E = V + 2 * VBytes;
  static constexpr int S = 0, N = 0;
  static constexpr int kBytes = E + 2 * kLEBytes;
  static constexpr bool kPublish = false;
  static constexpr int kTiles = 4;
  __device__ static int vunit(int row, int u) { return u ^ (4 * ((row >> 1) & 1)); }
};
constexpr int kMapStride = 72;  // bf16 row stride of the linear map's columns in LDS
constexpr int kScanLds = OutLds::kBytes;
static_assert(MapLds::kBytes <= kScanLds && 2 * kDK * kMapStride * 2 <= kScanLds, "shared by both");
static_assert(2 * kScanLds <= 160 * 1024, "two workgroups per compute unit");

__device__ __forceinline__ u32x4 lds16(const char *p) { return *reinterpret_cast<const u32x4 *>(p); }
__device__ __forceinline__ f32x4 lds4f(const char *p) { return *reinterpret_cast<const f32x4 *>(p); }
__device__ __forceinline__ u32x2 lds_tr(const char *p) {
  return ds_read_tr16(reinterpret_cast<const uint16_t *>(p));
}
// 16-byte unit u of K row `row` of a chunk in LDS (rows of 256 bytes).
__device__ __forceinline__ int kunit(int row, int u) {
  return row * 256 + 16 * (u ^ (4 * (row & 3) + ((row >> 3) & 3)));
}

// What a workgroup works on: chunks [0, nch) of a segment from token bos.
struct Segment {
  int bos, eos, nch;
  const char *rec;  // record of its first chunk
  size_t rec_step;
  __device__ __forceinline__ uint32_t len(int i) const {  // tokens of chunk i (0 past the end)
    const int rem = eos - bos - i * kChunk;
    return static_cast<uint32_t>(
        __builtin_amdgcn_readfirstlane(i >= nch || rem < 0 ? 0 : rem < kChunk ? rem : kChunk));
  }
  __device__ __forceinline__ size_t start(int i) const {
    return static_cast<size_t>(bos) + static_cast<size_t>(i) * kChunk;
  }
};

// A chain wave: column tile ct (16 state columns) for all 128 k.  Its columns
// are 64 (ct / 4) + vloc + 8 (r16 / 4) + r16 % 4, so that the tiles 2 p and
// 2 p + 1 together hold 8 consecutive columns per lane group.
struct Chain {
  f32x4 S[4][2];  // lane: S[k = 32 kk + 8 g + 4 t + r][column of r16]
  u32x4 th[6], tl[6];
  // LDS offsets of the lane: its K rows (k-step 0; step kk is at ka ^ 64 kk,
  // the unit permutation being an exclusive or), K^T rows, V rows, vectors
  int ka, kt, va[2], ea;
  int lane, w;

  template <typename L>
  __device__ __forceinline__ void init(int ct, int lane_) {
    lane = lane_;
    const int r16 = lane & 15, g = lane >> 4, rl = r16 >> 2, rm = r16 & 3;
    w = ct % L::kTiles;  // tile within the workgroup's columns
    ka = L::K + kunit(8 * rl + rm, g);
    kt = L::K + kunit(8 * g + rl, rm);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int row = 8 * g + 4 * t + rl;
      va[t] = L::V + row * L::VRow + 16 * L::vunit(row, 4 * (w >> 1) + rm) + 8 * (w & 1);
    }
    ea = L::E + 32 * g;
  }
  __device__ __forceinline__ void load_t(const Segment &sg, int i) {
    const auto rr = buf_rsrc(sg.rec + i * sg.rec_step, i < sg.nch ? kRecBytes : 0);
#pragma unroll
    for (int f = 0; f < 6; ++f) {
      th[f] = buf_load16(rr, kRecT + f * 2048 + lane * 16);
      tl[f] = buf_load16(rr, kRecT + f * 2048 + 1024 + lane * 16);
    }
  }
  template <typename L, int PAR>
  __device__ __forceinline__ void step(char *smem, const Segment &sg, int ci);
};

// One chunk.
template <typename L, int PAR>
__device__ __forceinline__ void Chain::step(char *smem, const Segment &sg, int ci) {
  // (the offsets' derived values are formed at each use: kept across the loop
  // they would spill)
  asm volatile("" : "+v"(ka), "+v"(kt), "+v"(lane));
  u32x4 kf[4][4], Sh[4], Sl[4];
  auto load_kf = [&](int kk) {
#pragma unroll
    for (int x = 0; x < 4; ++x)
      kf[kk][x] = lds16(smem + (ka ^ (64 * kk)) + PAR * kLKBytes + (x >> 1) * 8192 + (x & 1) * 1024);
  };
  auto split = [&](int kk) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      uint32_t h0, h1, l0, l1;
      split2_rne(S[kk][t][0], S[kk][t][1], h0, l0);
      split2_rne(S[kk][t][2], S[kk][t][3], h1, l1);
      Sh[kk][2 * t] = h0;
      Sh[kk][2 * t + 1] = h1;
      Sl[kk][2 * t] = l0;
      Sl[kk][2 * t + 1] = l1;
    }
    if (L::kPublish) *reinterpret_cast<u32x4 *>(smem + L::S + w * 4096 + kk * 1024 + lane * 16) = Sh[kk];
  };
  // (scheduling strategy: 1x8192 84.7 -> 80.7 us, 64 short prompts 80.4 -> 80.1)
  __builtin_amdgcn_iglp_opt(2);
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 X[4] = {zero, zero, zero, zero};
  auto mul_k = [&](int kk) {
#pragma unroll
    for (int x = 0; x < 4; ++x) X[x] = mfma_bf16(kf[kk][x], Sh[kk], X[x]);
#pragma unroll
    for (int x = 0; x < 4; ++x) X[x] = mfma_bf16(kf[kk][x], Sl[kk], X[x]);
  };
  // X = K S
  load_kf(0);
  load_kf(1);
  split(0);
  load_kf(2);
  mul_k(0);
  split(1);
  load_kf(3);
  mul_k(1);
  split(2);
  u32x2 vt[4];
  f32x4 eG[4], eD[4];
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    vt[x] = lds_tr(smem + va[x & 1] + PAR * L::VBytes + (x >> 1) * (32 * L::VRow));
    eG[x] = lds4f(smem + ea + PAR * kLEBytes + (32 * (x >> 1) + 4 * (x & 1)) * 4);
  }
  mul_k(2);
  split(3);
  mul_k(3);
  if (L::kPublish) __syncthreads();  // B
  // y = v - e^G X
  u32x4 Yh[2], Yl[2];
  auto form_y = [&](int jj) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int x = 2 * jj + t;
      const float y0 = fmaf(-eG[x][0], X[x][0], __uint_as_float(vt[x][0] << 16));
      const float y1 = fmaf(-eG[x][1], X[x][1], __uint_as_float(vt[x][0] & 0xffff0000u));
      const float y2 = fmaf(-eG[x][2], X[x][2], __uint_as_float(vt[x][1] << 16));
      const float y3 = fmaf(-eG[x][3], X[x][3], __uint_as_float(vt[x][1] & 0xffff0000u));
      uint32_t h0, h1, l0, l1;
      split2_rne(y0, y1, h0, l0);
      split2_rne(y2, y3, h1, l1);
      Yh[jj][2 * t] = h0;
      Yh[jj][2 * t + 1] = h1;
      Yl[jj][2 * t] = l0;
      Yl[jj][2 * t + 1] = l1;
    }
  };
  u32x4 kc[2][8];
  auto load_kt = [&](int ii) {
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      const char *p = smem + (kt ^ (64 * (x >> 1))) + PAR * kLKBytes + ii * 8192 + 8 * (x & 1);
      const u32x2 x0 = lds_tr(p), x1 = lds_tr(p + 1024);
      kc[ii][x] = u32x4{x0[0], x0[1], x1[0], x1[1]};
    }
  };
  form_y(0);
  load_kt(0);
  // v_new = T' y (fragments 0, 1, 2, 4: columns 0..31; 3, 5: 32..63)
  f32x4 W[4];
#pragma unroll
  for (int x = 0; x < 4; ++x) W[x] = mfma_bf16(th[x < 2 ? x : 2 * x - 2], Yh[0], zero);
#pragma unroll
  for (int x = 0; x < 4; ++x) W[x] = mfma_bf16(th[x < 2 ? x : 2 * x - 2], Yl[0], W[x]);
#pragma unroll
  for (int x = 0; x < 4; ++x) W[x] = mfma_bf16(tl[x < 2 ? x : 2 * x - 2], Yh[0], W[x]);
  form_y(1);
#pragma unroll
  for (int x = 0; x < 4; ++x)
    eD[x] = lds4f(smem + ea + PAR * kLEBytes + (64 + 32 * (x >> 1) + 4 * (x & 1)) * 4);
  const float eg = *reinterpret_cast<const float *>(smem + L::E + PAR * kLEBytes + 63 * 4);
  u32x4 Dh[2], Dl[2];
  auto form_d = [&](int ii) {
    u32x4 n;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const f32x4 w = W[2 * ii + t], d = eD[2 * ii + t];
      n[2 * t] = pk_bf16(w[0], w[1]);
      n[2 * t + 1] = pk_bf16(w[2], w[3]);
      uint32_t h0, h1, l0, l1;
      split2_rne(d[0] * w[0], d[1] * w[1], h0, l0);
      split2_rne(d[2] * w[2], d[3] * w[3], h1, l1);
      Dh[ii][2 * t] = h0;
      Dh[ii][2 * t + 1] = h1;
      Dl[ii][2 * t] = l0;
      Dl[ii][2 * t + 1] = l1;
    }
    if (L::kPublish) *reinterpret_cast<u32x4 *>(smem + L::N + w * 2048 + ii * 1024 + lane * 16) = n;
  };
#pragma unroll
  for (int x = 2; x < 4; ++x) W[x] = mfma_bf16(th[2 * x - 1], Yh[1], W[x]);
#pragma unroll
  for (int x = 2; x < 4; ++x) W[x] = mfma_bf16(th[2 * x - 1], Yl[1], W[x]);
#pragma unroll
  for (int x = 2; x < 4; ++x) W[x] = mfma_bf16(tl[2 * x - 1], Yh[1], W[x]);
  load_kt(1);
  form_d(0);
  // S <- e^{G_last} S + K^T (D v_new)
  f32x4 U[8];
#pragma unroll
  for (int x = 0; x < 8; ++x) U[x] = mfma_bf16(kc[0][x], Dh[0], zero);
#pragma unroll
  for (int x = 0; x < 8; ++x) U[x] = mfma_bf16(kc[0][x], Dl[0], U[x]);
  form_d(1);
  if (L::kPublish) load_t(sg, ci + 1);
#pragma unroll
  for (int x = 0; x < 8; ++x) U[x] = mfma_bf16(kc[1][x], Dh[1], U[x]);
#pragma unroll
  for (int x = 0; x < 8; ++x) U[x] = mfma_bf16(kc[1][x], Dl[1], U[x]);
  // (the map's waves, which also stage, have no registers for it earlier)
  if (!L::kPublish) load_t(sg, ci + 1);
#pragma unroll
  for (int x = 0; x < 8; ++x)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[x >> 1][x & 1][r] = fmaf(eg, S[x >> 1][x & 1][r], U[x][r]);
}

// K rows, V columns and the vectors of chunk i: from memory into registers
// (issue) and from there into LDS (put).  THREADS threads share the work;
// COLS columns of V from col0.
template <typename L, int THREADS, int COLS>
struct Stage {
  static constexpr int kRowsK = THREADS / 16, kNumK = kChunk / kRowsK;
  static constexpr int kUnitsV = COLS / 8, kRowsV = THREADS / kUnitsV, kNumV = kChunk / kRowsV;
  u32x4 kr[kNumK], vr[kNumV];
  float er;
  __device__ __forceinline__ void issue(const ScanArgs &A, const Segment &sg, int i, int th, int h,
                                        int hq, int col0, bool with_v) {
    const uint32_t len = sg.len(i);
    const size_t start = sg.start(i);
    const uint32_t ks = static_cast<uint32_t>(A.H.qk) * (kDK * 2);
    const uint32_t vs = static_cast<uint32_t>(A.H.v) * (kDV * 2);
    const auto rk = buf_rsrc(A.k + (start * A.H.qk + hq) * kDK, len * ks);
    const auto rv = buf_rsrc(A.v + (start * A.H.v + h) * kDV, with_v ? len * vs : 0);
    const auto rr = buf_rsrc(sg.rec + i * sg.rec_step, len > 0 ? kRecBytes : 0);
#pragma unroll
    for (int j = 0; j < kNumK; ++j)
      kr[j] = buf_load16(rk, static_cast<uint32_t>((th >> 4) + kRowsK * j) * ks + (th & 15) * 16);
#pragma unroll
    for (int j = 0; j < kNumV; ++j)
      vr[j] = buf_load16(rv, static_cast<uint32_t>(th / kUnitsV + kRowsV * j) * vs +
                                 (col0 + 8 * (th % kUnitsV)) * 2);
    er = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rr, kRecVec + (th & 127) * 4, 0, 0));
  }
  __device__ __forceinline__ void put(char *smem, int par, int th) const {
#pragma unroll
    for (int j = 0; j < kNumK; ++j)
      *reinterpret_cast<u32x4 *>(smem + L::K + par * kLKBytes +
                                 kunit((th >> 4) + kRowsK * j, th & 15)) = kr[j];
#pragma unroll
    for (int j = 0; j < kNumV; ++j) {
      const int row = th / kUnitsV + kRowsV * j;
      *reinterpret_cast<u32x4 *>(smem + L::V + par * L::VBytes + row * L::VRow +
                                 16 * L::vunit(row, th % kUnitsV)) = vr[j];
    }
    *reinterpret_cast<float *>(smem + L::E + par * kLEBytes + (th & 127) * 4) = er;
  }
};

// Slot of a segment's map, in four consecutive (chunk, v-head) slots of the
// segment's chunks (32 KB each, head-interleaved): the offset (the end state
// of a first segment) in the first two, the linear part in the last two.
struct SegSlot {
  char *base;   // slot of the segment's first chunk
  size_t step;  // bytes from one chunk's slot to the next
  // f32 state tile of column tile ct in register order
  __device__ __forceinline__ char *tile(int ct, int lane) const {
    return base + (ct >> 2) * step + (ct & 3) * 8192 + lane * 16;
  }
  // A operand fragment of the linear part: state tile x = 2 kk + t (rows),
  // k-step jb (columns), half 0 hi / 1 lo
  __device__ __forceinline__ char *frag(int x, int jb, int half, int lane) const {
    return base + (2 + (x >> 2)) * step + (((x & 3) * 4 + jb) * 2 + half) * 1024 + lane * 16;
  }
};
constexpr size_t kSegSlotBytes = static_cast<size_t>(kDV) * kDK * 2;

__device__ __forceinline__ void store_tile(const f32x4 (&S)[4][2], char *p) {
#pragma unroll
  for (int x = 0; x < 8; ++x) *reinterpret_cast<f32x4 *>(p + x * 1024) = S[x >> 1][x & 1];
}

// The map of a middle segment for 64 columns (half `half`): from the zero
// state (its offset) or, `linear`, from the identity with V = 0 (its linear
// part), by four chain waves, one per column tile.
__device__ __forceinline__ void map_unit(const ScanArgs &A, char *smem, const Segment &sg,
                                         const SegSlot &slot, int h, int hq, int half, bool linear) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  Chain c;
  c.init<MapLds>(wave, lane);
  const int col = 32 * (wave >> 1) + 4 * (wave & 1) + 8 * (r16 >> 2) + (r16 & 3);  // of the 64
#pragma unroll
  for (int x = 0; x < 8; ++x)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      c.S[x >> 1][x & 1][r] =
          linear && 32 * (x >> 1) + 8 * g + 4 * (x & 1) + r == kMapCols * half + col ? 1.f : 0.f;
  Stage<MapLds, 256, kMapCols> st;
  st.issue(A, sg, 0, tid, h, hq, kMapCols * half, !linear);
  c.load_t(sg, 0);
  st.put(smem, 0, tid);
  st.issue(A, sg, 1, tid, h, hq, kMapCols * half, !linear);
  __syncthreads();
  for (int i = 0; i < sg.nch; i += 2) {
    st.put(smem, 1, tid);
    st.issue(A, sg, i + 2, tid, h, hq, kMapCols * half, !linear);
    c.step<MapLds, 0>(smem, sg, i);
    __syncthreads();
    if (i + 1 < sg.nch) {
      st.put(smem, 0, tid);
      st.issue(A, sg, i + 3, tid, h, hq, kMapCols * half, !linear);
      c.step<MapLds, 1>(smem, sg, i + 1);
      __syncthreads();
    }
  }
  if (!linear) {
    store_tile(c.S, slot.tile(4 * half + wave, lane));
    return;
  }
  // M[k][j] (j this lane's column) to A operand fragments, through LDS
  uint16_t *const mh = reinterpret_cast<uint16_t *>(smem), *const ml = mh + kDK * kMapStride;
#pragma unroll
  for (int x = 0; x < 8; ++x)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float m = c.S[x >> 1][x & 1][r];
      const uint16_t hi = f32_to_bf16(m);
      const int at = (32 * (x >> 1) + 8 * g + 4 * (x & 1) + r) * kMapStride + col;
      mh[at] = hi;
      ml[at] = f32_to_bf16(m - bf16_to_f32(hi));
    }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int row = 32 * wave + 8 * (r16 >> 2) + 4 * t + (r16 & 3);
#pragma unroll
    for (int jb = 0; jb < 2; ++jb) {
      const int at = row * kMapStride + 32 * jb + 8 * g;
      *reinterpret_cast<u32x4 *>(slot.frag(2 * wave + t, 2 * half + jb, 0, lane)) =
          *reinterpret_cast<const u32x4 *>(&mh[at]);
      *reinterpret_cast<u32x4 *>(slot.frag(2 * wave + t, 2 * half + jb, 1, lane)) =
          *reinterpret_cast<const u32x4 *>(&ml[at]);
    }
  }
}

// Start state of segment `seg` (32 columns: the tiles ct0, ct0 + 1): the first
// segment's end state through the maps of the segments between, S <- M S + C,
// by all four waves.  Wave w computes the rows 32 w .. (k-step w of the next
// product) of both tiles from its share of M, read once per workgroup, and the
// split state of every wave, exchanged through LDS (two buffers, one barrier a
// map); the operands of the next two maps are on their way.  The chain waves
// (0, 1) receive the state of their tile in S.
__device__ __forceinline__ void start_state(char *smem, int seg_len, const SegSlot &slot0, int seg,
                                            int ct0, int wave, int lane, f32x4 (&S)[4][2]) {
  f32x4 R[2][2];  // [tile][t]: rows of state tile 2 wave + t
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int t = 0; t < 2; ++t)
      R[j][t] = *reinterpret_cast<const f32x4 *>(slot0.tile(ct0 + j, lane) + (2 * wave + t) * 1024);
  struct Operands {
    u32x4 mh[2][4], ml[2][4];
    f32x4 C[2][2];
  };
  auto request = [&](Operands &o, int m) {
    m = m < seg ? m : seg - 1;
    const SegSlot sl{slot0.base + static_cast<size_t>(m) * seg_len * slot0.step, slot0.step};
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int jb = 0; jb < 4; ++jb) {
        o.mh[t][jb] = *reinterpret_cast<const u32x4 *>(sl.frag(2 * wave + t, jb, 0, lane));
        o.ml[t][jb] = *reinterpret_cast<const u32x4 *>(sl.frag(2 * wave + t, jb, 1, lane));
      }
#pragma unroll
      for (int j = 0; j < 2; ++j)
        o.C[j][t] = *reinterpret_cast<const f32x4 *>(sl.tile(ct0 + j, lane) + (2 * wave + t) * 1024);
    }
  };
  auto apply = [&](Operands &o, int m) {
    char *const buf = smem + (m & 1) * 16384 + lane * 16;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      u32x4 hi, lo;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        uint32_t h0, h1, l0, l1;
        split2_rne(R[j][t][0], R[j][t][1], h0, l0);
        split2_rne(R[j][t][2], R[j][t][3], h1, l1);
        hi[2 * t] = h0;
        hi[2 * t + 1] = h1;
        lo[2 * t] = l0;
        lo[2 * t + 1] = l1;
      }
      *reinterpret_cast<u32x4 *>(buf + (j * 4 + wave) * 2048) = hi;
      *reinterpret_cast<u32x4 *>(buf + (j * 4 + wave) * 2048 + 1024) = lo;
    }
    __syncthreads();
    f32x4 a[2][2], b[2][2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int t = 0; t < 2; ++t) a[j][t] = b[j][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 sh[2][2], sl[2][2];  // [ring][tile]
    auto read = [&](int jb) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        sh[jb & 1][j] = lds16(buf + (j * 4 + jb) * 2048);
        sl[jb & 1][j] = lds16(buf + (j * 4 + jb) * 2048 + 1024);
      }
    };
    read(0);
    read(1);
#pragma unroll
    for (int jb = 0; jb < 4; ++jb) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          a[j][t] = mfma_bf16(o.mh[t][jb], sh[jb & 1][j], a[j][t]);
          b[j][t] = mfma_bf16(o.mh[t][jb], sl[jb & 1][j], b[j][t]);
        }
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int t = 0; t < 2; ++t) b[j][t] = mfma_bf16(o.ml[t][jb], sh[jb & 1][j], b[j][t]);
      __builtin_amdgcn_sched_barrier(0);
      if (jb < 2) read(jb + 2);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int t = 0; t < 2; ++t) R[j][t] = o.C[j][t] + (a[j][t] + b[j][t]);
  };
  if (seg > 1) {
    Operands p, q;
    request(p, 1);
    request(q, 2);
    // (straight-line pairs with one exit test, so that the waits at the loop
    // head cover exactly the set in use)
    int m = 1;
    for (; m + 2 <= seg; m += 2) {
      apply(p, m);
      request(p, m + 2);
      apply(q, m + 1);
      request(q, m + 3);
    }
    if (m < seg) apply(p, m);
  }
  char *const all = smem + OutLds::Q + lane * 16;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int t = 0; t < 2; ++t) *reinterpret_cast<f32x4 *>(all + (j * 8 + 2 * wave + t) * 1024) = R[j][t];
  __syncthreads();
  if (wave < 2) {
#pragma unroll
    for (int x = 0; x < 8; ++x) S[x >> 1][x & 1] = lds4f(all + (wave * 8 + x) * 1024);
  }
}
static_assert(OutLds::Q >= 32768 && OutLds::Q + 16384 <= kScanLds, "start_state's exchange");

// A segment with its output: 32 state columns (quarter `part`) by two chain
// waves, operands staged and output computed by two helper waves.  seg: the
// segment's number; slot0: slot of the sequence's first segment.
__device__ __forceinline__ void out_unit(const ScanArgs &A, char *smem, const Segment &sg, int seg, int seg_len,
                                         bool last, const SegSlot &slot0, size_t sbase, int h,
                                         int hq, int part) {
  const Heads &H = A.H;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int col0 = kOutCols * part;
  Chain c;
  if (seg > 0) start_state(smem, seg_len, slot0, seg, 2 * part, wave, lane, c.S);
  if (wave < 2) {
    const int ct = 2 * part + wave;
    const int vcol = col0 + 4 * wave + 8 * (r16 >> 2) + (r16 & 3);
    const size_t at = sbase + vcol * kDK + 8 * g;
    c.init<OutLds>(ct, lane);
    if (seg == 0) {
#pragma unroll
      for (int x = 0; x < 8; ++x)
        c.S[x >> 1][x & 1] =
            A.state != nullptr && sg.nch > 0
                ? __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(
                      A.state + at + 32 * (x >> 1) + 4 * (x & 1)))
                : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if (sg.nch > 0) {
      c.load_t(sg, 0);
      __syncthreads();  // the first chunk's operands are in LDS
      for (int i = 0; i < sg.nch; i += 2) {
        c.step<OutLds, 0>(smem, sg, i);
        __syncthreads();
        if (i + 1 < sg.nch) {
          c.step<OutLds, 1>(smem, sg, i + 1);
          __syncthreads();
        }
      }
    }
    if (last) {
#pragma unroll
      for (int x = 0; x < 8; ++x)
        __builtin_nontemporal_store(c.S[x >> 1][x & 1],
                                    reinterpret_cast<f32x4 *>(A.new_state + at + 32 * (x >> 1) + 4 * (x & 1)));
    } else if (seg == 0) {
      store_tile(c.S, slot0.tile(ct, lane));
    }
  } else if (sg.nch > 0) {
    // ---- helper wave: stages the operands, computes the output of the
    // token tiles mb0, mb0 + 1 ----
    const int ht = tid - 128;
    const int mb0 = 2 * (wave & 1);
    const uint32_t qk_stride = static_cast<uint32_t>(H.qk) * (kDK * 2);
    const uint32_t v_stride = static_cast<uint32_t>(H.v) * (kDV * 2);
    const int krow = ht >> 4;
    Stage<OutLds, 128, kOutCols> st;
    u32x4 qr[8], pr[2][2];
    f32x4 O[2][2];  // [token tile][column tile]
    auto issue_q = [&](int i) {
      const auto rq = buf_rsrc(A.q + (sg.start(i) * H.qk + hq) * kDK, sg.len(i) * qk_stride);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        qr[j] = buf_load16(rq, static_cast<uint32_t>(krow + 8 * j) * qk_stride + (ht & 15) * 16);
    };
    auto put_q = [&]() {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int row = krow + 8 * j;
        *reinterpret_cast<u32x4 *>(smem + OutLds::Q + row * 256 + 16 * ((ht & 15) ^ (row & 15))) = qr[j];
      }
    };
    auto issue_p = [&](int i) {  // P of chunk i, straight to the registers that use it
      const auto rr = buf_rsrc(sg.rec + i * sg.rec_step, kRecBytes);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const int mb = mb0 + m, x = mb < 2 ? mb : 2 * mb - 2;
        pr[m][0] = buf_load16(rr, kRecP + x * 1024 + lane * 16);
        // (tiles 0 and 1 see the tokens 0..31 only; their second fragment is not used)
        pr[m][1] = buf_load16(rr, kRecP + (mb0 ? x + 1 : x) * 1024 + lane * 16);
      }
    };
    auto out_state = [&](int par) {  // O = e^G (q S)^T
      u32x4 sh[2][4], qf[2][4];
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          sh[j][kk] = lds16(smem + OutLds::S + j * 4096 + kk * 1024 + lane * 16);
          qf[j][kk] = lds16(smem + OutLds::Q + (16 * (mb0 + j) + r16) * 256 + 16 * ((4 * kk + g) ^ r16));
        }
      float e[2];
#pragma unroll
      for (int m = 0; m < 2; ++m)
        e[m] = *reinterpret_cast<const float *>(smem + OutLds::E + par * kLEBytes + (16 * (mb0 + m) + r16) * 4);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int j = 0; j < 2; ++j) O[m][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int j = 0; j < 2; ++j) O[m][j] = mfma_bf16(sh[j][kk], qf[m][kk], O[m][j]);
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) O[m][j][r] *= e[m];
    };
    auto out_store = [&](int i) {  // o^T = scale (O + (P v_new)^T) of chunk i
      u32x4 n[2][2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
          n[j][jj] = lds16(smem + OutLds::N + j * 2048 + jj * 1024 + lane * 16);
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int j = 0; j < 2; ++j) O[m][j] = mfma_bf16(n[j][0], pr[m][0], O[m][j]);
      if (mb0) {
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int j = 0; j < 2; ++j) O[m][j] = mfma_bf16(n[j][1], pr[m][1], O[m][j]);
      }
      const auto ro = buf_rsrc(A.out + (sg.start(i) * H.v + h) * kDV, sg.len(i) * v_stride);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const u32x4 o = {pk_bf16(A.scale * O[m][0][0], A.scale * O[m][0][1]),
                         pk_bf16(A.scale * O[m][0][2], A.scale * O[m][0][3]),
                         pk_bf16(A.scale * O[m][1][0], A.scale * O[m][1][1]),
                         pk_bf16(A.scale * O[m][1][2], A.scale * O[m][1][3])};
        __builtin_amdgcn_raw_buffer_store_b128(
            o, ro, static_cast<uint32_t>(16 * (mb0 + m) + r16) * v_stride + (col0 + 8 * g) * 2, 0, 0);
      }
    };
    st.issue(A, sg, 0, ht, h, hq, col0, true);
    issue_q(0);
    st.put(smem, 0, ht);
    st.issue(A, sg, 1, ht, h, hq, col0, true);
    __syncthreads();
    for (int i = 0; i < sg.nch; ++i) {
      put_q();
      issue_q(i + 1);
      st.put(smem, (i + 1) & 1, ht);
      st.issue(A, sg, i + 2, ht, h, hq, col0, true);
      if (i > 0) out_store(i - 1);
      issue_p(i);
      __syncthreads();  // B
      out_state(i & 1);
      __syncthreads();  // A
    }
    out_store(sg.nch - 1);
  }
}

// Unit `id` of a launch of scan_chain_kernel: a segment's output or, `map`, a
// share of a middle segment's map.
template <bool SECOND>
__device__ __forceinline__ void chain_unit(const ScanArgs &A, char *smem, int id, bool map, int seg_len) {
  const Heads &H = A.H;
  // the same four workgroups for each slot: the quarters of the columns, or the
  // two halves of the offset (0, 1) and of the linear part (2, 3) of a map
  const int h = id % H.v, part = (id / H.v) & 3;
  const int hq = h / H.ratio;
  int s = id / H.v >> 2, seg = 0;
  if (SECOND || map) {
    if (seg_len == 0) return;
    // slot number -> (sequence, segment): nseg - 1 segments each here, nseg - 2
    // maps; lane n looks at sequence n (at most 64 are cut)
    const int j = s;
    const int lane = threadIdx.x & 63;
    int n = 0;
    if (lane < A.N) {
      const int lo = load_cu(A.cu, A.cu64, lane, A.T), hi = load_cu(A.cu, A.cu64, lane + 1, A.T);
      n = hi > lo ? (hi - lo + kChunk - 1) / kChunk : 0;
      if (A.offsets != nullptr) {
        const int m = A.offsets[lane + 1] - A.offsets[lane];
        n = m < n ? (m > 0 ? m : 0) : n;
      }
    }
    n = (n + seg_len - 1) / seg_len - (SECOND ? 1 : 2);
    n = n < 0 ? 0 : n;
    int incl = n;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(incl, off);
      if (lane >= off) incl += y;
    }
    const unsigned long long above = __ballot(incl > j);
    if (above == 0) return;
    s = __builtin_ctzll(above);
    seg = 1 + j - (__builtin_amdgcn_readlane(incl, s) - __builtin_amdgcn_readlane(n, s));
  }
  s = __builtin_amdgcn_readfirstlane(s);
  seg = __builtin_amdgcn_readfirstlane(seg);
  Segment sg;
  const int bos = __builtin_amdgcn_readfirstlane(load_cu(A.cu, A.cu64, s, A.T));
  sg.eos = __builtin_amdgcn_readfirstlane(load_cu(A.cu, A.cu64, s + 1, A.T));
  sg.eos = sg.eos < bos ? bos : sg.eos;
  int c0 = 0, nch = (sg.eos - bos + kChunk - 1) / kChunk;
  if (A.offsets != nullptr) {
    c0 = __builtin_amdgcn_readfirstlane(A.offsets[s]);
    const int n = __builtin_amdgcn_readfirstlane(A.offsets[s + 1]) - c0;
    nch = n < nch ? (n > 0 ? n : 0) : nch;
  }
  const int first = seg * seg_len;  // the segment's first chunk of the sequence
  const int left = nch - first;
  const bool last = seg_len == 0 || left <= seg_len;
  sg.nch = last ? left : seg_len;
  sg.bos = bos + first * kChunk;
  sg.rec_step = static_cast<size_t>(H.v) * kRecStride;
  sg.rec = A.rec + (static_cast<size_t>(c0 + first) * H.v + h) * kRecStride;
  const size_t step = static_cast<size_t>(H.v) * kSegSlotBytes;
  const SegSlot slot0{A.seg + (static_cast<size_t>(c0) * H.v + h) * kSegSlotBytes, step};
  if (map)
    map_unit(A, smem, sg, SegSlot{slot0.base + static_cast<size_t>(first) * step, step}, h, hq, part & 1, part >> 1);
  else
    out_unit(A, smem, sg, seg, seg_len, last, slot0, (static_cast<size_t>(s) * H.v + h) * kDV * kDK, h, hq, part);
}

// Launch 1 (SECOND = false): the first segment of every (sequence, v-head)
// with its output, and the maps of the middle segments.  Launch 2: the other
// segments with their output.  LOOP (launch 1 without maps, which would spill):
// the output units by a capped grid (PrefillPlan::scan_grid), a workgroup taking
// every out_grid-th one.
template <bool SECOND, bool LOOP>
__global__ __launch_bounds__(kScanThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void scan_chain_kernel(ScanArgs A) {
  __shared__ __align__(16) char smem[kScanLds];
  const Heads &H = A.H;
  const CoveredRows rows = covered_rows(A.cu, A.cu64, A.N, A.T);
  if (A.offsets != nullptr && __builtin_amdgcn_readfirstlane(A.offsets[A.N + 1]))
    return;  // the sequential kernel owns the batch
  const bool map = !SECOND && !LOOP && static_cast<int>(blockIdx.x) >= A.out_grid;
  int id = map ? blockIdx.x - A.out_grid : blockIdx.x;
  const int seg_len = A.seg_len != nullptr ? __builtin_amdgcn_readfirstlane(*A.seg_len) : 0;
  for (;;) {
    chain_unit<SECOND>(A, smem, id, map, seg_len);
    if (!LOOP) break;
    id += A.out_grid;
    if (id >= A.out_units) break;
    __syncthreads();  // the unit's LDS is free
  }
  if (!SECOND && !map) zero_rows_outside(A.out, rows, A.T, H.v, blockIdx.x, A.out_grid);
}

int scan_launch(const uint16_t *q, const uint16_t *k, const uint16_t *v, const float *state,
                const float *A_log, const uint16_t *a, const float *dt_bias, const uint16_t *b,
                const void *cu, int cu64, int N, int T, const Heads &H, const PrefillLayout &L,
                const PrefillPlan &P, float scale, uint16_t *out, float *new_state, char *ws,
                hipStream_t stream, const char *what) {
  int4 *chunks = reinterpret_cast<int4 *>(ws + L.chunks);
  int *offsets = reinterpret_cast<int *>(ws + L.offsets);
  int *status = reinterpret_cast<int *>(ws + L.status);
  char *rec = ws + L.w;
  const OneSeq one{P.single ? cu : nullptr, cu64, T};
  const SelfIndex si{P.self_index ? cu : nullptr, cu64, N, T, P.choose, -1, P.form,
                     chunks, offsets, status, nullptr, 0, P.scan_more};
  hipLaunchKernelGGL(scan_intra_kernel, dim3(static_cast<unsigned>(chunk_head_grid(L.nt_max, H))),
                     dim3(256), 0, stream, q, k, A_log, a, dt_bias, b, chunks, one, L.nt_max, H, si,
                     rec);
  if (int rc = check_launch(what)) return rc;
  if (P.choose != 0 && P.self_index) {
    if (int rc = recurrent_launch(q, k, v, state, A_log, a, dt_bias, b, cu, cu64, N, T, 0,
                                  offsets + N + 1, nullptr, H, scale, out, new_state, stream,
                                  P.seq_variant, what))
      return rc;
  }
  const long long out_units = static_cast<long long>(N) * H.v * 4;
  const ScanArgs A{q, k, v, state, new_state, out, cu, cu64, N, T,
                   P.single ? nullptr : offsets, rec, ws + L.ht,
                   P.scan_more > 0 ? offsets + N + 2 : nullptr,
                   static_cast<int>(out_units), static_cast<int>(P.scan_grid), H, scale};
  const long long maps = P.scan_more > 1 ? static_cast<long long>(P.scan_more - 1) * H.v * 4 : 0;
  const auto first = P.scan_grid < out_units ? scan_chain_kernel<false, true> : scan_chain_kernel<false, false>;
  hipLaunchKernelGGL(first, dim3(static_cast<unsigned>(P.scan_grid + maps)), dim3(kScanThreads), 0,
                     stream, A);
  if (int rc = check_launch(what)) return rc;
  if (P.scan_more > 0) {
    hipLaunchKernelGGL((scan_chain_kernel<true, false>),
                       dim3(static_cast<unsigned>(static_cast<long long>(P.scan_more) * H.v * 4)),
                       dim3(kScanThreads), 0, stream, A);
    return check_launch(what);
  }
  return GDN_OK;
}

}  // namespace gdn
