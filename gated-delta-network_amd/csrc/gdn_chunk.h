// Device code shared by the chunked prefill kernels (gdn_prefill.hip and
// gdn_scan.hip): the chunk table's readers, the path choice, the mapping of
// workgroups to (chunk, v-head), and the triangular inverse of a chunk.
#pragma once

#include "gdn_device.h"

namespace gdn {

// LDS row strides (elements), padded by 16 bytes against bank conflicts.
constexpr int kStrideK = 136;  // bf16 [64][128] tiles
constexpr int kStrideT = 72;   // bf16 [*][64]   tiles

// Maximum of x over the workgroup into *dst (LDS, initially <= every x): a
// butterfly within each wave, then one LDS atomic per wave (1024 atomics on
// one word serialize: ~2 us).
__device__ __forceinline__ void block_max_into(int x, int *dst) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const int y = __shfl_xor(x, off);
    x = y > x ? y : x;
  }
  if ((threadIdx.x & 63) == 0) atomicMax(dst, x);
}

// Sum of x over the workgroup into *dst (LDS, initially 0), the same way.
__device__ __forceinline__ void block_sum_into(int x, int *dst) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
  if ((threadIdx.x & 63) == 0) atomicAdd(dst, x);
}

// The path the device picks (choose != 0, set on the host): sequential (true)
// or chunks, from the batch's longest sequence and chunk count (the form the
// chunks would take: `form` 0 / 1 as set, else t_form_wins).
__device__ __forceinline__ bool device_picks_sequential(int choose, int rec_max, int longest,
                                                        int chunks, int N, int T, int hv,
                                                        int form) {
  if (choose == 1) return longest <= rec_max;
  if (choose < 2) return false;
  const float L = static_cast<float>(longest), fhv = static_cast<float>(hv);
  const float g = static_cast<float>(N) * fhv;
  const float by_seq = choose == 2 ? cost_by_token(L, static_cast<float>(T), fhv, g)
                                   : cost_by_block(L, g);
  const float fnt = static_cast<float>(chunks);
  const bool t = form == 1 ||
                 (form != 0 && t_form_wins(fnt, ceilf(L / kChunk), state_units(static_cast<float>(N), fhv)));
  return by_seq + kSeqChoiceMargin <= cost_by_chunks_form(L, fnt, fhv, static_cast<float>(N), t);
}

// Sum over the wave (in every lane): DPP within each row of 16 lanes, then
// the four row sums through readlane.
__device__ __forceinline__ int wave_sum(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x141, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x140, 0xf, 0xf, false);
  return __builtin_amdgcn_readlane(x, 0) + __builtin_amdgcn_readlane(x, 16) +
         __builtin_amdgcn_readlane(x, 32) + __builtin_amdgcn_readlane(x, 48);
}

// Fused scan: the segment length (segment_choice) for sequences of n chunks
// each (lane s of the one wave that calls it: sequence s, at most 64).
__device__ __forceinline__ int segment_length(int n, int max_more, int hv) {
  return segment_choice(static_cast<int>(wave_max(static_cast<float>(n))), max_more, hv,
                        [n](auto f) { return wave_sum(f(n)); });
}

// Chunk c of the table; for a single sequence (one.cu != nullptr) there is no
// table and the entry is computed from the sequence's bounds.
__device__ __forceinline__ int4 chunk_info(const int4 *chunks, int c, const OneSeq &one) {
  if (one.cu != nullptr) {
    int bos, eos;
    one_seq_bounds(one, bos, eos);
    const int start = bos + c * kChunk, rest = eos - start;
    return rest > 0 ? make_int4(0, start, rest < kChunk ? rest : kChunk, c) : make_int4(-1, 0, 0, 0);
  }
  // the same entry in every lane: keep it in SGPRs (buffer descriptors built
  // from it are then uniform, with no per-lane loop around each load)
  const int4 e = chunks[c];
  return make_int4(__builtin_amdgcn_readfirstlane(e.x), __builtin_amdgcn_readfirstlane(e.y),
                   __builtin_amdgcn_readfirstlane(e.z), __builtin_amdgcn_readfirstlane(e.w));
}

// ---------------------------------------------------------------------------
// 1b. the chunk table built inside the intra kernel (several sequences, at
// most kSelfIndexMax, and an intra grid of at most kSelfIndexMaxGrid
// workgroups; gdn_common.h): each workgroup scans cu_seqlens itself -- one
// sequence per thread, a prefix sum of the chunk counts in LDS -- and finds
// its own chunk by binary search; workgroup 0 writes offsets, the chunk
// count and the flags, and the workgroup of v-head 0 of each chunk slot its
// chunk-table entry, for the state and output kernels.  A batch then needs no
// index launch (~4.7 us): the intra kernel is the first launch, the path the
// device picks included (the sequential kernel runs after it and reads the
// flag).  Same results as the index kernel, entry by entry.
// ---------------------------------------------------------------------------
struct SelfIndex {
  const void *cu;  // nullptr: the index kernel built the table
  int cu64, N, T, choose, rec_max, form;
  int4 *chunks;
  int *offsets;
  int *status;     // per-sequence contract bits (also for one sequence)
  int *early;      // one sequence: words of the two-segment scan's early output,
  int n_early;     // zeroed by the first workgroups (nullptr: none)
  int max_more;    // fused scan: segment_length's bound (0: no sequence is cut)
};
constexpr int kSelfIndexLds = 3 * kSelfIndexMax * 4 + 16 * 4;

struct SelfIndexed {
  int nt, form;
};

__device__ __forceinline__ SelfIndexed self_index(char *smem, const SelfIndex &si, int nt_max,
                                                  int hv) {
  int *const s_incl = reinterpret_cast<int *>(smem);
  int *const s_bos = s_incl + kSelfIndexMax;
  int *const s_eos = s_bos + kSelfIndexMax;
  int *const s_red = s_eos + kSelfIndexMax;  // longest, most chunks, wave totals [4..7]
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int N = si.N, T = si.T;
  int n = 0, len = 0;
  if (tid < 2) s_red[tid] = 0;
  if (tid < N) {
    const long long lo = raw_cu(si.cu, si.cu64, tid), hi = raw_cu(si.cu, si.cu64, tid + 1);
    if (blockIdx.x == 0) si.status[tid] = cu_status_bits(lo, hi, T);
    const int bos = static_cast<int>(lo < 0 ? 0 : lo > T ? T : lo);
    int eos = static_cast<int>(hi < 0 ? 0 : hi > T ? T : hi);
    eos = eos < bos ? bos : eos;
    len = eos - bos;
    n = (len + kChunk - 1) / kChunk;
    s_bos[tid] = bos;
    s_eos[tid] = eos;
  }
  int incl = n;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(incl, off);
    if (lane >= off) incl += y;
  }
  if (lane == 63) s_red[4 + wv] = incl;
  __syncthreads();
  for (int w = 0; w < wv; ++w) incl += s_red[4 + w];
  s_incl[tid] = incl;
  block_max_into(len, &s_red[0]);
  block_max_into(n, &s_red[1]);
  __syncthreads();
  const int total = s_incl[N - 1];
  const bool sequential = device_picks_sequential(si.choose, si.rec_max, s_red[0], total, N, T,
                                                  hv, si.form);
  const int nt = sequential ? 0 : (total < nt_max ? total : nt_max);
  const int form = (si.form == 0 || si.form == 1)
                       ? si.form
                       : (t_form_wins(static_cast<float>(nt), static_cast<float>(s_red[1]),
                                      state_units(static_cast<float>(N), static_cast<float>(hv)))
                              ? 1
                              : 0);
  if (blockIdx.x == 0) {
    if (tid < N) {
      const int first = sequential ? 0 : s_incl[tid] - n;
      si.offsets[tid] = first < nt_max ? first : nt_max;
    }
    if (tid == 0) {
      si.offsets[N] = nt;
      si.offsets[N + 1] = sequential ? 1 : 0;
      si.offsets[N + 2] = form;
    }
    if (si.max_more > 0 && tid < 64) {  // (N <= 64)
      const int seg = segment_length(n, si.max_more, hv);
      if (tid == 0) si.offsets[N + 2] = seg;
    }
  }
  return SelfIndexed{nt, form};
}

// Entry c of the chunk table from the self index's LDS arrays.
__device__ __forceinline__ int4 self_chunk(const char *smem, int N, int c, int nt) {
  if (c >= nt) return make_int4(-1, 0, 0, 0);
  const int *const s_incl = reinterpret_cast<const int *>(smem);
  const int *const s_bos = s_incl + kSelfIndexMax;
  const int *const s_eos = s_bos + kSelfIndexMax;
  int lo = 0, hi = N - 1;  // first sequence with s_incl > c
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (s_incl[mid] > c) hi = mid; else lo = mid + 1;
  }
  const int local = c - (lo == 0 ? 0 : s_incl[lo - 1]);
  const int start = s_bos[lo] + local * kChunk;
  const int len = s_eos[lo] - start < kChunk ? s_eos[lo] - start : kChunk;
  return make_int4(lo, start, len, local);
}

// Workgroup id -> (chunk c, v-head h) for the per-(chunk, head) kernels, so
// that the `ratio` v-heads reading one q/k head of one chunk are dispatched
// back to back on the same XCD: ids are dealt round-robin over the 8 XCDs,
// so id = 8 s + x runs on XCD x, and consecutive s on one XCD take the
// v-heads of one (chunk, q/k head) pair -- the second and later ones find
// that chunk's q/k rows in the XCD's L2.  Pairs are numbered P = 8 p + x in
// chunk-major order.  False for ids past the last pair.
__device__ __forceinline__ bool chunk_head_of(int id, int nt, const Heads &H, int &c, int &h) {
  const int x = id & 7, sl = id >> 3;
  const int p = sl / H.ratio, r = sl - p * H.ratio;
  const long long P = 8LL * p + x;
  if (P >= static_cast<long long>(nt) * H.qk) return false;
  c = static_cast<int>(P / H.qk);
  h = static_cast<int>(P - static_cast<long long>(c) * H.qk) * H.ratio + r;
  return true;
}

constexpr int kABlk = 16 * 20;  // one 16x16 f32 block of A, rows padded to 20

// Block (ib, jb), jb <= ib, of the compact lower-triangular A.
__device__ __forceinline__ int ablk(int ib, int jb) { return (ib * (ib + 1) / 2 + jb) * kABlk; }

// A = strictly-lower(beta_i exp(G_i - G_j) K K^T) of one chunk from its K
// rows in LDS (row-major, stride kStrideK), as the ten lower 16x16 blocks of
// sA (ablk; rows padded to 20 floats).  Wave w computes blocks w, w + 4 and
// (waves 0, 1) w + 8, the three as independent MFMA chains side by side (one
// block at a time left each wave waiting on its LDS reads and a 4-deep MFMA
// chain per block).  G_i - G_j <= 0 for every kept entry (g <= 0); the clamp
// keeps the others finite; exp is the hardware exp2 of x log2(e) (a few
// 2^-24 relative, far below the split-bf16 products' 2^-17).
__device__ __forceinline__ void build_A(const uint16_t *sK, float *sA, const float *sG,
                                        const float *sBeta, int len, int wave, int lane) {
  const int r16 = lane & 15, g = lane >> 4, kg = 8 * g;
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  int mb[3], nb[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    int t = wv + 4 * q;
    t = t < 10 ? t : 9;  // waves 2, 3 repeat block 9 as their third (not stored)
    // t = 0..9 -> (mb, nb) = (3,3) (3,2) (3,1) (3,0) (2,2) (2,1) (2,0) (1,1) (1,0) (0,0)
    mb[q] = t < 4 ? 3 : t < 7 ? 2 : t < 9 ? 1 : 0;
    nb[q] = t < 4 ? 3 - t : t < 7 ? 6 - t : t < 9 ? 8 - t : 0;
  }
  f32x4 acc[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) acc[q] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const u32x4 af = *reinterpret_cast<const u32x4 *>(&sK[(16 * mb[q] + r16) * kStrideK + 32 * kk + kg]);
      const u32x4 bf = *reinterpret_cast<const u32x4 *>(&sK[(16 * nb[q] + r16) * kStrideK + 32 * kk + kg]);
      acc[q] = mfma_bf16(af, bf, acc[q]);
    }
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    if (q == 2 && wv >= 2) break;
    const float Gj = sG[16 * nb[q] + r16];
    const f32x4 Gi = *reinterpret_cast<const f32x4 *>(&sG[16 * mb[q] + 4 * g]);
    const f32x4 Bi = *reinterpret_cast<const f32x4 *>(&sBeta[16 * mb[q] + 4 * g]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * mb[q] + 4 * g + r, j = 16 * nb[q] + r16;
      const float d = __builtin_amdgcn_exp2f(fminf(Gi[r] - Gj, 0.f) * 1.44269504088896341f);
      const float e = Bi[r] * d * acc[q][r];
      sA[ablk(mb[q], nb[q]) + (4 * g + r) * 20 + r16] = (i > j && i < len) ? e : 0.f;
    }
  }
}

// Diagonal blocks D_w = (I + A_ww)^-1 in place of A_ww: wave w, lane j < 16
// solves column j, column-oriented (each solved x_m is applied to all later
// rows at once, so the serial chain is one FMA per row).  Every read of A_ww
// precedes the writes in the wave's program order.
__device__ __forceinline__ void diag_inverse(float *sA, int wave, int lane) {
  if (lane < 16) {
    float *Aw = sA + ablk(wave, wave);
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = i == lane ? 1.f : 0.f;
#pragma unroll
    for (int m = 0; m < 15; ++m) {
      const float xm = x[m];
#pragma unroll
      for (int i = m + 1; i < 16; ++i) x[i] -= Aw[i * 20 + m] * xm;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) Aw[i * 20 + lane] = x[i];
  }
}

// Block column j = wave of T = (I + A)^-1 from the ten lower blocks of sA
// (A, with the diagonal inverses D_i in place of A_ii): T_jj = D_j and, for
// i > j, T_ij = -D_i sum_{j<=m<i} A_im T_mj, on split-bf16 16x16x16 MFMAs (a
// result tile's layout is the next product's B-operand layout, so the column
// stays in registers).  Tc[i] = T_ij in MFMA result order (lane holds rows
// 4g..4g+3, column r16); zero above the diagonal.
__device__ __forceinline__ void t_column(const float *sA, int wave, int g, int r16,
                                         f32x4 (&Tc)[4]) {
  const int j = wave;
  u32x2 Th[4], Tl[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i < j) {  // above the diagonal
      Tc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      Th[i] = Tl[i] = u32x2{0u, 0u};
    } else if (i == j) {  // T_jj = D_j
      const float *d = &sA[ablk(i, i) + (4 * g) * 20 + r16];
      Tc[i] = f32x4{d[0], d[20], d[40], d[60]};
      split4(Tc[i], Th[i], Tl[i]);
    } else {
      // Z = -sum_{j<=m<i} A_im T_mj, then T_ij = D_i Z
      f32x4 Z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int m = 0; m < i; ++m) {
        if (m < j) continue;
        const f32x4 la = *reinterpret_cast<const f32x4 *>(&sA[ablk(i, m) + r16 * 20 + 4 * g]);
        u32x2 lh, ll;
        split4(-la, lh, ll);
        Z = mfma16_x3(lh, ll, Th[m], Tl[m], Z);
      }
      const f32x4 d4 = *reinterpret_cast<const f32x4 *>(&sA[ablk(i, i) + r16 * 20 + 4 * g]);
      u32x2 dh, dl, zh, zl;
      split4(d4, dh, dl);
      split4(Z, zh, zl);
      Tc[i] = mfma16_x3(dh, dl, zh, zl, f32x4{0.f, 0.f, 0.f, 0.f});
      split4(Tc[i], Th[i], Tl[i]);
    }
  }
}

}  // namespace gdn
