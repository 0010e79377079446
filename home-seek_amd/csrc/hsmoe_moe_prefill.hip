// Routed-expert SwiGLU FFN for many tokens (prefill): a grouped GEMM over the
// experts the tokens select, each expert's weights streamed from HBM once per
// chunk of its tokens (gate/up: up to 32, or 64 for an expert with more than
// 32; down: up to 32, or 64 in the wide kernels).
//
// Restates FusedMoEFFN._forward_legacy at B > 8 and the FP4 grouped route of
// fused_expert_ffn_triton (fused_moe.py:269-380, 458-551) plus the shared
// expert add of _forward_ffn (engine.py:1530-1536), with the arithmetic of
// the decode kernels:
//   gate = x W1^T, up = x W3^T (fp32 accumulation of exact bf16 products);
//   a = w * min(g,L) sigmoid(min(g,L)) clamp(u,-L,L);  y = a W2^T
//   out[t] = sum_j y[t, j] (slot order) + shared(t)
// W = bf16(dequant(FP4)) decoded in registers; the activation enters the down
// GEMM as a bf16 hi + lo pair.  Unlike the reference's dense union GEMM
// (every token through every selected expert), only the (token, expert) pairs
// that routing selects are computed.
//
// Launches (no host synchronisation; "wide" below for the form that calls with
// many pairs per expert take instead of gate_up and down):
//   group    workgroup e buckets the pairs (t, j) routed to expert e, in (t, j)
//            order (stable, deterministic); one more workgroup places the
//            shared expert's M pairs.  Each bucket is cut into gate/up chunks
//            (<= 32 pairs, or <= 64 for a bucket of more than 32, those first)
//            and into down chunks of <= 32 pairs.
//   gate_up  grid (chunk, 64-row block of I): wave w takes rows
//            +16w..+16 of W1 and W3 over all of D in K-chunks of 256 columns.
//            While chunk kc is multiplied, the token tile of kc+1 is in flight
//            to registers (then LDS) and the weights of kc+2 to a third
//            register buffer (a 64-pair chunk: no weights ahead, for the
//            registers of its four token tiles).  Writes the weighted
//            activation (hi, lo).
//   down     grid (chunk, 128-row block of D), same pipeline over W2 (32 rows
//            per wave) with the activation tile (hi and lo planes); writes one
//            fp32 partial row per pair (no atomics).
//   wide     the same two passes for the shared expert's chunks and those of
//            routed experts with more than 32 pairs, on 32-row tiles (beside
//            gate_up and down, which then take the other experts).
//   combine  out[t] = partials of t's pairs in slot order, then the shared one.
// The grids are sized for the most chunks the routing can produce; workgroups
// past the actual count (read from the workspace) exit at once.
#include <math.h>

#include "hsmoe_common.h"
#include "hsmoe_internal.h"
#include "hsmoe_tiles.h"

namespace hsmoe {
namespace {

constexpr int kThreads = 256;
constexpr int kChunk = 32;        // tokens per chunk (two 16-token MFMA tiles)
constexpr int kBigChunk = 64;     // tokens per chunk of an expert with more than kChunk pairs
constexpr int kGuRT = 1;          // 16-row tiles per wave, gate/up (W1 and W3)
constexpr int kDnRT = 2;          // 16-row tiles per wave, down (W2)
constexpr int kGuRows = 64 * kGuRT;  // weight rows per workgroup
constexpr int kDnRows = 64 * kDnRT;
constexpr int kCols = 256;        // columns per K-chunk (2 steps of 128)
constexpr int kPad = 8;           // bf16 elements of padding per LDS row
constexpr int kMaxPairs = 12288;  // m * top_k per call (LDS of the group kernel)
constexpr int kMaxExperts = 1024;

struct Header {
  int n_gu;   // gate/up chunks: the shared expert's, then the routed experts' (big ones' first)
  int n_dn;   // down chunks: the shared expert's, then the routed experts'
  int n_big;  // gate/up chunks of the shared expert and the big routed experts
};

struct PrefillParams {
  const uint16_t* x;       // bf16 [m, d]
  const int64_t* idx;      // [m, top_k]
  const float* wts;        // [m, top_k]
  const uint64_t* table;   // [n_experts][6]
  const uint64_t* shared;  // [6] or null
  Header* hdr;
  int* pair_tok;           // [max_pairs] token of pair p
  float* pair_w;           // [max_pairs] routing weight of pair p
  int* pidx;               // [m][top_k + 1] pair of (t, j); j = top_k: shared; -1 = none
  int* chunk_e;            // [max_chunks] expert (n_experts = shared)
  int* chunk_p0;           // [max_chunks] first pair
  int* chunk_n;            // [max_chunks] pairs in the chunk
  int* dn_e;               // [max_chunks] down chunks: every expert's pairs in chunks of kChunk
  int* dn_p0;
  int* dn_n;
  uint16_t* act_hi;        // bf16 [max_pairs][i]
  uint16_t* act_lo;        // bf16 [max_pairs][i]
  float* part;             // fp32 [max_pairs][d]
  float* out_f32;          // [m, d] or null
  uint16_t* out_bf16;      // [m, d] or null
  int n_experts;
  int m, d, i, top_k;
  int n_sh_gu, n_sh_dn;  // chunks of the shared expert's m pairs in either list
  int small, big_chunk;  // an expert of more than `small` pairs is cut into chunks of big_chunk
  int by_rows;           // wide kernels: every chunk placed on the XCDs by row block
  int wide;              // the first n_big gate/up chunks go to the wide kernels, in both passes
  float limit;
};

// ---------------------------------------------------------------- group
// Pairs per gate/up chunk of an expert with cnt pairs: an expert with more
// than p.small (kChunk) pairs is cut into chunks of kBigChunk, so that its W1 and W3
// are streamed half as often; big experts' chunks come first, so that the
// longer workgroups start first.  The down pass keeps chunks of kChunk (its
// token tile's size), in expert order: a second list (the wide kernels and what
// runs beside them take the gate/up list in both passes).
__device__ __forceinline__ int chunk_size(const PrefillParams& p, int cnt) {
  return cnt > p.small ? p.big_chunk : kChunk;
}

// Sum over the block of v (every thread passes its own value).
template <int kWaves>
__device__ __forceinline__ int block_sum(int v, int* s_red) {
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) v += __shfl_xor(v, off, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = v;
  __syncthreads();
  int t = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) t += s_red[w];
  return t;
}

// Workgroup e < n_experts places the pairs of expert e; workgroup n_experts
// writes the header, the shared expert's pairs and the slots of invalid ids.
// Every workgroup histograms the whole pair list in LDS, so the offsets of
// expert e (pairs and chunks of the experts before it) need no second pass.
// Within an expert, pairs keep (t, j) order: each wave counts, then places, the
// hits of its contiguous share of the list, ranked by ballots.  The shared
// expert's chunks come first in both lists: every token is in one of them, so
// its workgroups are the fullest, and they run under the routed stream (as
// launches of their own they took 25 MB of weights 60 + 40 us at m = 509).
template <int kGroupThreads>
__global__ void __launch_bounds__(kGroupThreads) prefill_group_kernel(PrefillParams p) {
  constexpr int kWaves = kGroupThreads / 64;
  __shared__ uint16_t s_e[kMaxPairs];  // expert of pair q, kNone: invalid id or absent expert
  __shared__ int s_cnt[kMaxExperts];
  __shared__ bool s_ok[kMaxExperts];  // expert e has a table entry
  __shared__ int s_red[kWaves];
  __shared__ int s_wc[kWaves];
  constexpr int kNone = 0xffff;
  const int E = p.n_experts, K = p.top_k, P = p.m * K, me = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // which experts have a table entry: one load per expert, not one per pair
  for (int e = threadIdx.x; e < E; e += kGroupThreads) {
    s_cnt[e] = 0;
    s_ok[e] = p.table[(int64_t)e * 6] != 0;
  }
  __syncthreads();
  // the pair ids, kIdBatch loads of a thread in flight at once
  constexpr int kIdBatch = 8;
  for (int q0 = threadIdx.x; q0 < P; q0 += kIdBatch * kGroupThreads) {
    int64_t ev[kIdBatch];
#pragma unroll
    for (int j = 0; j < kIdBatch; ++j) ev[j] = q0 + j * kGroupThreads < P ? p.idx[q0 + j * kGroupThreads] : -1;
#pragma unroll
    for (int j = 0; j < kIdBatch; ++j) {
      const int q = q0 + j * kGroupThreads;
      if (q >= P) break;
      const int64_t e = ev[j];
      const bool ok = e >= 0 && e < E && s_ok[e];
      s_e[q] = (uint16_t)(ok ? (int)e : kNone);
      if (ok) atomicAdd(&s_cnt[e], 1);
    }
  }
  __syncthreads();
  if (me == E) {
    int pairs = 0, chunks = 0, dchunks = 0, small = 0;
    for (int e = threadIdx.x; e < E; e += kGroupThreads) {
      pairs += s_cnt[e];
      chunks += (s_cnt[e] + chunk_size(p, s_cnt[e]) - 1) / chunk_size(p, s_cnt[e]);
      small += s_cnt[e] > 0 && s_cnt[e] <= p.small;
      dchunks += (s_cnt[e] + kChunk - 1) / kChunk;
    }
    pairs = block_sum<kWaves>(pairs, s_red);
    chunks = block_sum<kWaves>(chunks, s_red);
    dchunks = block_sum<kWaves>(dchunks, s_red);
    small = block_sum<kWaves>(small, s_red);
    if (threadIdx.x == 0) {
      p.hdr->n_gu = p.n_sh_gu + chunks;
      p.hdr->n_dn = p.n_sh_dn + dchunks;
      p.hdr->n_big = p.n_sh_gu + chunks - small;
    }
    for (int q = threadIdx.x; q < P; q += kGroupThreads)
      if (s_e[q] == kNone) p.pidx[(q / K) * (K + 1) + q % K] = -1;
    for (int t = threadIdx.x; t < p.m; t += kGroupThreads) {
      const int pos = pairs + t;
      p.pidx[t * (K + 1) + K] = p.shared ? pos : -1;
      if (!p.shared) continue;
      p.pair_tok[pos] = t;
      p.pair_w[pos] = 1.0f;
      if (t % kBigChunk == 0) {
        p.chunk_e[t / kBigChunk] = E;
        p.chunk_p0[t / kBigChunk] = pos;
        p.chunk_n[t / kBigChunk] = min(kBigChunk, p.m - t);
      }
      if (t % kChunk == 0) {
        p.dn_e[t / kChunk] = E;
        p.dn_p0[t / kChunk] = pos;
        p.dn_n[t / kChunk] = min(kChunk, p.m - t);
      }
    }
    return;
  }
  const int cnt = s_cnt[me];
  if (cnt == 0) return;  // uniform across the workgroup
  // chunks: the big experts' (expert order), then one per small expert (expert order)
  const bool big = cnt > p.small;
  int off = 0, choff = 0, dnoff = 0;
  for (int e = threadIdx.x; e < E; e += kGroupThreads) {
    const int c = s_cnt[e];
    if (e < me) off += c;
    if (e < me) dnoff += (c + kChunk - 1) / kChunk;
    if (c > p.small && (!big || e < me)) choff += (c + p.big_chunk - 1) / p.big_chunk;  // every big expert's chunks first
    else if (!big && e < me && c > 0) ++choff;
  }
  off = block_sum<kWaves>(off, s_red);
  choff = p.n_sh_gu + block_sum<kWaves>(choff, s_red);
  dnoff = p.n_sh_dn + block_sum<kWaves>(dnoff, s_red);
  const int cs = chunk_size(p, cnt);
  // this wave's share of the list: its hits, then their places
  const int per = (P + 64 * kWaves - 1) / (64 * kWaves) * 64;
  const int q_lo = min(wave * per, P), q_hi = min(q_lo + per, P);
  int hits = 0;
  for (int q0 = q_lo; q0 < q_hi; q0 += 64)
    hits += __popcll(__ballot(q0 + lane < q_hi && s_e[min(q0 + lane, P - 1)] == me));
  if (lane == 0) s_wc[wave] = hits;
  __syncthreads();
  int base = off;
  for (int w = 0; w < wave; ++w) base += s_wc[w];
  for (int q0 = q_lo; q0 < q_hi; q0 += 64) {
    const int q = q0 + lane;
    const bool hit = q < q_hi && s_e[min(q, P - 1)] == me;
    const unsigned long long bal = __ballot(hit);
    if (hit) {
      const int pos = base + __popcll(bal & ((1ull << lane) - 1ull));
      p.pair_tok[pos] = q / K;
      p.pair_w[pos] = p.wts[q];
      p.pidx[(q / K) * (K + 1) + q % K] = pos;
    }
    base += __popcll(bal);
  }
  for (int c = threadIdx.x; c * cs < cnt; c += kGroupThreads) {
    p.chunk_e[choff + c] = me;
    p.chunk_p0[choff + c] = off + c * cs;
    p.chunk_n[choff + c] = min(cs, cnt - c * cs);
  }
  for (int c = threadIdx.x; c * kChunk < cnt; c += kGroupThreads) {
    p.dn_e[dnoff + c] = me;
    p.dn_p0[dnoff + c] = off + c * kChunk;
    p.dn_n[dnoff + c] = min(kChunk, cnt - c * kChunk);
  }
}

// B operand (16 token columns x 32 k) from an LDS tile [kChunk][cols + kPad]:
// lane (c, g) takes token tile*16 + c, columns 128*st + 32g + 8j .. +8.
__device__ __forceinline__ bf16x8 tile_frag(const uint16_t* t, int cols, int tile, int c, int g, int st, int j) {
  return *reinterpret_cast<const bf16x8*>(t + (tile * 16 + c) * (cols + kPad) + st * 128 + g * 32 + 8 * j);
}

struct Chunk {
  int e, p0, n;
  bool shared;
  const uint64_t* ent;
};

// Chunk q of the gate/up list or (kDown) the down list; beside the wide
// kernels chunk q of the gate/up list's small experts, which both passes take
// (one chunk of at most kChunk pairs each); kWide: of its big part.
template <bool kDown, bool kWide = false>
__device__ __forceinline__ bool load_chunk(const PrefillParams& p, int q, Chunk& ch) {
  if (!kWide && p.wide) q += p.hdr->n_big;
  const bool dn = kDown && !p.wide;
  if (q >= (kWide ? p.hdr->n_big : dn ? p.hdr->n_dn : p.hdr->n_gu)) return false;
  ch.e = dn ? p.dn_e[q] : p.chunk_e[q];
  ch.p0 = dn ? p.dn_p0[q] : p.chunk_p0[q];
  ch.n = dn ? p.dn_n[q] : p.chunk_n[q];
  ch.shared = ch.e == p.n_experts;
  ch.ent = ch.shared ? p.shared : p.table + (int64_t)ch.e * 6;
  return true;
}

// This thread's share of a token tile [kC][kCols] of kPlanes planes,
// held in registers between its global loads and its LDS store.  Rows past
// the chunk's n tokens are zero and never loaded.
template <int kPlanes, int kC>
struct XStage {
  static constexpr int kPer = kC * kCols / 8 / kThreads;  // uint4 per thread and plane
  uint4 v[kPlanes][kPer];
  template <typename Src>
  __device__ __forceinline__ void load(Src& src, int kc, int n) {
#pragma unroll
    for (int pl = 0; pl < kPlanes; ++pl)
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int q = threadIdx.x + u * kThreads, tt = q / (kCols / 8), cc = q % (kCols / 8);
        v[pl][u] = tt < n ? ldg<uint4>(src(pl, tt) + kc * kCols + cc * 8) : make_uint4(0, 0, 0, 0);
      }
  }
  __device__ __forceinline__ void store(uint16_t* lds) const {
#pragma unroll
    for (int pl = 0; pl < kPlanes; ++pl)
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int q = threadIdx.x + u * kThreads, tt = q / (kCols / 8), cc = q % (kCols / 8);
        *reinterpret_cast<uint4*>(lds + pl * kC * (kCols + kPad) + tt * (kCols + kPad) + cc * 8) = v[pl][u];
      }
  }
};

// The weights of one K-chunk for a wave: kMats matrices x kRT row tiles.
template <int F, int kMats, int kRT>
struct WBuf {
  static constexpr int kSteps = kCols / 128;
  Batch<F, kSteps> b[kMats][kRT];
  __device__ __forceinline__ void load(const Mat (&mats)[kMats], int row, int k, int kc, int g) {
#pragma unroll
    for (int q = 0; q < kMats; ++q)
#pragma unroll
      for (int rt = 0; rt < kRT; ++rt) b[q][rt].load(mats[q], row + 16 * rt, k, kc * kSteps, g);
  }
};

// Software pipeline over K-chunks of the kMats matrices ([n_rows][k]) at
// ent[w_slot], ent[w_slot + 2], ...  While chunk kc is multiplied, the token
// tile of kc + 1 is in flight to registers and the weights of kc + 2 to the
// third weight buffer; the tile loads are issued before the weight loads.
// Buffers rotate statically (three steps per loop turn).
// kC: token tile rows; kBufs: weight buffers (3: the weights of kc + 2 in
// flight, 2: those of kc + 1, 1: none ahead, for the larger token tile's
// register budget).
template <int F, int kMats, int kRT, int kPlanes, int kC, int kBufs, typename Src, typename Mul>
__device__ __forceinline__ void pipeline(const uint64_t* ent, int w_slot, int n_rows, int row, int k, int g, int n,
                                         uint16_t* lds, Src&& src, Mul&& mul) {
  using W = WBuf<F, kMats, kRT>;
  const int nkc = k / kCols;
  Mat mats[kMats];
#pragma unroll
  for (int q = 0; q < kMats; ++q) mats[q] = make_mat<F>(ent[w_slot + 2 * q], ent[w_slot + 2 * q + 1], n_rows, k);
  XStage<kPlanes, kC> xr;
  if constexpr (F == kBf16 || kBufs == 1) {
    // bf16 weights (a compatibility format, 4x the bytes), or one buffer
    // asked for: no weight prefetch, so that this path never raises the
    // kernel's registers
    W w;
    for (int kc = 0; kc < nkc; ++kc) {
      xr.load(src, kc, n);
      w.load(mats, row, k, kc, g);
      __syncthreads();
      xr.store(lds);
      __syncthreads();
      mul(w);
    }
    return;
  }
  if constexpr (kBufs == 2) {
    W w0, w1;
    xr.load(src, 0, n);
    w0.load(mats, row, k, 0, g);
    auto step2 = [&](const W& wc, W& wl, int kc) {
      __syncthreads();
      xr.store(lds);
      __syncthreads();
      if (kc + 1 < nkc) {
        xr.load(src, kc + 1, n);
        wl.load(mats, row, k, kc + 1, g);
      }
      mul(wc);
    };
    for (int kc = 0; kc < nkc; kc += 2) {
      step2(w0, w1, kc);
      if (kc + 1 < nkc) step2(w1, w0, kc + 1);
    }
    return;
  }
  W w0, w1, w2;
  xr.load(src, 0, n);
  w0.load(mats, row, k, 0, g);
  if (nkc > 1) w1.load(mats, row, k, 1, g);
  auto step = [&](const W& wc, W& wl, int kc) {
    __syncthreads();
    xr.store(lds);
    __syncthreads();
    if (kc + 1 < nkc) xr.load(src, kc + 1, n);
    if (kc + 2 < nkc) wl.load(mats, row, k, kc + 2, g);
    mul(wc);
  };
  for (int kc = 0; kc < nkc; kc += 3) {
    step(w0, w2, kc);
    if (kc + 1 < nkc) step(w1, w0, kc + 1);
    if (kc + 2 < nkc) step(w2, w1, kc + 2);
  }
}

// ---------------------------------------------------------------- gate / up
// The E8M0 scale bytes lane (r, g) needs for steps [s0, s0 + kSteps) of
// weight row `row` (k columns): byte j of c[q] is the group-g scale of step
// s0 + 4q + j.  A K-chunk uses two steps' bytes; reading them per K-chunk
// touched each row's 128-byte scale line sixteen times, far enough apart in
// time that the weight stream had evicted it from L2 in between (measured:
// ~0.6 GB of the gate/up fetch of the M=512 prefill against 0.13 GB of
// scales).  fill() reads the row's kSteps steps of scales once (lane g: steps
// s0 + 4g .. +3, 16 bytes) and deals each step's word to the row's four lanes
// (ds_bpermute from lanes r + 16q); consume() advances past a K-chunk.
struct ScaleCache {
  static constexpr int kSteps = 16;  // 8 K-chunks
  uint32_t c[4];
  __device__ __forceinline__ void fill(const BufRsrc& s, int row, int k, int s0, int g) {
    const int r = (threadIdx.x & 63) & 15;
    const uint4 u = bload128(s, (uint32_t)row * (uint32_t)(k / 32) + (uint32_t)(s0 + 4 * g) * 4);
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) c[q] = 0u;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t v = (uint32_t)__builtin_amdgcn_ds_bpermute((r + 16 * q) * 4, (int)w[j]);
        c[q] |= ((v >> (8 * g)) & 0xffu) << (8 * j);
      }
  }
  // scale byte of step b of K-chunk kc (two steps per K-chunk)
  __device__ __forceinline__ uint32_t byte(int kc, int b) const { return (c[0] >> (8 * (2 * (kc & 1) + b))) & 0xffu; }
  __device__ __forceinline__ void consume(int kc) {
    if (kc & 1) {
#pragma unroll
      for (int q = 0; q < 3; ++q) c[q] = c[q + 1];
      c[3] = 0u;
    }
  }
};

// Wave rows r0 .. r0+16*kGuRT-1 of W1 and W3 against the chunk's tokens; lane
// (r, g) ends holding rows r0 + 16 rt + 4g + q of token tile*16 + r.
// F = kFp4E8M0Split: E8M0 scales through a ScaleCache per matrix (the same
// decoded weights as kFp4E8M0).
template <int F, int kC, int kBufs>
__device__ void gate_up_chunk(const PrefillParams& p, const Chunk& ch, int r0, uint16_t* xs, const int* s_tok) {
  using W = WBuf<F, 2, kGuRT>;
  constexpr int kTiles = kC / 16;
  constexpr bool kSplit = F == kFp4E8M0Split;
  static_assert(!kSplit || (kGuRT == 1 && W::kSteps == 2), "scale cache: one row tile, two steps per K-chunk");
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int ntile = (ch.n + 15) / 16;
  f32x4 ag[kGuRT][kTiles], au[kGuRT][kTiles];
#pragma unroll
  for (int rt = 0; rt < kGuRT; ++rt)
#pragma unroll
    for (int t = 0; t < kTiles; ++t) ag[rt][t] = au[rt][t] = f32x4{0, 0, 0, 0};
  ScaleCache s1, s3;
  const BufRsrc sr1 = make_mat<F>(ch.ent[0], ch.ent[1], p.i, p.d).s, sr3 = make_mat<F>(ch.ent[2], ch.ent[3], p.i, p.d).s;
  if constexpr (kSplit) {
    s1.fill(sr1, r0 + r, p.d, 0, g);
    s3.fill(sr3, r0 + r, p.d, 0, g);
  }
  int kc = 0;
  auto src = [&](int, int tt) { return p.x + (int64_t)s_tok[tt] * p.d; };
  pipeline<F, 2, kGuRT, 1, kC, kBufs>(ch.ent, 0, p.i, r0 + r, p.d, g, ch.n, xs, src, [&](const W& w) {
    if constexpr (kSplit) {
      if (kc > 0 && (kc & (ScaleCache::kSteps / 2 - 1)) == 0) {  // the next kSteps steps' scales
        s1.fill(sr1, r0 + r, p.d, 2 * kc, g);
        s3.fill(sr3, r0 + r, p.d, 2 * kc, g);
      }
    }
#pragma unroll
    for (int b = 0; b < W::kSteps; ++b) {
      uint32_t e1 = 0, e3 = 0;
      if constexpr (kSplit) {
        e1 = s1.byte(kc, b);
        e3 = s3.byte(kc, b);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int rt = 0; rt < kGuRT; ++rt) {
          bf16x8 f1, f3;
          if constexpr (kSplit) {
            f1 = w.b[0][rt].frag_e(b, j, e1);
            f3 = w.b[1][rt].frag_e(b, j, e3);
          } else {
            f1 = w.b[0][rt].frag(b, j, g);
            f3 = w.b[1][rt].frag(b, j, g);
          }
#pragma unroll
          for (int tile = 0; tile < kTiles; ++tile) {
            if (tile >= ntile) break;
            const bf16x8 xf = tile_frag(xs, kCols, tile, r, g, b, j);
            ag[rt][tile] = mfma16x16x32(f1, xf, ag[rt][tile]);
            au[rt][tile] = mfma16x16x32(f3, xf, au[rt][tile]);
          }
        }
      }
    }
    if constexpr (kSplit) {
      s1.consume(kc);
      s3.consume(kc);
    }
    ++kc;
  });
#pragma unroll
  for (int tile = 0; tile < kTiles; ++tile) {
    const int tt = tile * 16 + r;
    if (tile >= ntile || tt >= ch.n) continue;
    const int64_t pr = ch.p0 + tt;
    const float wt = p.pair_w[pr];
#pragma unroll
    for (int rt = 0; rt < kGuRT; ++rt) {
      uint32_t hi[4], lo[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float a = __fmul_rn(wt, swiglu(ag[rt][tile][q], au[rt][tile][q], p.limit));
        hi[q] = f32_to_bf16_bits(a);
        lo[q] = f32_to_bf16_bits(__fadd_rn(a, -bf16_bits_to_f32(hi[q])));
      }
      const int64_t o = pr * p.i + r0 + 16 * rt + 4 * g;
      *reinterpret_cast<uint2*>(p.act_hi + o) = make_uint2(hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16));
      *reinterpret_cast<uint2*>(p.act_lo + o) = make_uint2(lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16));
    }
  }
}

// F: format of the routed FP4 experts of the call's scale kind; the shared
// expert's chunks are FP8; entries without scales (of either) take the bf16 path.
template <int F>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4)))
prefill_gate_up_kernel(PrefillParams p) {
  __shared__ __align__(16) uint16_t xs[kBigChunk * (kCols + kPad)];
  __shared__ int s_tok[kBigChunk];
  const int nrb = p.i / kGuRows;
  Chunk ch;
  if (!load_chunk<false>(p, blockIdx.x / nrb, ch)) return;
  if (threadIdx.x < kBigChunk) s_tok[threadIdx.x] = threadIdx.x < ch.n ? p.pair_tok[ch.p0 + threadIdx.x] : 0;
  __syncthreads();
  const int r0 = (blockIdx.x % nrb) * kGuRows + 16 * kGuRT * (threadIdx.x >> 6);
  // routed E8M0 chunks read their scales through a per-lane cache (same weights)
  constexpr int FG = F == kFp4E8M0 ? kFp4E8M0Split : F;
  if (!ch.ent[1] || ch.shared) {  // bf16 or FP8 weights: a chunk of more than kChunk pairs as two halves (registers)
    for (int h0 = 0; h0 < ch.n; h0 += kChunk) {
      Chunk sub = ch;
      sub.p0 = ch.p0 + h0;
      sub.n = min(kChunk, ch.n - h0);
      if (ch.ent[1]) gate_up_chunk<kFp8Block, kChunk, 1>(p, sub, r0, xs, s_tok + h0);
      else gate_up_chunk<kBf16, kChunk, 1>(p, sub, r0, xs, s_tok + h0);
    }
  } else if (ch.n > kChunk) {
    gate_up_chunk<FG, kBigChunk, 1>(p, ch, r0, xs, s_tok);
  } else {
    gate_up_chunk<FG, kChunk, 3>(p, ch, r0, xs, s_tok);
  }
}

// ---------------------------------------------------------------- down
// F = kFp4E8M0Split: W2's E8M0 scales through a ScaleCache per row tile.
template <int F, int kBufs>
__device__ void down_chunk(const PrefillParams& p, const Chunk& ch, int r0, uint16_t* as) {
  using W = WBuf<F, 1, kDnRT>;
  constexpr bool kSplit = F == kFp4E8M0Split;
  static_assert(!kSplit || W::kSteps == 2, "scale cache: two steps per K-chunk");
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int ntile = (ch.n + 15) / 16;
  const uint16_t* ls = as + kChunk * (kCols + kPad);
  f32x4 acc[kDnRT][2];
#pragma unroll
  for (int rt = 0; rt < kDnRT; ++rt) acc[rt][0] = acc[rt][1] = f32x4{0, 0, 0, 0};
  ScaleCache sc[kDnRT];
  const BufRsrc sr = make_mat<F>(ch.ent[4], ch.ent[5], p.d, p.i).s;
  if constexpr (kSplit) {
#pragma unroll
    for (int rt = 0; rt < kDnRT; ++rt) sc[rt].fill(sr, r0 + r + 16 * rt, p.i, 0, g);
  }
  int kc = 0;
  auto src = [&](int pl, int tt) { return (pl ? p.act_lo : p.act_hi) + (int64_t)(ch.p0 + tt) * p.i; };
  pipeline<F, 1, kDnRT, 2, kChunk, kBufs>(ch.ent, 4, p.d, r0 + r, p.i, g, ch.n, as, src, [&](const W& w) {
    if constexpr (kSplit) {
      if (kc > 0 && (kc & (ScaleCache::kSteps / 2 - 1)) == 0) {  // the next kSteps steps' scales
#pragma unroll
        for (int rt = 0; rt < kDnRT; ++rt) sc[rt].fill(sr, r0 + r + 16 * rt, p.i, 2 * kc, g);
      }
    }
#pragma unroll
    for (int b = 0; b < W::kSteps; ++b) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int tile = 0; tile < 2; ++tile) {
          if (tile >= ntile) break;
          const bf16x8 hf = tile_frag(as, kCols, tile, r, g, b, j), lf = tile_frag(ls, kCols, tile, r, g, b, j);
#pragma unroll
          for (int rt = 0; rt < kDnRT; ++rt) {
            bf16x8 wf;
            if constexpr (kSplit) wf = w.b[0][rt].frag_e(b, j, sc[rt].byte(kc, b));
            else wf = w.b[0][rt].frag(b, j, g);
            acc[rt][tile] = mfma16x16x32(wf, hf, acc[rt][tile]);
            acc[rt][tile] = mfma16x16x32(wf, lf, acc[rt][tile]);
          }
        }
      }
    }
    if constexpr (kSplit) {
#pragma unroll
      for (int rt = 0; rt < kDnRT; ++rt) sc[rt].consume(kc);
    }
    ++kc;
  });
#pragma unroll
  for (int tile = 0; tile < 2; ++tile) {
    const int tt = tile * 16 + r;
    if (tile >= ntile || tt >= ch.n) continue;
#pragma unroll
    for (int rt = 0; rt < kDnRT; ++rt) {
      float* o = p.part + (int64_t)(ch.p0 + tt) * p.d + r0 + 16 * rt + 4 * g;
      *reinterpret_cast<float4*>(o) = make_float4(acc[rt][tile][0], acc[rt][tile][1], acc[rt][tile][2], acc[rt][tile][3]);
    }
  }
}

template <int F>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(3)))
prefill_down_kernel(PrefillParams p) {
  __shared__ __align__(16) uint16_t as[2 * kChunk * (kCols + kPad)];  // hi plane, lo plane
  const int nrb = p.d / kDnRows;
  Chunk ch;
  if (!load_chunk<true>(p, blockIdx.x / nrb, ch)) return;
  const int r0 = (blockIdx.x % nrb) * kDnRows + 16 * kDnRT * (threadIdx.x >> 6);
  if (!ch.ent[1]) down_chunk<kBf16, 1>(p, ch, r0, as);
  else if (ch.shared) down_chunk<kFp8Block, 1>(p, ch, r0, as);
  else down_chunk<F == kFp4E8M0 ? kFp4E8M0Split : F, 3>(p, ch, r0, as);  // routed E8M0: cached scales
}

// ---------------------------------------------------------------- wide
// Gate/up (kDown false) and down for calls whose experts hold many pairs: a
// workgroup takes a chunk of up to 64 pairs and 128 rows of W1 and W3 (32 per
// wave and matrix), or 256 rows of W2 (two tiles of 32 per wave), on
// v_mfma_f32_32x32x16_bf16.  With the 16-row tiles above every 16-byte LDS read
// feeds two 16x16x32 products, which takes the LDS as long as the matrix cores,
// and every row block of 64 reads the tokens again; here a read feeds two
// products of twice the size and half as many row blocks read the tokens.  Two
// waves per SIMD (256 registers) hold 64 accumulators, the unit of weights
// being multiplied and the next one, and the next token tile on its way to the
// other half of the LDS: one barrier per stage, a step's LDS reads and decode
// under the products of the step before.
// Measured at 12288 pairs of 256 experts and 2048 of the shared one, d = 4096,
// i = 2048: gate/up 720 us, down 570 (0.86 and 1.09 PFLOP/s of issued products;
// 455 and 375 with no loads in the loop), a layer of 4096 tokens 3290 -> 2820.
//
// Columns: a K-chunk is 256 columns; lane (c, h) of a wave owns columns
// 128h .. +127 of it, as 4 groups of 32 (16 bytes of FP4 each), so that its 4
// E8M0 scales are one aligned word.  A weight unit is 64 bytes of a lane's
// columns per matrix: all 4 groups in FP4, 2 in FP8, 1 in bf16.  A stage is an
// LDS tile: 64 tokens x 256 columns (gate/up), or the hi and lo planes of
// 64 pairs x 128 columns (down: groups 2t and 2t + 1 of either half).  The LDS
// rows are unpadded, 16-byte unit u of row t stored at u ^ (t & 15).
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWideGuRows = 128;  // rows of W1 and W3 per workgroup
constexpr int kWideDnRows = 256;  // rows of W2 per workgroup
constexpr int kStage16 = 2048;    // 16-byte units per LDS stage

__device__ __forceinline__ uint4 bload128s(BufRsrc r, uint32_t off, uint32_t soff) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, (int)soff, 0);
  return make_uint4(v[0], v[1], v[2], v[3]);
}

// Dword v of q, v a constant after unrolling.
__device__ __forceinline__ uint32_t dword(const uint4& q, int v) {
  return v == 0 ? q.x : v == 1 ? q.y : v == 2 ? q.z : q.w;
}

// One exchange of a transpose over lanes: `odd` lanes give a and take the
// other lane's b for it, the others give b and take a (kCtrl: the quad_perm
// that names the other lane).
template <int kCtrl>
__device__ __forceinline__ void swap_pieces(uint4& a, uint4& b, bool odd) {
  auto one = [odd](uint32_t& x, uint32_t& y) {
    // (both moves run on every lane: they read the other's register)
    const uint32_t ox = (uint32_t)__builtin_amdgcn_mov_dpp((int)x, kCtrl, 0xf, 0xf, true);
    const uint32_t oy = (uint32_t)__builtin_amdgcn_mov_dpp((int)y, kCtrl, 0xf, 0xf, true);
    x = odd ? oy : x;
    y = odd ? y : ox;
  };
  one(a.x, b.x);
  one(a.y, b.y);
  one(a.z, b.z);
  one(a.w, b.w);
}

// A unit of both matrices (or row tiles), its fp32 scales beside it.
template <int F>
struct WideUnit {
  static constexpr int kUnits = F == kBf16 ? 4 : F == kFp8Block ? 2 : 1;  // per K-chunk
  static constexpr int kGroups = 4 / kUnits;                              // of 32 columns, per half
  static constexpr int kChunkBytes = 256 * kUnits / 2;                    // of a row, per K-chunk
  uint4 q[2][4];
  uint4 sf[2];  // kFp4F32: the 4 groups' scales
  float s8[2];  // kFp8Block: the half's block scale
  // q[t][v]: bytes 16 (c % 4) .. +15 of the unit of row 4 (c / 4) + v (wo: that
  // of v = 0), so that four neighbouring lanes read one 64-byte run (a lane per
  // row touches four times as many lines per load: a layer of 4096 tokens 2970
  // us against 2856); turn() then gives lane c its own row's 64 bytes.
  __device__ __forceinline__ void load(const Mat (&m)[2], const uint32_t (&wo)[2], const uint32_t (&so)[2], int kc,
                                       int u, int row_bytes) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int v = 0; v < 4; ++v)
        q[t][v] = bload128s(m[t].w, wo[t] + 64 * u, (uint32_t)kc * kChunkBytes + (uint32_t)(v * row_bytes));
      if constexpr (F == kFp4F32) sf[t] = bload128s(m[t].s, so[t], (uint32_t)kc * 32);
      if constexpr (F == kFp8Block)
        s8[t] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(m[t].s, (int)so[t], kc * 8, 0));
    }
  }
  // 4 x 4 transpose of the 16-byte pieces over each quad of lanes
  __device__ __forceinline__ void turn() {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      swap_pieces<0xB1>(q[t][0], q[t][1], (lane & 1) != 0);
      swap_pieces<0xB1>(q[t][2], q[t][3], (lane & 1) != 0);
      swap_pieces<0x4E>(q[t][0], q[t][2], (lane & 2) != 0);
      swap_pieces<0x4E>(q[t][1], q[t][3], (lane & 2) != 0);
    }
  }
  // columns 8j .. +7 of the unit's group s (group gi of the half); e: the half's 4 E8M0 bytes
  __device__ __forceinline__ bf16x8 frag(int t, int s, int gi, int j, uint32_t e) const {
    if constexpr (F == kFp4E8M0) {
      return fp4x8_to_bf16_e8m0(dword(q[t][s], j), e8m0_as_f32((e >> (8 * gi)) & 0xffu));
    } else if constexpr (F == kFp4F32) {
      return fp4x8_to_bf16_f32(dword(q[t][s], j), __uint_as_float(dword(sf[t], gi)));
    } else if constexpr (F == kFp8Block) {
      const uint4& w = q[t][2 * s + j / 2];
      bf16x8 f;
      fp8x4_to_bf16(dword(w, 2 * (j & 1)), s8[t], f, 0);
      fp8x4_to_bf16(dword(w, 2 * (j & 1) + 1), s8[t], f, 1);
      return f;
    } else {
      return __builtin_bit_cast(bf16x8, q[t][j]);
    }
  }
};

// The E8M0 bytes of 4 K-chunks: a lane reads 16 of a row's 32 bytes and the
// two halves swap, so that w[q] is the lane's word of K-chunk q.
struct WideScales {
  uint32_t w[4];
  __device__ __forceinline__ void deal(const uint4& raw) {
    const auto a = __builtin_amdgcn_permlane32_swap(raw.x, raw.y, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(raw.z, raw.w, false, false);
    w[0] = a[0];
    w[2] = a[1];
    w[1] = b[0];
    w[3] = b[1];
  }
};

// One chunk's rows r0 .. of this wave; kTiles: 32-pair tiles of the chunk.
template <int F, bool kDown, int kTiles>
__device__ __forceinline__ void wide_chunk(const PrefillParams& p, const Chunk& ch, int r0, uint4* lds) {
  using U = WideUnit<F>;
  constexpr int kPlanes = kDown ? 2 : 1, kStages = kDown ? 2 : 1;  // planes per stage, stages per K-chunk
  constexpr int kRow16 = kDown ? 16 : 32;                          // 16-byte units per LDS row
  constexpr int kPer = kTiles * 32 * kRow16 / kThreads;            // units per thread and plane
  constexpr int kStageGroups = 4 / kStages;
  // units held: the one multiplied and those in flight (a bf16 unit is multiplied in 256 to 512 cycles, less
  // than a load takes: three ahead where a chunk of one tile leaves the registers)
  constexpr int kBufs = F == kBf16 && kTiles == 1 ? 4 : 2, kAhead = kBufs - 1;
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int K = kDown ? p.i : p.d, nkc = K / kCols, row_bytes = nkc * U::kChunkBytes;
  // weights: W1 and W3 at one row, or W2 at two
  Mat m[2];
  uint32_t wo[2], so[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int slot = kDown ? 4 : 2 * t;
    const uint32_t row = (uint32_t)(r0 + (kDown ? 32 * t : 0) + c);
    m[t] = make_mat<F>(ch.ent[slot], ch.ent[slot + 1], kDown ? p.d : p.i, K);
    wo[t] = (row - c % 4) * (uint32_t)row_bytes + h * (U::kChunkBytes / 2) + c % 4 * 16;
    if constexpr (F == kFp4E8M0) so[t] = row * (uint32_t)(K / 32) + 16 * h;
    else if constexpr (F == kFp4F32) so[t] = 4 * (row * (uint32_t)(K / 32) + 4 * h);
    else so[t] = 4 * (row / 128 * (uint32_t)(K / 128) + h);
  }
  // the token tile: rows past the chunk's pairs repeat its last one (their results are dropped)
  uint32_t xo[kPer];
  uint4 xr[kPlanes][kPer];
#pragma unroll
  for (int v = 0; v < kPer; ++v) {
    const int q = (int)threadIdx.x + v * kThreads, un = q % kRow16, src = min(q / kRow16, ch.n - 1);
    if constexpr (kDown) xo[v] = 2 * ((uint32_t)src * (uint32_t)p.i + (un >> 3) * 128 + (un & 7) * 8);
    else xo[v] = 2 * ((uint32_t)p.pair_tok[ch.p0 + src] * (uint32_t)p.d + un * 8);
  }
  BufRsrc xb[kPlanes];
  if constexpr (kDown) {
    xb[0] = make_buf((uint64_t)(p.act_hi + (int64_t)ch.p0 * p.i), 2u * ch.n * p.i);
    xb[1] = make_buf((uint64_t)(p.act_lo + (int64_t)ch.p0 * p.i), 2u * ch.n * p.i);
  } else {
    xb[0] = make_buf((uint64_t)p.x, 2u * p.m * p.d);
  }
  // this thread's first unit of the LDS tile; its later ones are 8 (gate/up) or 16 rows on
  const int x_row = (int)threadIdx.x / kRow16, x_un = (int)threadIdx.x % kRow16;
  const int xl0 = x_row * kRow16 + (x_un ^ (x_row & 15)), xl1 = kDown ? xl0 : xl0 ^ 8;
  auto xload = [&](int kc, int st) {
#pragma unroll
    for (int pl = 0; pl < kPlanes; ++pl)
#pragma unroll
      for (int v = 0; v < kPer; ++v) xr[pl][v] = bload128s(xb[pl], xo[v], (uint32_t)(kc * kCols + st * 64) * 2);
  };
  auto xstore = [&](int buf) {
#pragma unroll
    for (int pl = 0; pl < kPlanes; ++pl)
#pragma unroll
      for (int v = 0; v < kPer; ++v)
        lds[buf * kStage16 + pl * (kStage16 / 2) + (v & 1 ? xl1 : xl0) + v * kThreads] = xr[pl][v];
  };
  f32x16 acc[2][kTiles];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int tile = 0; tile < kTiles; ++tile)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[t][tile][q] = 0.0f;
  U w[kBufs];
  uint4 raw[2];
  WideScales sc[2];
  xload(0, 0);
#pragma unroll
  for (int u = 0; u < kAhead; ++u) w[u].load(m, wo, so, 0, u, row_bytes);
  if constexpr (F == kFp4E8M0) {
#pragma unroll
    for (int t = 0; t < 2; ++t) raw[t] = bload128(m[t].s, so[t]);
  }
  xstore(0);
  // 16-byte unit of (group 0, j = 0) of this lane's columns in LDS row c; the
  // others differ from it in the low bits only
  const int lb = c * kRow16 + ((h * (kRow16 / 2)) ^ (c & 15));
  for (int kc = 0; kc < nkc; kc += 2) {  // (K is a multiple of 512)
    if constexpr (F == kFp4E8M0) {
      if ((kc & 2) == 0) {
#pragma unroll
        for (int t = 0; t < 2; ++t) sc[t].deal(raw[t]);
      } else {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          sc[t].w[0] = sc[t].w[2];
          sc[t].w[1] = sc[t].w[3];
          raw[t] = bload128(m[t].s, so[t] + (uint32_t)(kc + 2) * 8);  // (past the row or the end: unused)
        }
      }
    }
#pragma unroll
    for (int k2 = 0; k2 < 2; ++k2) {
#pragma unroll
      for (int st = 0; st < kStages; ++st) {
        const int buf = (k2 * kStages + st) & 1;
        const bool last = k2 == 1 && st == kStages - 1;
        const bool more = !last || kc + 2 < nkc;
        __syncthreads();
        if (more) xload(st == kStages - 1 ? kc + k2 + 1 : kc + k2, st == kStages - 1 ? 0 : st + 1);
        const uint4* const tile16 = lds + buf * kStage16;
        // steps of the stage: (group, j, plane); step k + 1's operands are read
        // and decoded while step k is multiplied
        constexpr int kSteps = kStageGroups * 4 * kPlanes;
        bf16x8 a[2][2], bt[2][kTiles];
        auto read_b = [&](int k) {
          const int un = lb ^ (k / kPlanes), pl = k % kPlanes;
#pragma unroll
          for (int tile = 0; tile < kTiles; ++tile)
            bt[k & 1][tile] =
                *reinterpret_cast<const bf16x8*>(tile16 + pl * (kStage16 / 2) + tile * 32 * kRow16 + un);
        };
        auto decode = [&](int k) {  // k: (group, j)
          const int gi = st * kStageGroups + k / 4, u = gi / U::kGroups;
          U& wc = w[(k2 * U::kUnits + u) % kBufs];
          if (gi % U::kGroups == 0 && k % 4 == 0) wc.turn();  // (the unit's first use)
#pragma unroll
          for (int t = 0; t < 2; ++t)
            a[k & 1][t] = wc.frag(t, gi % U::kGroups, gi, k % 4, F == kFp4E8M0 ? sc[t].w[k2] : 0u);
        };
        read_b(0);
        decode(0);
#pragma unroll
        for (int k = 0; k < kSteps; ++k) {
          const int kd = k / kPlanes, gi = st * kStageGroups + kd / 4, u = gi / U::kGroups;
          if (k % (4 * kPlanes) == 0 && gi % U::kGroups == 0) {  // a unit's first step: the weights of the unit kAhead on
            const int un = k2 * U::kUnits + u + kAhead, ahead = un / U::kUnits;  // (counted from K-chunk kc)
            if (ahead < 2 || kc + 2 < nkc) w[un % kBufs].load(m, wo, so, kc + ahead, un % U::kUnits, row_bytes);
            __builtin_amdgcn_sched_barrier(0);  // (the scheduler would sink the loads to their uses)
          }
          if (k + 1 < kSteps) read_b(k + 1);
          if (k % kPlanes == kPlanes - 1 && k + 1 < kSteps) decode(kd + 1);
#pragma unroll
          for (int tile = 0; tile < kTiles; ++tile)
#pragma unroll
            for (int t = 0; t < 2; ++t)
              acc[t][tile] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kd & 1][t], bt[k & 1][tile], acc[t][tile], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (more) xstore(buf ^ 1);
      }
    }
  }
  // lane (c, h) holds rows 8 (q / 4) + 4h + q % 4 of pair 32 tile + c
#pragma unroll
  for (int tile = 0; tile < kTiles; ++tile) {
    const int tt = tile * 32 + c;
    if (tt >= ch.n) continue;
    const int64_t pr = ch.p0 + tt;
    if constexpr (kDown) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int q = 0; q < 16; q += 4)
          *reinterpret_cast<float4*>(p.part + pr * p.d + r0 + 32 * t + 2 * q + 4 * h) =
              make_float4(acc[t][tile][q], acc[t][tile][q + 1], acc[t][tile][q + 2], acc[t][tile][q + 3]);
    } else {
      const float wt = p.pair_w[pr];
#pragma unroll
      for (int q = 0; q < 16; q += 4) {
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float a = __fmul_rn(wt, swiglu(acc[0][tile][q + v], acc[1][tile][q + v], p.limit));
          hi[v] = f32_to_bf16_bits(a);
          lo[v] = f32_to_bf16_bits(__fadd_rn(a, -bf16_bits_to_f32(hi[v])));
        }
        const int64_t o = pr * p.i + r0 + 2 * q + 4 * h;
        *reinterpret_cast<uint2*>(p.act_hi + o) = make_uint2(hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16));
        *reinterpret_cast<uint2*>(p.act_lo + o) = make_uint2(lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16));
      }
    }
  }
}

template <int F, bool kDown>
__device__ __forceinline__ void wide_any(const PrefillParams& p, const Chunk& ch, int r0, uint4* lds) {
  if (ch.n > 32) wide_chunk<F, kDown, 2>(p, ch, r0, lds);
  else wide_chunk<F, kDown, 1>(p, ch, r0, lds);
}

// F: format of the routed FP4 experts of the call's scale kind.
template <int F, bool kDown>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
prefill_wide_kernel(PrefillParams p) {
  __shared__ uint4 lds[2 * kStage16];
  constexpr int kRows = kDown ? kWideDnRows : kWideGuRows;
  // Workgroup b runs on XCD b % 8.  A routed chunk's row blocks go to one XCD,
  // whose L2 then holds the chunk's tokens.  Chunks of one expert (the shared
  // one's, or those of a call with few experts) go row block by row block, so
  // that an XCD's L2 holds its share of the weights for all of them.
  const int nrb = (kDown ? p.d : p.i) / kRows, n_rows = p.by_rows ? p.hdr->n_big * nrb : p.n_sh_gu * nrb;
  int q, rb;
  if ((int)blockIdx.x < n_rows) {
    q = blockIdx.x / nrb;
    rb = blockIdx.x % nrb;
  } else {
    const int b = blockIdx.x - n_rows, b8 = b / 8;
    q = p.n_sh_gu + b8 / nrb * 8 + b % 8;
    rb = b8 % nrb;
  }
  Chunk ch;
  if (p.by_rows && (int)blockIdx.x >= n_rows) return;
  if (!load_chunk<kDown, true>(p, q, ch)) return;
  const int r0 = rb * kRows + kRows / 4 * (threadIdx.x >> 6);
  if (!ch.ent[1]) wide_any<kBf16, kDown>(p, ch, r0, lds);
  else if (ch.shared) wide_any<kFp8Block, kDown>(p, ch, r0, lds);
  else wide_any<F, kDown>(p, ch, r0, lds);
}

// ---------------------------------------------------------------- combine
// grid (m, d / 1024): thread -> 4 consecutive columns of one token.
__global__ void __launch_bounds__(kThreads) prefill_combine_kernel(PrefillParams p) {
  const int t = blockIdx.x;
  const int col = (blockIdx.y * kThreads + threadIdx.x) * 4;
  if (col >= p.d) return;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  const int* pi = p.pidx + (int64_t)t * (p.top_k + 1);
  for (int j = 0; j <= p.top_k; ++j) {
    const int pr = pi[j];
    if (pr < 0) continue;
    const float4 v = *reinterpret_cast<const float4*>(p.part + (int64_t)pr * p.d + col);
    acc.x = __fadd_rn(acc.x, v.x);
    acc.y = __fadd_rn(acc.y, v.y);
    acc.z = __fadd_rn(acc.z, v.z);
    acc.w = __fadd_rn(acc.w, v.w);
  }
  const int64_t o = (int64_t)t * p.d + col;
  if (p.out_f32) *reinterpret_cast<float4*>(p.out_f32 + o) = acc;
  if (p.out_bf16)
    *reinterpret_cast<uint2*>(p.out_bf16 + o) =
        make_uint2(f32_to_bf16_bits(acc.x) | (f32_to_bf16_bits(acc.y) << 16),
                   f32_to_bf16_bits(acc.z) | (f32_to_bf16_bits(acc.w) << 16));
}

size_t align256(size_t n) { return (n + 255) / 256 * 256; }

struct Layout {
  size_t hdr, pair_tok, pair_w, pidx, chunk_e, chunk_p0, chunk_n, dn_e, dn_p0, dn_n, act_hi, act_lo, part, total;
};

int64_t max_pairs(int64_t m, int top_k) { return m * top_k + m; }
// Chunks of the routed experts in either list: at most sum over experts of
// ceil(n_e / kChunk) <= (experts with a pair) + (pairs) / kChunk (a gate/up
// chunk of kBigChunk covers two down chunks).
int64_t max_routed_chunks(int64_t m, int64_t n_experts, int top_k) {
  const int64_t pk = m * top_k;
  return (n_experts < pk ? n_experts : pk) + (pk + kChunk - 1) / kChunk;
}
int64_t max_chunks(int64_t m, int64_t n_experts, int top_k) {
  return max_routed_chunks(m, n_experts, top_k) + (m + kChunk - 1) / kChunk;
}

Layout layout(int64_t m, int64_t d, int64_t i, int64_t n_experts, int top_k) {
  const int64_t P = max_pairs(m, top_k), C = max_chunks(m, n_experts, top_k);
  Layout L;
  size_t o = 0;
  L.hdr = o;
  o += 256;
  L.pair_tok = o;
  o += align256((size_t)P * 4);
  L.pair_w = o;
  o += align256((size_t)P * 4);
  L.pidx = o;
  o += align256((size_t)m * (top_k + 1) * 4);
  L.chunk_e = o;
  o += align256((size_t)C * 4);
  L.chunk_p0 = o;
  o += align256((size_t)C * 4);
  L.chunk_n = o;
  o += align256((size_t)C * 4);
  L.dn_e = o;
  o += align256((size_t)C * 4);
  L.dn_p0 = o;
  o += align256((size_t)C * 4);
  L.dn_n = o;
  o += align256((size_t)C * 4);
  L.act_hi = o;
  o += align256((size_t)P * i * 2);
  L.act_lo = o;
  o += align256((size_t)P * i * 2);
  L.part = o;
  o += align256((size_t)P * d * 4);
  L.total = o;
  return L;
}

}  // namespace
}  // namespace hsmoe

using namespace hsmoe;

extern "C" size_t hsmoe_moe_prefill_workspace_size(int64_t m, int64_t d, int64_t i, int64_t n_experts, int top_k) {
  if (m < 1 || d < 1 || i < 1 || n_experts < 1 || top_k < 1) return 0;
  return layout(m, d, i, n_experts, top_k).total;
}

extern "C" int hsmoe_moe_prefill(const void* x, int64_t m, int64_t d, int64_t i, const int64_t* topk_idx,
                                 const float* topk_w, int top_k, const uint64_t* expert_table, int64_t n_experts,
                                 int scale_kind, const uint64_t* shared, float swiglu_limit, float* out_f32,
                                 void* out_bf16, void* workspace, size_t workspace_bytes, hsmoe_stream_t stream) {
  const char* name = "hsmoe_moe_prefill";
  if (!x || !topk_idx || !topk_w || !expert_table || (!out_f32 && !out_bf16))
    return fail(HSMOE_ERR_ARG, "%s: null pointer or no output", name);
  if (scale_kind != HSMOE_SCALE_E8M0 && scale_kind != HSMOE_SCALE_F32)
    return fail(HSMOE_ERR_ARG, "%s: unknown scale_kind %d", name, scale_kind);
  if (n_experts < 1 || n_experts > kMaxExperts || top_k < 1 || top_k > 16 || m < 1 || m * top_k > kMaxPairs)
    return fail(HSMOE_ERR_SHAPE, "%s: need 1 <= n_experts <= %d, 1 <= top_k <= 16, 1 <= m*top_k <= %d", name,
                kMaxExperts, kMaxPairs);
  if (d % 1024 != 0 || i % 512 != 0 || d > 65536 || i > 65536)
    return fail(HSMOE_ERR_SHAPE, "%s: d must be a multiple of 1024 and i of 512 (d=%lld i=%lld)", name, (long long)d,
                (long long)i);
  if (!expert_fits(d, i))
    return fail(HSMOE_ERR_SHAPE, "%s: d*i too large (an expert matrix must stay below 4 GiB)", name);
  if (!aligned(x, 16) || (out_f32 && !aligned(out_f32, 16)) || (out_bf16 && !aligned(out_bf16, 8)))
    return fail(HSMOE_ERR_SHAPE, "%s: x and out_f32 must be 16-byte aligned, out_bf16 8-byte aligned", name);
  const Layout L = layout(m, d, i, n_experts, top_k);
  if (!workspace || workspace_bytes < L.total || !aligned(workspace, 256))
    return fail(HSMOE_ERR_WORKSPACE, "%s: workspace of %zu bytes (256-byte aligned) needed", name, L.total);
  char* ws = (char*)workspace;
  PrefillParams p;
  p.x = (const uint16_t*)x;
  p.idx = topk_idx;
  p.wts = topk_w;
  p.table = expert_table;
  p.shared = shared;
  p.hdr = (Header*)(ws + L.hdr);
  p.pair_tok = (int*)(ws + L.pair_tok);
  p.pair_w = (float*)(ws + L.pair_w);
  p.pidx = (int*)(ws + L.pidx);
  p.chunk_e = (int*)(ws + L.chunk_e);
  p.chunk_p0 = (int*)(ws + L.chunk_p0);
  p.chunk_n = (int*)(ws + L.chunk_n);
  p.dn_e = (int*)(ws + L.dn_e);
  p.dn_p0 = (int*)(ws + L.dn_p0);
  p.dn_n = (int*)(ws + L.dn_n);
  p.act_hi = (uint16_t*)(ws + L.act_hi);
  p.act_lo = (uint16_t*)(ws + L.act_lo);
  p.part = (float*)(ws + L.part);
  p.out_f32 = out_f32;
  p.out_bf16 = (uint16_t*)out_bf16;
  p.n_experts = (int)n_experts;
  p.m = (int)m;
  p.d = (int)d;
  p.i = (int)i;
  p.top_k = top_k;
  p.limit = swiglu_limit;
  hipStream_t st = (hipStream_t)stream;
  p.n_sh_gu = shared ? (int)((m + kBigChunk - 1) / kBigChunk) : 0;
  p.n_sh_dn = shared ? (int)((m + kChunk - 1) / kChunk) : 0;
  const int64_t pk = m * top_k, touched = n_experts < pk ? n_experts : pk;
  // The wide kernels take calls of 24 pairs per expert and more (32 without the
  // shared expert, whose 64-pair chunks gain most) whose chunks fill the chip
  // about four times (two workgroups per CU, i / 128 or d / 256 of them per chunk
  // of ~48 pairs), and every call of one expert with more than a chunk of pairs.
  // Small / wide kernels, us, d = 4096, i = 2048, with the shared expert: 256
  // experts of 12, 16, 23, 32 and 47 pairs 844 / 867, 925 / 927, 1060 / 1018,
  // 1307 / 1195, 1640 / 1388; 64 experts of 28 pairs (two rounds of workgroups)
  // 319 / 358.  Without it: 256 experts of 28, 31 and 38 pairs 973 / 1012,
  // 1028 / 1031, 1143 / 1126 (d = 2048, fp32 scales 658 / 685, 702 / 698,
  // 780 / 738).  One bf16 expert of 40, 500 and 4096 pairs 154 / 117, 170 / 122,
  // 836 / 407.
  const bool one = n_experts == 1;
  p.wide = one ? pk > kChunk : pk >= (shared ? 24 : 32) * n_experts && pk * i >= (int64_t)12288 * 1024;
  p.small = p.wide && one ? 0 : kChunk;
  // One expert's chunks are of 32 pairs where these give either pass at most one
  // workgroup per CU, or one pass at most 3/4 of that (which 64-pair chunks would
  // halve): us with 32 / 64, d = 4096, i = 2048, bf16, 500 and 700 pairs 85 / 99,
  // 124 / 102; d = 1024, i = 2048, E8M0, 700, 1500 and 3000 pairs 44 / 55,
  // 53 / 64, 88 / 83 (the small kernels 49, 62, 94), bf16 60 / 66, 74 / 80,
  // 124 / 104.
  const int64_t n32 = (pk + kChunk - 1) / kChunk, gu_blocks = n32 * (i / kWideGuRows), dn_blocks = n32 * (d / kWideDnRows);
  const int64_t more = gu_blocks > dn_blocks ? gu_blocks : dn_blocks, fewer = gu_blocks + dn_blocks - more;
  const bool few = more <= device_cus() || 4 * fewer <= 3 * device_cus();
  p.big_chunk = p.wide && one && few ? kChunk : kBigChunk;
  p.by_rows = n_experts < 8;
  // chunks of the small kernels (beside the wide ones at most one per expert), and of the wide ones
  const int64_t C = p.wide ? (p.small ? touched : 0) : p.n_sh_gu + max_routed_chunks(m, n_experts, top_k);
  const int64_t Cd = p.wide ? C : p.n_sh_dn + max_routed_chunks(m, n_experts, top_k);
  const int64_t n_bigs = pk / (p.small + 1) < touched ? pk / (p.small + 1) : touched;
  const int64_t big = p.wide ? p.n_sh_gu + (pk / p.big_chunk + n_bigs + 7) / 8 * 8 : 0;
  // 256 threads per expert up to three pairs each, then 1024 (starting 16 waves
  // costs what they save before): us with 256 / 1024, 64 experts and 54, 600,
  // 1200, 1800, 12288 pairs 4.1 / 5.0, 5.2 / 5.4, 6.1 / 5.8, 7.8 / 6.1, 27 / 13;
  // one expert and 36, 600, 1200, 1800 3.3 / 4.2, 4.4 / 5.0, 5.8 / 5.8, 8.9 / 8.0
  // (a call of 1008 pairs of 64 small experts 39.0 / 38.6).
  if (pk <= 768) hipLaunchKernelGGL(prefill_group_kernel<256>, dim3((unsigned)n_experts + 1), dim3(256), 0, st, p);
  else hipLaunchKernelGGL(prefill_group_kernel<1024>, dim3((unsigned)n_experts + 1), dim3(1024), 0, st, p);
  int rc = check_launch(name);
  if (rc) return rc;
  const dim3 blk(kThreads);
  const bool e8m0 = scale_kind == HSMOE_SCALE_E8M0;
  if (big > 0) {
    const dim3 gu((unsigned)(big * (i / kWideGuRows)));
    if (e8m0) hipLaunchKernelGGL((prefill_wide_kernel<kFp4E8M0, false>), gu, blk, 0, st, p);
    else hipLaunchKernelGGL((prefill_wide_kernel<kFp4F32, false>), gu, blk, 0, st, p);
    if ((rc = check_launch(name))) return rc;
  }
  if (C > 0) {
    const dim3 gu((unsigned)(C * (i / kGuRows)));
    if (e8m0) hipLaunchKernelGGL(prefill_gate_up_kernel<kFp4E8M0>, gu, blk, 0, st, p);
    else hipLaunchKernelGGL(prefill_gate_up_kernel<kFp4F32>, gu, blk, 0, st, p);
    if ((rc = check_launch(name))) return rc;
  }
  if (big > 0) {
    const dim3 dn((unsigned)(big * (d / kWideDnRows)));
    if (e8m0) hipLaunchKernelGGL((prefill_wide_kernel<kFp4E8M0, true>), dn, blk, 0, st, p);
    else hipLaunchKernelGGL((prefill_wide_kernel<kFp4F32, true>), dn, blk, 0, st, p);
    if ((rc = check_launch(name))) return rc;
  }
  if (C > 0) {
    const dim3 dn((unsigned)(Cd * (d / kDnRows)));
    if (e8m0) hipLaunchKernelGGL(prefill_down_kernel<kFp4E8M0>, dn, blk, 0, st, p);
    else hipLaunchKernelGGL(prefill_down_kernel<kFp4F32>, dn, blk, 0, st, p);
    if ((rc = check_launch(name))) return rc;
  }
  hipLaunchKernelGGL(prefill_combine_kernel, dim3((unsigned)m, (unsigned)(d / (4 * kThreads))), dim3(kThreads), 0,
                     st, p);
  return check_launch(name);
}
