// bucket_impl.hpp -- device code of the stable (token, expert) bucketing,
// shared by the bucketing kernels (bucket.hip) and the fused route + bucket
// kernel of small batches (router.hip).
//
// Output positions follow the counting-sort definition: pair i (flat index
// t*k + j) of expert e goes to offsets[e] + #{i' < i : inds[i'] == e}.  That is
// exactly a stable argsort of the flat indices (reference gather_sort,
// src/common/switch_layers.cpp:17-30), computed with integer counts only, so
// it is bit-exact and deterministic.
#pragma once

#include "internal.hpp"

namespace moe {
namespace {

constexpr int kFusedMaxP = 4096;    // single-workgroup path up to this many pairs
constexpr int kFusedMaxE = 512;

__device__ __forceinline__ uint64_t lanemask_lt() {
  const int l = lane_id();
  return (l == 0) ? 0ull : (~0ull >> (64 - l));
}

// Mask of lanes holding the same key (keys < 2^nbits).
__device__ __forceinline__ uint64_t match_key(uint32_t key, int nbits) {
  uint64_t peers = ~0ull;
  for (int b = 0; b < nbits; ++b) {
    const bool bit = (key >> b) & 1u;
    const uint64_t m = __ballot(bit);
    peers &= bit ? m : ~m;
  }
  return peers;
}

// Block-wide exclusive scans of four ints per thread at once (NT threads, one
// LDS round, one barrier): v becomes the exclusive prefixes, *total the sums.
// May run once per kernel (its LDS is not protected against a second use).
template <int NT>
__device__ void block_exclusive_scan4(int4& v, int4* total) {
  __shared__ int4 wsum[NT / 64];
  const int lane = lane_id(), wave = threadIdx.x >> 6;
  // wave inclusive scans on DPP: shifts of 1, 2, 4, 8 within each row of 16
  // (lanes without a source add 0), then row 15's total into the next row
  // and lane 31's into rows 2 and 3
  auto wave_scan = [](int incl) {
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x111, 0xf, 0xf, true);  // row_shr:1
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x112, 0xf, 0xf, true);  // row_shr:2
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x114, 0xf, 0xf, true);  // row_shr:4
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x118, 0xf, 0xf, true);  // row_shr:8
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x142, 0xa, 0xf, false);  // row_bcast:15 -> rows 1, 3
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x143, 0xc, 0xf, false);  // row_bcast:31 -> rows 2, 3
    return incl;
  };
  const int4 in = make_int4(wave_scan(v.x), wave_scan(v.y), wave_scan(v.z), wave_scan(v.w));
  if (lane == 63) wsum[wave] = in;
  __syncthreads();
  int4 pre = make_int4(0, 0, 0, 0), tot = pre;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) {  // (every read in flight at once)
    const int4 t = wsum[w];
    if (w == wave) pre = tot;
    tot.x += t.x;
    tot.y += t.y;
    tot.z += t.z;
    tot.w += t.w;
  }
  v = make_int4(pre.x + in.x - v.x, pre.y + in.y - v.y, pre.z + in.z - v.z, pre.w + in.w - v.w);
  *total = tot;
}

// The expert of pair i (E: none, or out of range)
__device__ __forceinline__ uint32_t pair_expert(const uint32_t* inds, int64_t i, int64_t P, int E, const BucketOut& o) {
  if (i >= P) return static_cast<uint32_t>(E);
  const uint32_t v = inds[o.M == 1 ? i : static_cast<int64_t>(static_cast<uint32_t>(i) / static_cast<uint32_t>(o.M))];
  return v < static_cast<uint32_t>(E) ? v : static_cast<uint32_t>(E);
}

// The outputs at sorted position pos, which holds pair i
__device__ __forceinline__ void write_sorted(uint32_t i, int pos, int k, const BucketOut& o) {
  if (o.perm) o.perm[pos] = static_cast<int32_t>(i);
  if (o.sorted_token) o.sorted_token[pos] = static_cast<int32_t>(i / static_cast<uint32_t>(k));
  if (o.in_rows) {
    const uint32_t M = static_cast<uint32_t>(o.M), b = M == 1 ? i : i / M;
    const uint32_t row = (o.lhs ? o.lhs[b] : b) * M + (i - b * M);
    o.in_rows[pos] = static_cast<int32_t>(row);
    if (o.far && row >= o.far_row) *o.far = 1;
  }
}

// Scatter one sub-chunk of NW*64 consecutive pairs, this thread's being pair i
// of expert e (E: none), given running[e] = next free position of expert e.
// wcnt is [NW][E] LDS, all zero on entry and, unless this is the last
// sub-chunk, on exit.
template <int NW>
__device__ void scatter_subchunk(const uint32_t e, const int64_t i, int64_t P, int E, int k, int nbits, int* running,
                                 int* wcnt, const BucketOut& o, bool last) {
  const int wave = threadIdx.x >> 6;
  const uint64_t peers = match_key(e, nbits);
  const int rank = __popcll(peers & lanemask_lt());
  const bool leader = (peers & lanemask_lt()) == 0;
  const bool valid = e < static_cast<uint32_t>(E);
  if (valid && leader) wcnt[wave * E + e] = __popcll(peers);
  __syncthreads();
  if (valid) {
    int pos = running[e] + rank;
#pragma unroll
    for (int w = 0; w < NW; ++w) {  // (every read in flight at once)
      const int c = wcnt[w * E + e];
      pos += w < wave ? c : 0;
    }
    if (o.inv_perm) o.inv_perm[i] = pos;
    if (o.sorted_expert) o.sorted_expert[pos] = e;
    write_sorted(static_cast<uint32_t>(i), pos, k, o);
  } else if (o.zero_out && i < P) {
    for (int c = 0; c < o.zero_N; ++c) o.zero_out[i * o.zero_N + c] = 0;
  }
  if (last) return;
  __syncthreads();
  for (int x = threadIdx.x; x < E; x += NW * 64) {
    int s = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      s += wcnt[w * E + x];
      wcnt[w * E + x] = 0;
    }
    running[x] += s;
  }
  __syncthreads();
}

// Writes offsets (and the active-expert list and the token-tile table) from
// per-expert totals held in `tot` (LDS [E]); offs_lds [E+1] receives the
// offsets.  Requires E <= NT <= 1024; once per kernel.
template <int NT>
__device__ void finish_offsets(const int* tot, int64_t P, int E, int* offs_lds, const BucketOut& o) {
  static_assert(NT < 1 << 15, "the packed counts below (one per expert at most) stay under 2^15");
  const int e = threadIdx.x;
  const int c = e < E ? tot[e] : 0;
  int c4 = 0, c3 = 0, c2 = 0, c1 = 0;
  const int ct = e < E ? c : e == E ? o.sh_rows : 0;  // (the shared expert: tiles only; E < NT then)
  tile_counts(ct, c4, c3, c2, c1);
  const int nz = c > 0 ? 1 : 0;
  // rows, 128-row tiles, non-empty | 32-row tiles, 96- | 64-row tiles
  int4 ex = make_int4(c, c4, nz | (c1 << 16), c3 | (c2 << 16)), n;
  block_exclusive_scan4<NT>(ex, &n);
  if (e < E) offs_lds[e] = ex.x;
  if (e == 0) offs_lds[E] = n.x;
  if (o.offsets) {
    if (e < E) o.offsets[e] = ex.x;
    if (e == 0) o.offsets[E] = n.x;
  }
  // positions past the buckets (pairs of out-of-range experts): a valid row, so
  // that a pass over all P positions reads in bounds
  if (o.in_rows)
    for (int64_t x = static_cast<int64_t>(n.x) + e; x < P; x += NT) o.in_rows[x] = 0;
  if (o.active) {
    // one 16-byte record per slot, so a GEMM workgroup finds its expert and
    // rows with a single load; slots past the count get rows = 0
    const int na = n.z & 0xffff;
    int4* rec = reinterpret_cast<int4*>(o.active);
    if (nz) rec[ex.z & 0xffff] = make_int4(e, ex.x, c, 0);
    if (e < E && e >= na) rec[e] = make_int4(0, 0, 0, 0);
    if (e == 0 && o.num_active) o.num_active[0] = na;
  }
  if (__builtin_expect(o.tiles != nullptr, 0)) {  // the large-bucket GEMM's token-tile table (out of line)
    const int n4 = n.y, n3 = n.w & 0xffff, n2 = n.w >> 16, n1 = n.z >> 16;
    // tiles of at most 64 rows: a 128-row one as two, a 96-row one as 64 + 32
    const bool half = 2 * (n4 + n3) + n2 + n1 <= o.half_max.tiles &&
                      4 * n4 + 3 * n3 + 2 * n2 + n1 <= o.half_max.units;  // (uniform)
    if (e == 0)
      reinterpret_cast<int4*>(o.tiles)[0] = half ? make_int4(0, 0, 2 * n4 + n3 + n2, n3 + n1) : make_int4(n4, n3, n2, n1);
    if (e <= E)
      write_tiles(o.tiles, e < E ? e : -1, e < E ? ex.x : 0, ct, half, c4, c3, c2, c1, ex.y, ex.w & 0xffff,
                  ex.w >> 16, ex.z >> 16, n4, n3, n2);
  }
  __syncthreads();
}

// Orders this wave's LDS accesses: its earlier LDS reads and writes complete
// (from every lane) before later ones, and the compiler keeps them in order.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
}

// LDS ints of the single-workgroup bucketing of P pairs with NW waves
template <int NW>
__host__ __device__ constexpr size_t bucket_fused_lds_ints(int E, int64_t P) {
  return static_cast<size_t>(E + (E + 1) + NW * E) + static_cast<size_t>(P);
}

// The bucketing of P <= kFusedMaxP pairs by one workgroup of NW waves (E <=
// kFusedMaxE); lds: bucket_fused_lds_ints<NW>(E, P) ints.  Every thread of the
// workgroup calls it.  Wave w takes a contiguous run of pairs, 64 a round: each
// pair's rank among the wave's pairs of its expert is its rank in the round
// (match_key) plus the wave's count so far, so no barrier runs between rounds;
// then the counts are scanned over the waves and the experts, and the sorted
// outputs, collected in LDS, are written in order.  Bound by the rounds' ballots
// and LDS round trips on one CU.  Measured (events, 128 experts): 15.7 -> 11.4
// us for 4000 pairs, 11.4 -> 9.3 for 2048, against one LDS histogram and then
// sub-chunks of 1024 pairs with three barriers and 16 count reads per pair.
template <int NW>
__device__ void bucket_fused_body(const uint32_t* __restrict__ inds, int64_t P, int E, int k, int nbits,
                                  const BucketOut& o, int* lds) {
  constexpr int kPer = (kFusedMaxP + NW * 64 - 1) / (NW * 64);  // rounds at most
  int* tot = lds;                   // [E]
  int* offs = tot + E;              // [E+1]
  int* wcnt = offs + E + 1;         // [NW][E]
  int* sp = wcnt + NW * E;          // [P]
  if (o.far && threadIdx.x == 0) *o.far = 0;
  const int lane = lane_id(), wave = threadIdx.x >> 6;
  const int rounds = (static_cast<int>(P) + NW * 64 - 1) / (NW * 64);
  const int i0 = wave * rounds * 64 + lane;
  uint32_t ex[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) ex[j] = pair_expert(inds, j < rounds ? i0 + 64 * j : P, P, E, o);
  for (int x = threadIdx.x; x < NW * E; x += NW * 64) wcnt[x] = 0;
  __syncthreads();
  int* mine = wcnt + wave * E;
  int rank[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    rank[j] = 0;
    if (j >= rounds) continue;  // (uniform)
    const uint64_t peers = match_key(ex[j], nbits);
    const int below = __popcll(peers & lanemask_lt());
    const bool valid = ex[j] < static_cast<uint32_t>(E);
    const int before = valid ? mine[ex[j]] : 0;
    rank[j] = before + below;
    wave_lds_sync();  // every lane has read its count
    if (valid && below == 0) mine[ex[j]] = before + __popcll(peers);
    wave_lds_sync();
  }
  __syncthreads();
  for (int x = threadIdx.x; x < E; x += NW * 64) {  // wave counts -> starts within the expert, and its total
    int c[NW], s = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) c[w] = wcnt[w * E + x];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      wcnt[w * E + x] = s;
      s += c[w];
    }
    tot[x] = s;
  }
  __syncthreads();
  finish_offsets<NW * 64>(tot, P, E, offs, o);
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int i = i0 + 64 * j;
    if (j >= rounds || i >= P) continue;
    if (ex[j] < static_cast<uint32_t>(E)) {
      const int pos = offs[ex[j]] + mine[ex[j]] + rank[j];
      sp[pos] = i;
      if (o.inv_perm) o.inv_perm[i] = pos;
      if (o.sorted_expert) o.sorted_expert[pos] = ex[j];
    } else if (o.zero_out) {
      for (int c = 0; c < o.zero_N; ++c) o.zero_out[static_cast<int64_t>(i) * o.zero_N + c] = 0;
    }
  }
  __syncthreads();
  const int n = offs[E];  // pairs in buckets
  for (int pos = threadIdx.x; pos < n; pos += NW * 64) write_sorted(static_cast<uint32_t>(sp[pos]), pos, k, o);
}

// Wave-wide exclusive prefix sum of one int per lane; *total gets the sum.
__device__ __forceinline__ int wave_exclusive_scan(int v, int* total) {
  const int lane = lane_id();
  int incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(incl, off, 64);
    if (lane >= off) incl += o;
  }
  *total = __shfl(incl, 63, 64);
  return incl - v;
}

// The stable bucketing of a small batch (P <= kSmallMaxP pairs, E <= 512)
// by one wave with no workgroup barrier: histogram by LDS atomics, the
// exclusive scan over the experts (lane l owns experts V*l .. V*l + V - 1),
// then the scatter 64 pairs at a time, each pair's position its expert's
// running offset plus its rank among the chunk's pairs of the same expert.
// Same outputs as bucket_fused_body except the token-tile table.  inds: LDS
// [P]; cnt, offs: LDS [E + 1] each.  Only the calling wave may touch them.
constexpr int kSmallMaxP = 256;
[[maybe_unused]] __device__ void bucket_small_wave(const uint32_t* inds, int P, int E, int k, int nbits, const BucketOut& o,
                                  int* cnt, int* offs) {
  const int lane = lane_id();
  for (int x = lane; x <= E; x += 64) cnt[x] = 0;
  wave_lds_sync();
  for (int i = lane; i < P; i += 64) {
    const uint32_t v = inds[i];
    if (v < static_cast<uint32_t>(E)) atomicAdd(&cnt[v], 1);
  }
  wave_lds_sync();
  const int V = (E + 63) >> 6;
  int c[8];
  int sum = 0, nzc = 0;
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    const int e = V * lane + v;
    c[v] = v < V && e < E ? cnt[e] : 0;
    sum += c[v];
    nzc += c[v] > 0 ? 1 : 0;
  }
  int total, nact;
  int run = wave_exclusive_scan(sum, &total);
  int slot = wave_exclusive_scan(nzc, &nact);
  int4* rec = reinterpret_cast<int4*>(o.active);
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    const int e = V * lane + v;
    if (v < V && e < E) {
      offs[e] = run;
      if (o.offsets) o.offsets[e] = run;
      if (rec && c[v] > 0) rec[slot++] = make_int4(e, run, c[v], 0);
      run += c[v];
    }
  }
  if (lane == 0) {
    offs[E] = total;
    if (o.offsets) o.offsets[E] = total;
    if (o.num_active) o.num_active[0] = nact;
  }
  if (rec)
    for (int x = nact + lane; x < E; x += 64) rec[x] = make_int4(0, 0, 0, 0);
  wave_lds_sync();
  for (int first = 0; first < P; first += 64) {
    const int i = first + lane;
    uint32_t e = static_cast<uint32_t>(E);  // sentinel for "no pair"
    if (i < P) {
      const uint32_t v = inds[i];
      if (v < static_cast<uint32_t>(E)) e = v;
    }
    const uint64_t peers = match_key(e, nbits);
    const uint64_t below = peers & lanemask_lt();
    const bool valid = e < static_cast<uint32_t>(E);
    const int base = valid ? offs[e] : 0;
    if (valid) {
      const int pos = base + __popcll(below);
      if (o.perm) o.perm[pos] = i;
      if (o.inv_perm) o.inv_perm[i] = pos;
      if (o.sorted_expert) o.sorted_expert[pos] = e;
      if (o.sorted_token) o.sorted_token[pos] = i / k;
    }
    wave_lds_sync();
    if (valid && below == 0) offs[e] = base + __popcll(peers);
    wave_lds_sync();
  }
}

int bits_for(int E) {
  int n = 0;
  while ((1 << n) <= E) ++n;  // keys 0..E (E = sentinel)
  return n;
}

}  // namespace
}  // namespace moe
