// gather_mm.hip -- grouped dense (bf16) matmul, the gather_mm that
// SwitchLinear runs for experts that are not quantized (reference
// src/common/switch_layers.cpp:103-109), gfx950.
//
// Rows are the expert buckets of the sorted pairs, as in the quantized
// kernels (qmm.hip), cut into the token tiles of the bucketing's table
// (tile_counts).  fp32 accumulation, one bf16 rounding (and SwitchLinear's
// bias, switch_layers.cpp:111-114, on the rounded value).
#include "internal.hpp"

namespace moe {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// A workgroup of four waves computes a tile of 32*MT bucket rows x 128*NT
// weight rows; wave w owns every token row and weight rows 32*NT*w .. +32*NT-1
// of the tile.  Each 32-wide K step (64 bytes of a row) of the token and weight
// rows goes straight to LDS (4 lanes per row, whole half lines), into a ring of
// ST steps: the loads of step s + ST - 1 are issued when step s starts, so
// ST - 1 steps are in flight, and one LDS-only barrier per step orders the
// ring.  The 16-byte chunk c of row r sits at slot c ^ ((r / 4) % 4): the 16
// lanes that a 128-bit LDS read serves per clock never share a bank.
//
// What bounds it: up to a few dozen rows per expert the weights' HBM stream
// (every weight is read once per token tile).  At 94 rows (T = 1500 below) the
// weights come at 3.5 TB/s, and by counters neither the MFMA pipe (busy 15 % of
// the cycles) nor LDS (0.13 conflict cycles per instruction, 1 % of the waves'
// time waiting for it) is what it waits for: the waves wait for loads and the
// step's barrier 25 % of their time and to issue 62 %.  Measured on [E 128, N 768,
// K 2048], k = 8, the whole gather_mm call (us): T = 1500 916 -> 116, T = 4096
// 2427 -> 179, T = 256 194 -> 94, T = 16 57 -> 40, T = 1 23.8 -> 19.7, against a
// kernel without LDS whose waves read every weight row from L2 again for each 32
// tokens and awaited each step's loads before its MFMAs.
struct GMArgs {
  const uint16_t* x;
  const int32_t* row_in;
  const int32_t* row_out;
  const int32_t* tiles;  // token-tile table (tile_counts / write_tiles)
  const uint16_t* w;
  const uint16_t* lb;
  int N, K, ntiles;
  int wide;              // 16-byte output stores (N % 8 == 0, out aligned)
  uint16_t* out;
};

template <int MT, int NT, int ST>
constexpr int mm_tile_lds() {
  constexpr int ring = ST * (32 * MT + 128 * NT) * 64, outb = 32 * MT * (128 * NT + 8) * 2;
  return ring > outb ? ring : outb;
}

template <int MT, int NT, int ST>
__device__ __forceinline__ void mm_tile(const GMArgs& a, uint8_t* lds, const int e, const int row0,
                                        const int rows, const int ntile) {
  constexpr int BM = 32 * MT, BN = 128 * NT;
  constexpr int kStage = (BM + BN) * 64;
  constexpr int AI = (MT + 1) / 2;  // DMA instructions per wave per step: token rows (16 rows each) ...
  constexpr int BI = 2 * NT;        // ... and the wave's weight rows
  constexpr int OS = BN + 8;        // LDS row stride of the output tile (elements)
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, l32 = lane & 31;
  const int S = a.K >> 5;

  // producers: lane -> row lane/4 of its instruction's 16 rows, LDS slot
  // lane%4.  2*MT instructions cover the token rows; a wave past them (MT odd)
  // repeats an instruction of another wave, the same bytes to the same place,
  // so that every wave issues AI of them and the wait count is one constant
  const uint16_t* asrc[AI];
  int adst[AI];
#pragma unroll
  for (int j = 0; j < AI; ++j) {
    const int ins = (wave + 4 * j) % (2 * MT);
    const int r = 16 * ins + (lane >> 2);
    const int pos = row0 + min(r, rows - 1);  // rows past the tile: its last row again (never stored)
    asrc[j] = a.x + static_cast<int64_t>(a.row_in[pos]) * a.K + 8 * ((lane & 3) ^ ((r >> 2) & 3));
    adst[j] = ins * 1024;
  }
  const uint16_t* bsrc[BI];
#pragma unroll
  for (int j = 0; j < BI; ++j) {
    const int r = 32 * NT * wave + 16 * j + (lane >> 2);
    const int n = min(ntile * BN + r, a.N - 1);  // columns past N: the last row again (never stored)
    bsrc[j] = a.w + (static_cast<int64_t>(e) * a.N + n) * a.K + 8 * ((lane & 3) ^ ((r >> 2) & 3));
  }
  auto issue = [&](int s, int stage) {
    const int k = 32 * min(s, S - 1);  // past the end: the last step again (in bounds, never read)
    uint8_t* sb = lds + stage * kStage;
#pragma unroll
    for (int j = 0; j < AI; ++j) load_lds16(asrc[j] + k, sb + adst[j]);
#pragma unroll
    for (int j = 0; j < BI; ++j) load_lds16(bsrc[j] + k, sb + BM * 64 + (32 * NT * wave + 16 * j) * 64);
  };
  // consumers: lane half h of substep u holds K 16u + 8h .. +7, chunk 2u + h
  int off[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) off[u] = l32 * 64 + 16 * ((2 * u + h) ^ ((l32 >> 2) & 3));

  f32x16 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mt][nt][r] = 0.0f;

#pragma unroll
  for (int i = 0; i < ST - 1; ++i) issue(i, i);
  int st = 0;
  for (int s = 0; s < S; ++s) {
    wait_vmcnt<(ST - 2) * (AI + BI)>();  // this wave's loads of step s have landed (later steps' may be in flight)
    lds_barrier();                       // every wave's have, and step s - 1's stage is free
    issue(s + ST - 1, st == 0 ? ST - 1 : st - 1);
    const uint8_t* sa = lds + st * kStage;
    const uint8_t* sb = sa + BM * 64 + 32 * NT * wave * 64;
    bf16x8 bf[NT][2];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int u = 0; u < 2; ++u)
        bf[nt][u] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(sb + 32 * 64 * nt + off[u]));
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      bf16x8 af[2];
#pragma unroll
      for (int u = 0; u < 2; ++u)
        af[u] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(sa + 32 * 64 * mt + off[u]));
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[u], bf[nt][u], acc[mt][nt], 0, 0, 0);
    }
    st = st == ST - 1 ? 0 : st + 1;
  }

  // SwitchLinear's bias of this lane's columns, and the output rows of this
  // thread's chunks, loaded before any store
  constexpr int CPR = BN / 8, RPP = 256 / CPR, NPASS = BM / RPP;  // chunks per row, rows per pass
  float lbv[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int n = min(ntile * BN + 32 * NT * wave + 32 * nt + l32, a.N - 1);
    lbv[nt] = a.lb ? bf2f(a.lb[static_cast<int64_t>(e) * a.N + n]) : 0.0f;
  }
  int orow[NPASS];
#pragma unroll
  for (int j = 0; j < NPASS; ++j) {
    const int m = min(tid / CPR + RPP * j, rows - 1);
    orow[j] = a.row_out ? a.row_out[row0 + m] : row0 + m;
  }
  wait_vmcnt<0>();  // no DMA into the ring outstanding, the loads above landed
  lds_barrier();
  // the tile goes through LDS for 16-byte row-segment stores.  D layout of the
  // 32x32 MFMA: column lane%32, row 8*(r/4) + 4*(lane/32) + r%4; rows r and
  // r + 1 of a lane pair are exchanged (DPP), so each lane writes one dword of
  // two adjacent columns
  uint16_t* ot = reinterpret_cast<uint16_t*>(lds);
  const bool odd = l32 & 1;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const int m0 = mt * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
        float v0 = acc[mt][nt][r], v1 = acc[mt][nt][r + 1];
        if (a.lb) {
          v0 = bfr(v0) + lbv[nt];
          v1 = bfr(v1) + lbv[nt];
        }
        const float partner = dpp_f<kDppQuadXor1>(odd ? v0 : v1);
        *reinterpret_cast<uint32_t*>(ot + (m0 + (odd ? 1 : 0)) * OS + 32 * NT * wave + 32 * nt + (l32 & ~1)) =
            odd ? pack_bf16x2(partner, v1) : pack_bf16x2(v0, partner);
      }
  lds_barrier();
  const int c0 = 8 * (tid % CPR), col = ntile * BN + c0;
#pragma unroll
  for (int j = 0; j < NPASS; ++j) {
    const int m = tid / CPR + RPP * j;
    if (m >= rows || col >= a.N) continue;
    const uint16_t* src = ot + m * OS + c0;
    uint16_t* dst = a.out + static_cast<int64_t>(orow[j]) * a.N + col;
    if (a.wide)
      __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(src), reinterpret_cast<u32x4*>(dst));
    else
      for (int c = 0; c < 8 && col + c < a.N; ++c) dst[c] = src[c];
  }
}

// Workgroup -> (token tile, column tile): the large-bucket GEMM's order (each
// XCD a contiguous eighth of the 128- and 96-row tiles, whose column tiles and
// neighbours share its L2, then the short tiles dealt round robin).  SHORT:
// every tile as a sequence of 32-row ones (few rows per expert: almost every
// tile is one; its LDS then holds a deeper ring and more workgroups per CU).
template <int NT, int ST, bool SHORT>
__global__ __launch_bounds__(256, 2) void grouped_mm_tile_kernel(GMArgs a) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[mm_tile_lds<SHORT ? 1 : 4, NT, ST>()];
  const int4 cnt = reinterpret_cast<const int4*>(a.tiles)[0];  // {n4, n3, n2, n1}
  const int nt = a.ntiles;
  const int xcd = blockIdx.x & 7, i = blockIdx.x >> 3;
  const int nlong = cnt.x + cnt.y;
  const int vl = nlong * nt;
  const int perl = (vl + 7) >> 3;
  int slot, ntile;
  if (i < perl) {
    const int v = xcd * perl + i;
    if (v >= vl) return;
    slot = v / nt;
    ntile = v - slot * nt;
  } else {
    const int v = (i - perl) * 8 + xcd;
    if (v >= (cnt.z + cnt.w) * nt) return;
    const int q = v / nt;
    ntile = v - q * nt;
    slot = nlong + q;
  }
  const int4 t = reinterpret_cast<const int4*>(a.tiles)[1 + slot];
  if constexpr (SHORT) {
    for (int m = 0; m < t.z; m += 32) {
      if (m > 0) lds_barrier();  // the output staging of the rows before has been read
      mm_tile<1, NT, ST>(a, lds, t.x, t.y + m, min(32, t.z - m), ntile);
    }
  } else {
    if (slot < cnt.x) mm_tile<4, NT, ST>(a, lds, t.x, t.y, t.z, ntile);
    else if (slot < nlong) mm_tile<3, NT, ST>(a, lds, t.x, t.y, t.z, ntile);
    else if (slot < nlong + cnt.z) mm_tile<2, NT, ST>(a, lds, t.x, t.y, t.z, ntile);
    else mm_tile<1, NT, ST>(a, lds, t.x, t.y, t.z, ntile);
  }
}

}  // namespace

int grouped_mm(const uint16_t* x, const int32_t* row_in, const int32_t* row_out, const int32_t* tiles, int slots,
               int64_t P, const uint16_t* w, const uint16_t* linear_bias, int N, int K, uint16_t* out,
               hipStream_t stream) {
  if (!x || !row_in || !tiles || !w || !out || slots < 0 || N <= 0 || K <= 0) return MOE_E_INVALID_ARG;
  if (K % 32 != 0 || (reinterpret_cast<uintptr_t>(x) & 15u) || (reinterpret_cast<uintptr_t>(w) & 15u))
    return MOE_E_UNSUPPORTED;
  if (slots == 0) return MOE_OK;
  // Measured (whole calls, us; five-stage 32-row tiles | 128 columns | 256
  // columns per workgroup), shapes [E, N, K]:
  //   rows per expert 4:  [128, 768, 2048]  87 |  92 | 100, [8, 2048, 4096] 49 | 59 | 69
  //   8:                  [128, 768, 2048] 104 |  98 | 105, [8, 2048, 4096] 53 | 61 | 75
  //   12 - 16:            [128, 768, 2048] 121 | 104 | 112, [64, 512, 2304] 52 | 45 | 58
  //   32 - 94:            [128, 768, 2048] 239 | 135 | 128 (94), [32, 1024, 1024] 43 | 27 | 38 (32)
  //   256 - 1024:         [128, 768, 2048] 459 | 240 | 205, [8, 2048, 4096] 556 | 258 | 245,
  //                       [32, 1024, 1024] 145 |  74 |  81 (K = 1024: the tile's fill and epilogue weigh more)
  // (nearly even loads; 32-row tiles | 128 columns where an eighth of the experts
  // hold all rows, the first shape: 4 rows per expert on average 32 | 25, 8: 44 |
  // 27.  The kernel before took 54 and 81.)
  // so: 32-row tiles up to 8 rows per expert, 256 columns (half the LDS reads
  // per MFMA, two workgroups per CU) from 32 rows where K >= 2048 and the grid
  // still fills the CUs.
  const int64_t ttiles = P / 128 + std::min<int64_t>(slots, P);
  const int nt2 = (N + 255) / 256, nt1 = (N + 127) / 128;
  const bool few = P <= 8 * static_cast<int64_t>(slots);
  const bool wide_n = !few && P >= 32 * static_cast<int64_t>(slots) && K >= 2048 && ttiles * nt2 >= 256;
  const int64_t nt = wide_n ? nt2 : nt1;
  // per XCD: an eighth of the 128- and 96-row tiles, then of the short ones
  // (n4 + n3 <= P/128 + slots, n2 + n1 <= slots: one remainder tile per expert)
  const int64_t grid = 8 * (((P / 128 + slots) * nt + 7) / 8 + (2 * slots * nt + 7) / 8);
  if (grid > 0x7fffffffLL) return MOE_E_UNSUPPORTED;
  const dim3 g(static_cast<unsigned>(grid));
  const int wide = N % 8 == 0 && (reinterpret_cast<uintptr_t>(out) & 15u) == 0;
  GMArgs a{x, row_in, row_out, tiles, w, linear_bias, N, K, static_cast<int>(nt), wide, out};
  if (few)
    MOE_LAUNCH("gather_mm", (grouped_mm_tile_kernel<1, 5, true>), g, dim3(256), 0, stream, a);
  else if (wide_n)
    MOE_LAUNCH("gather_mm", (grouped_mm_tile_kernel<2, 3, false>), g, dim3(256), 0, stream, a);
  else
    MOE_LAUNCH("gather_mm", (grouped_mm_tile_kernel<1, 3, false>), g, dim3(256), 0, stream, a);
  return launch_status("gather_mm");
}

}  // namespace moe
