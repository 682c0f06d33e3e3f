// E8-D4 Linear for 17..128 rows (a full serving batch, a short prompt chunk)
// on the matrix cores, every index decoded once for up to 64 rows.
//
// The operand mapping of decode_mfma.hip (decoded weights as the MFMA's A
// operand in registers, rows of x as its 16 columns), with TT groups of 16
// rows per workgroup: a decoded operand is used TT times.
//
// Tiles.  A workgroup (8 waves) owns 8 block rows (64 outputs) of one layer
// and 16·TT rows of x; its waves split its columns in blocks of 64.  Layers
// with few tiles have their columns split over P workgroups more, whose fp32
// sums meet in the workspace as in decode_mfma.hip.  More than 64 rows are
// token groups of the grid, the groups of a tile placed on one XCD so that
// its indices come from memory once.
//
// Loads.  Each wave brings its own blocks of x, indices and scales into LDS by
// DMA, two or three blocks deep, and waits for exactly those (no barrier in
// the column loop).  An x fragment is 16 rows at one 16-byte chunk: loaded
// from memory as that, every lane is a cache line of its own (62 cycles of
// the CU's address unit per instruction); by DMA four or eight consecutive
// lanes share a line (27 cycles).  That address time is what bounds the column
// loop (64 rows, one workgroup per CU: 3.3 us per 1024 columns; a 16-wave form
// kept 3.5 of its 3.7 with the table lookups and the MFMAs taken out), beside
// a start and end of ~8 us.  Two row tiles per workgroup (half the x loads per
// output, 219 registers) and 16 waves per workgroup measured slower or level.
//
// Measured (Llama-2-7B, q|k|v / o / gate|up / down): 32 rows 18 / 13 / 22 /
// 17 us, 64 rows 20 / 16 / 33 / 20, 128 rows 32 / 16 / 51 / 25; a 16-row slice
// of decode_mfma.hip, of which these rows took two, four and eight, 12 / 8 /
// 22 / 13.
//
// Scales.  h is on x, as in decode_mfma.hip: the operand is fp16(x · hs) with
// hs = fp16(h · 2^-e), |hs| <= 1, where 2^e >= max |h| over the wave's own
// columns (no wave waits for another's); 2^e is restored in fp32 before the
// waves' sums meet.  The S row is on the weight: fp16(t · S).  bf16 x is taken
// to fp16 first, exactly in fp16's normal range.
//
// Critical blocks replace the table vectors in registers: the tile's CSR
// entries are staged in LDS and each lane walks those of its block row with a
// cursor.  Entries past the stage are corrected after the column loop.

#include <type_traits>

#include "mfma_decode.h"

namespace eptq {
namespace dwide {

using dec::gp;
using dec::h2;
using dec::pk_mul;
using mdec::ld16;
using mdec::rsrc;

constexpr int kTile = 8;          // block rows per tile (64 outputs)
constexpr int kS = 8;             // waves per workgroup
constexpr int kNT = 64 * kS;
constexpr int kRedLd = 68;        // floats per row of x in a wave's partial sums
constexpr int kFar = 0x40000000;  // a buffer offset past every operand (a load there reads zeros)
constexpr int kMaxParts = 8;
constexpr int kSc1 = 16;          // buffer access at device scope
constexpr int kLdsBytes = 160 * 1024 - 4608;   // less the static part (the table above all)

// Column blocks and dynamic LDS.  Up to 32 rows of x: blocks of 32 columns,
// three in the ring, so that two workgroups fit a CU and one's start and end
// run under the other's column loop.  Up to 64 rows: blocks of 64 columns (a
// whole cache line of each row per load), two in the ring.
// During the column loop: per wave the ring, each slot the block's x tile
// (16·TT rows), index tile (8 rows) and scale rows (h and S), then the staged
// critical blocks (18 bytes each).  After it: the waves' partial sums
// red[kS][32][kRedLd], 32 rows of x at a time.
template <int TT> struct Lay {
  static constexpr int kBlk = TT <= 2 ? 32 : 64, kRing = TT <= 2 ? 3 : 2;
  static constexpr int CH = kBlk / 8, RB = 2 * kBlk;       // 16-byte chunks and bytes of a row
  static constexpr int XB = 16 * TT * RB, QB = kTile * RB, HB = 2 * RB;
  static constexpr int Slot = XB + QB + HB;
  static constexpr int E0 = kS * kRing * Slot;
  static constexpr int Red = kS * 32 * kRedLd * 4;
  static constexpr int kRoom = ((TT <= 2 ? 80 * 1024 - 4608 : kLdsBytes) - E0) / 18 / 8 * 8;
  static constexpr int kEnt = kRoom < 1024 ? kRoom : 1024;
  static constexpr int Loop = E0 + kEnt * 18;
  static constexpr int Bytes = Loop > Red ? Loop : Red;
  static_assert(kEnt >= 384 && Bytes <= kLdsBytes, "room for the usual critical blocks");
  // Chunk c of row r lies at place c ^ swz(r): the fragment reads (16 rows at
  // one chunk) then hit distinct banks.
  __device__ static constexpr int swz(int r) { return kBlk == 32 ? (r >> 2) & 3 : (r >> 1) & 7; }
};

struct Split {
  int units;    // workgroups of one token group: T1 whole tiles, then P per tile
  int P, T1, TG;
  int tiles;
  int* cnt;     // arrival counters [TG][tiles]
  float* part;  // sums [TG][split tile][P][16·TT][64]
};

// One LDS DMA instruction: lane l's 16 bytes at buffer offset voff (at address
// p) go to LDS byte lds + 16·l.  Offsets past the buffer write zeros.  In
// assembly, and counted by the waits below, because the compiler would make
// every later LDS read wait for all of them.
__device__ __forceinline__ void dma16(u32x4 r, int voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds), "v"(voff), "s"(r)
               : "memory");
}
__device__ __forceinline__ void dma16g(const void* p, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(p) : "memory");
}
__device__ __forceinline__ u32x4 desc(const void* p, int bytes) {
  const uint64_t v = (uint64_t)p;
  return (u32x4){(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v),
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32)) & 0xffffu,
                 (uint32_t)__builtin_amdgcn_readfirstlane(bytes), (uint32_t)dec::kBufferWord3};
}

template <int TT, bool HAS_S, typename XT>
__global__ __launch_bounds__(kNT, TT <= 2 ? 4 : 2) void k_decode_wide(MultiArgs ma, Split sp) {
  using L = Lay<TT>;
  constexpr int kBlk = L::kBlk, kRing = L::kRing;
  __shared__ f16x4 tab[512];
  __shared__ int rfirst[kTile], rcnt[kTile];   // per block row: first entry and entries in this part's columns
  __shared__ int last_part;
  extern __shared__ __attribute__((aligned(256))) char dyn[];

  // Workgroups are dealt to the 8 XCDs round-robin: the token groups of a
  // unit sit 8 workgroups apart.
  const int g = (int)blockIdx.x;
  const int tg = (g >> 3) % sp.TG;
  const int unit = ((g >> 3) / sp.TG) * 8 + (g & 7);
  if (unit >= sp.units) return;
  const int Pt = unit < sp.T1 ? 1 : sp.P;
  const int tile_g = unit < sp.T1 ? unit : sp.T1 + (unit - sp.T1) / sp.P;
  const int part = unit < sp.T1 ? 0 : (unit - sp.T1) - (tile_g - sp.T1) * sp.P;
  int li = 0;
#pragma unroll
  for (int l = 1; l < kMaxLayers; ++l)
    if (l < ma.n && tile_g >= ma.start[l]) li = l;
  const LinearArgs a = li == 0 ? ma.l[0] : li == 1 ? ma.l[1] : li == 2 ? ma.l[2] : ma.l[3];
  const int tile = tile_g - ma.start[li];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int M = a.M, N = a.N, ldx = a.ldx;
  const int m0 = tile * kTile;
  const int t0 = tg * 16 * TT;
  const int Bt = a.B - t0 < 16 * TT ? a.B - t0 : 16 * TT;   // rows of x here
  u32x4* const eov = (u32x4*)(dyn + L::E0);
  uint16_t* const ecol = (uint16_t*)(eov + L::kEnt);
  float (*red)[32][kRedLd] = (float (*)[32][kRedLd])dyn;

  // This wave's column blocks [blo, blo + n) of the part's [plo, plo + pnb).
  const int nb = (N + kBlk - 1) / kBlk;
  const int plo = part * nb / Pt, pnb = (part + 1) * nb / Pt - plo;
  const int blo = plo + wave * pnb / kS, n = plo + (wave + 1) * pnb / kS - blo;
  const int i = lane & 15, kg = lane >> 4;

  // Table, row pointers and first entries of block row `wave`, h (its maximum
  // over the wave's columns).
  static_assert(kNT == 512 && kS == kTile, "a table row per thread, a block row per wave");
  const f16x4 tload = *gp((const f16x4*)a.codes + tid);
  const int mr = m0 + wave;
  const int r0 = mr < M ? a.O_row_ptr[mr] : 0, r1 = mr < M ? a.O_row_ptr[mr + 1] : 0;
  const __amdgpu_buffer_rsrc_t rh = rsrc(a.h, N * 2);
  constexpr int kH = 4;   // up to 2048 columns per wave at once
  const int nch = n * (kBlk / 8), c0 = blo * (kBlk / 8);
  u32x4 hw[kH];
#pragma unroll
  for (int k = 0; k < kH; ++k) hw[k] = ld16(rh, 64 * k + lane < nch ? (c0 + 64 * k + lane) * 16 : kFar);
  int col0 = 0x7fffffff;
  u32x4 eo0 = {};
  if (r0 + lane < r1) {
    col0 = gp(a.O_col)[r0 + lane];
    eo0 = *gp((const u32x4*)a.O + r0 + lane);
  }

  // LDS DMA of block k into a ring slot, kRow lanes' 16-byte chunks a row.
  const u32x4 dx = desc(a.x + (size_t)t0 * ldx, ((Bt - 1) * ldx + N) * 2);
  const uint32_t lds0 =
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)dyn + (uint32_t)wave * (kRing * L::Slot);
  constexpr int kRow = L::CH, kRows = 64 / kRow;         // rows per instruction
  const int drow = lane / kRow, dl = lane % kRow;
  constexpr int kQRows = kRows < kTile ? kRows : kTile;
  static_assert(kQRows == kTile, "the index tile is one instruction");
  const int qr = m0 + (drow & 7) < M ? m0 + (drow & 7) : M - 1;   // rows past M: loaded, never stored
  const int qc = 8 * (dl ^ L::swz(drow & 7));
  const int16_t* const qp = a.Q + (size_t)qr * N;
  // Scale rows: kRow lanes h, kRow lanes S; with 32-column blocks they ride in
  // the index tile's instruction (lanes 32 ..).
  const int hl = kBlk == 32 ? lane - 32 : lane;
  const f16* const hp = HAS_S && hl >= kRow ? a.S + (size_t)((8 * m0) / a.qb) * N : a.h;
  const bool hlive = hl >= 0 && hl < (HAS_S ? 2 : 1) * kRow;
  constexpr int kXI = 16 * TT / kRows;                   // instructions of the x tile
  int xo[kXI], xc[kXI];
#pragma unroll
  for (int u = 0; u < kXI; ++u) {
    const int row = kRows * u + drow;
    xc[u] = 8 * (dl ^ L::swz(row & 15));
    xo[u] = (row * ldx + xc[u]) * 2;
  }
  constexpr int C = kXI + (kBlk == 32 ? 1 : 2);          // DMA instructions per block
  auto issue = [&](int slot, int k) {
    const int col = (blo + k) * kBlk;                    // uniform
    const uint32_t base = lds0 + slot * L::Slot;
    // Index and scale chunks past N read the row's last one (x is zero there).
    const void* q = qp + (col + qc < N ? col + qc : N - 8);
    const int hc = col + 8 * (hl & (kRow - 1));
    const void* h = hp + (hc < N ? hc : N - 8);
    if (kBlk == 32) {
      if (lane < 32 || hlive) dma16g(lane < 32 ? q : h, base + L::XB);
    } else {
      dma16g(q, base + L::XB);
      if (hlive) dma16g(h, base + L::XB + L::QB);
    }
#pragma unroll
    for (int u = 0; u < kXI; ++u) dma16(dx, col + xc[u] < N ? xo[u] + col * 2 : kFar, base + 1024 * u);
  };

  float mx = 0.0f;
  auto amax = [&](const u32x4 h) {
    const f16x8 hv = __builtin_bit_cast(f16x8, h);
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf((float)hv[e]));
  };
  for (int c = 64 * kH + lane; c < nch; c += 64) amax(ld16(rh, (c0 + c) * 16));
  // The row's entries in this part's columns.
  const int klo = plo * kBlk, khi = (plo + pnb) * kBlk;
  const int left0 = __popcll(__ballot(col0 < klo));   // of the first 64: left of the part's columns
  int left = left0, inn = __popcll(__ballot(col0 < khi)) - left0;
  for (int e = r0 + 64; e < r1; e += 64) {
    const int c = e + lane < r1 ? gp(a.O_col)[e + lane] : 0x7fffffff;
    const int l = __popcll(__ballot(c < klo));
    left += l;
    inn += __popcll(__ballot(c < khi)) - l;
  }
  if (lane == 0) {
    rfirst[wave] = r0 + left;
    rcnt[wave] = inn;
  }
  tab[tid ^ 0x100] = tload;
#pragma unroll
  for (int k = 0; k < kH; ++k) amax(hw[k]);
#pragma unroll
  for (int k = 0; k < kRing; ++k)
    if (k < n) issue(k, k);
  mx = fmaxf(mx, partner<1>(mx));
  mx = fmaxf(mx, partner<2>(mx));
  mx = fmaxf(mx, partner<4>(mx));
  mx = fmaxf(mx, partner<8>(mx));
  mx = fmaxf(mx, partner<16>(mx));
  mx = fmaxf(mx, partner<32>(mx));
  int ex = 0;
  if (mx > 1.0f) ex = (int)((__builtin_bit_cast(uint32_t, mx) >> 23) & 0xff) - 126;   // 2^ex >= mx
  const float out_scale = __builtin_ldexpf(1.0f, ex);
  const f16 down = (f16)__builtin_ldexpf(1.0f, -ex);
  const uint32_t down2 = __builtin_bit_cast(uint32_t, (h2){down, down});
  __syncthreads();

  // Stage the entries, row after row; entries past the stage stay in memory.
  // (Only LDS writes of registers for rows of up to 64 entries.)
  const int lq = (lane & 15) >> 1;
  int ec = 0, ee = 0, es_w = 0, total = 0;
#pragma unroll
  for (int r = 0; r < kTile; ++r) {
    const int c = rcnt[r];
    if (r == wave) es_w = total;
    if (r == lq) {
      ec = total;
      ee = total + c < L::kEnt ? total + c : L::kEnt;
    }
    total += c;
  }
  const int at = es_w + lane - left0;
  if (col0 >= klo && col0 < khi && at < L::kEnt) {
    ecol[at] = (uint16_t)col0;
    eov[at] = eo0;
  }
  for (int e = r0 + 64 + lane; e < r1; e += 64) {
    const int c = gp(a.O_col)[e];
    const int at2 = es_w + e - (r0 + left);
    if (c >= klo && c < khi && at2 < L::kEnt) {
      ecol[at2] = (uint16_t)c;
      eov[at2] = *gp((const u32x4*)a.O + e);
    }
  }
  __syncthreads();
  // The cursor of this lane's block row: its first staged entry at or past
  // the wave's first column, the entry's column and this lane's half of O.
  for (int hi = ee; ec < hi;) {
    const int mid = (ec + hi) >> 1;
    if (ecol[mid] < blo * kBlk) ec = mid + 1; else hi = mid;
  }
  int ncol;
  u32x2 nov;
  auto fetch = [&]() {
    const int e = ec < L::kEnt ? ec : 0;
    ncol = ec < ee ? (int)ecol[e] : 0x7fffffff;
    nov = *(const u32x2*)((const char*)&eov[e] + 8 * (lane & 1));
  };
  fetch();

  f32x4 acc[4][TT];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int j = 0; j < TT; ++j) acc[c][j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  const mdec::Half half(i);
  const char* __restrict__ tabB = (const char*)tab;
  const char* const slots = dyn + wave * (kRing * L::Slot);

  auto block = [&](int slot, int k) {
    const char* xs = slots + slot * L::Slot;
    const char* qs = xs + L::XB;
    const char* hb = qs + L::QB;
#pragma unroll
    for (int g2 = 0; g2 < kBlk / 32; ++g2) {
    const int ch = 4 * g2 + kg, c8 = (blo + k) * kBlk + 8 * ch;   // this lane's chunk and its first column
    const u32x4 q = *(const u32x4*)(qs + lq * L::RB + ((ch ^ L::swz(lq)) << 4));
    u32x4 hv = *(const u32x4*)(hb + 16 * ch);
    u32x4 bx[TT];
#pragma unroll
    for (int j = 0; j < TT; ++j) bx[j] = *(const u32x4*)(xs + (16 * j + i) * L::RB + ((ch ^ L::swz(i)) << 4));
    u32x2 lo[4], hi[4];
    half.lookup(q, tabB, lo, hi);
    if (HAS_S) {
      const f16x8 sf = *(const f16x8*)(hb + L::RB + 16 * ch);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const uint32_t sl = __builtin_bit_cast(uint32_t, (h2){sf[2 * w], sf[2 * w]});
        const uint32_t sh = __builtin_bit_cast(uint32_t, (h2){sf[2 * w + 1], sf[2 * w + 1]});
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          lo[w][p] = pk_mul(lo[w][p], sl);
          hi[w][p] = pk_mul(hi[w][p], sh);
        }
      }
    }
    while (ncol < c8 + 8) {
      if (ncol >= c8) {
        const int jc = ncol - c8;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          if (jc == 2 * w) lo[w] = nov;
          if (jc == 2 * w + 1) hi[w] = nov;
        }
      }
      ++ec;
      fetch();
    }
#pragma unroll
    for (int w = 0; w < 4; ++w) hv[w] = pk_mul(hv[w], down2);
#pragma unroll
    for (int j = 0; j < TT; ++j)
#pragma unroll
      for (int w = 0; w < 4; ++w) bx[j][w] = pk_mul(to_f16x2<XT>(bx[j][w]), hv[w]);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const f16x8 aw = __builtin_bit_cast(f16x8, mdec::Half::operand(lo, hi, c));
#pragma unroll
      for (int j = 0; j < TT; ++j)
        acc[c][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(aw, __builtin_bit_cast(f16x8, bx[j]), acc[c][j], 0, 0, 0);
    }
    }
  };
  int slot = 0;
  for (int k = 0; k < n; ++k) {
    // Block k has landed (the next kRing - 1 may be in flight).
    if (kRing == 3 && k + 2 < n) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * C) : "memory");
    } else if (k + 1 < n) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    block(slot, k);
    if (k + kRing < n) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slot's reads are done
      issue(slot, k + kRing);
    }
    slot = slot == kRing - 1 ? 0 : slot + 1;
  }

  // Entries past the stage (dense critical blocks only): the loop multiplied
  // table row 511 at their columns; add the difference.  Lane group kg holds
  // block rows 2kg and 2kg + 1 of a tile, feature 16·kg + 4v + c.
  if (total > L::kEnt) {
    const f16x4 t5 = tab[511 ^ 0x100];
#pragma unroll
    for (int b2 = 0; b2 < 2; ++b2) {
      const int rw = 2 * kg + b2;
      int st = 0;
      for (int r = 0; r < rw; ++r) st += rcnt[r];
      const int skip = st < L::kEnt ? L::kEnt - st : 0;   // staged entries of this row
#pragma unroll 1
      for (int e = rfirst[rw] + skip; e < rfirst[rw] + rcnt[rw]; ++e) {
        const int col = gp(a.O_col)[e];
        if (col < blo * kBlk || col >= (blo + n) * kBlk) continue;
        const f16x8 o = *gp((const f16x8*)a.O + e);
        const f16 h1 = (f16)(gp(a.h)[col] * down);
        const f16 s1 = HAS_S ? gp(a.S)[(size_t)((8 * m0) / a.qb) * N + col] : (f16)1.0f;
        float dv[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) dv[r] = (float)o[r] - (float)(f16)(t5[r & 3] * s1);
#pragma unroll
        for (int j = 0; j < TT; ++j) {
          const int tk = 16 * j + i;
          const float xf = tk < Bt ? (float)(f16)(to_f16<XT>(gp(a.x)[(size_t)(t0 + tk) * ldx + col]) * h1) : 0.0f;
#pragma unroll
          for (int r = 0; r < 8; ++r) acc[r & 3][j][2 * b2 + (r >> 2)] += dv[r] * xf;   // 8·b2 + r = 4v + c
        }
      }
    }
  }

  // The slots and entries are no longer read: the partial sums take their
  // place, red[wave][row of x][output], 32 rows at a time.  Output item it of
  // thread tid: row of x 32·it + tid/16, outputs 4(tid%16) ..
  constexpr int kIt = (TT + 1) / 2;
  const int r = (tid & 15) * 4, br = tid >> 4;
  f32x4 sum[kIt];
#pragma unroll
  for (int it = 0; it < kIt; ++it) {
    __syncthreads();
#pragma unroll
    for (int j = 2 * it; j < 2 * it + 2 && j < TT; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        *(f32x4*)&red[wave][16 * (j - 2 * it) + i][16 * kg + 4 * v] =
            (f32x4){acc[0][j][v] * out_scale, acc[1][j][v] * out_scale, acc[2][j][v] * out_scale, acc[3][j][v] * out_scale};
    __syncthreads();
    sum[it] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    if (32 * it + br < 16 * TT) {
#pragma unroll
      for (int w = 0; w < kS; ++w) sum[it] += *(const f32x4*)&red[w][br][r];
    }
  }
  const bool ok0 = br < Bt, ok1 = 32 + br < Bt;   // items 0 and 1

  // Split columns: publication and order as in decode_mfma.hip (device-scope
  // stores complete before the count, the last part adds all in part order
  // and resets the count).
  if (Pt > 1) {
    constexpr int kPart = 16 * TT * 64 * 4;   // bytes of a part's sums
    const int split = sp.tiles - sp.T1;
    const __amdgpu_buffer_rsrc_t rp =
        rsrc((const char*)sp.part + ((size_t)tg * split + (tile_g - sp.T1)) * Pt * kPart, Pt * kPart);
    auto at = [&](int q, int it) {
      return (it == 0 ? ok0 : ok1) ? q * kPart + it * 32 * 256 + (br * 64 + r) * 4 : kFar;
    };
#pragma unroll
    for (int it = 0; it < kIt; ++it)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, sum[it]), rp, at(part, it), 0, kSc1);
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
    __syncthreads();
    if (tid == 0) {
      int* c = sp.cnt + tg * sp.tiles + tile_g;
      const int old = __hip_atomic_fetch_add(c, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last_part = old == Pt - 1;
      if (old == Pt - 1) __hip_atomic_store(c, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!last_part) return;
    // Every part's sums at once (a part past Pt reads past the buffer), so
    // that the reads are one round trip.
    auto gather = [&](auto parts) {
      constexpr int kP = decltype(parts)::value;
      f32x4 v[kP][kIt];
#pragma unroll
      for (int q = 0; q < kP; ++q)
#pragma unroll
        for (int it = 0; it < kIt; ++it)
          v[q][it] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rp, at(q, it), 0, kSc1));
#pragma unroll
      for (int it = 0; it < kIt; ++it) {
        f32x4 u = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < kP; ++q) {
          if (q >= Pt) break;   // uniform
          u += q == part ? sum[it] : v[q][it];
        }
        sum[it] = u;
      }
    };
    if (Pt <= 4) gather(std::integral_constant<int, 4>{});
    else gather(std::integral_constant<int, kMaxParts>{});
  }
  const int orow = 8 * m0 + r;   // whole block rows: four outputs are all in range or none is
  if (orow >= 8 * M) return;
  const h2 g01 = *(const h2*)(a.g + orow), g23 = *(const h2*)(a.g + orow + 2);
  h2 b01 = {(f16)0.0f, (f16)0.0f}, b23 = b01;
  if (a.bias) {
    b01 = *(const h2*)(a.bias + orow);
    b23 = *(const h2*)(a.bias + orow + 2);
  }
#pragma unroll
  for (int it = 0; it < kIt; ++it) {
    if (!(it == 0 ? ok0 : ok1)) continue;
    const f32x4 v = sum[it];
    uint32_t* yp = (uint32_t*)(a.y + (size_t)(t0 + 32 * it + br) * a.ldy + orow);
    gp(yp)[0] = (uint32_t)Act<XT>::from_f32(v[0] * (float)g01[0] + (float)b01[0]) |
                ((uint32_t)Act<XT>::from_f32(v[1] * (float)g01[1] + (float)b01[1]) << 16);
    gp(yp)[1] = (uint32_t)Act<XT>::from_f32(v[2] * (float)g23[0] + (float)b23[0]) |
                ((uint32_t)Act<XT>::from_f32(v[3] * (float)g23[1] + (float)b23[1]) << 16);
  }
}

struct Plan {
  int T1, P;
  double cost;
};

template <int TT, bool HAS_S, typename XT>
int launch_t(const LinearArgs* l, int n, const Plan& pl, int TG, hipStream_t s, void* work, size_t off) {
  MultiArgs ma;
  ma.n = n;
  ma.act = nullptr;
  ma.start[0] = 0;
  for (int k = 0; k < kMaxLayers; ++k) {
    ma.l[k] = l[k < n ? k : 0];
    ma.start[k + 1] = ma.start[k] + (k < n ? (l[k].M + kTile - 1) / kTile : 0);
  }
  const int tiles = ma.start[n];
  Split sp;
  sp.units = pl.T1 + (tiles - pl.T1) * pl.P;
  sp.P = pl.P;
  sp.T1 = pl.T1;
  sp.TG = TG;
  sp.tiles = tiles;
  sp.cnt = (int*)work;
  sp.part = (float*)((char*)work + off);
  auto kern = k_decode_wide<TT, HAS_S, XT>;
  constexpr int dyn = Lay<TT>::Bytes;
  static bool attr = false;
  if (!attr) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, dyn) != hipSuccess) return -1;
    attr = true;
  }
  kern<<<(sp.units + 7) / 8 * 8 * TG, kNT, dyn, s>>>(ma, sp);
  return 0;
}

template <bool HAS_S, typename XT>
int launch_tt(const LinearArgs* l, int n, hipStream_t s, void* work, long long work_bytes) {
  // Whole groups of 16 rows, at most four per workgroup, spread evenly.
  const int t16 = (l[0].B + 15) / 16;
  const int TG = (t16 + 3) / 4, TT = (t16 + TG - 1) / TG < 2 ? 2 : (t16 + TG - 1) / TG;
  // The column split, by the least estimated time: rounds of the workgroups a
  // CU holds x (a start and end of F us, and the columns at C us per 1024 and
  // wave slot: measured one workgroup per CU, 16384 rows, 512 to 4096
  // columns), and ~2.5 us where parts meet in the workspace.  The sums go to
  // the workspace's prefill area if there is one, else after the counters.
  const size_t whole = (size_t)decode_mfma_work_bytes();
  const size_t off = work_bytes > (long long)whole + (64 << 10) ? whole : kSplitCounterBytes;
  const size_t room = work && (size_t)work_bytes > off ? (size_t)work_bytes - off : 0;
  const int cu = dec::cu_count(), nb = (l[0].N + 63) / 64;
  int tiles = 0;
  for (int k = 0; k < n; ++k) tiles += (l[k].M + kTile - 1) / kTile;
  Plan best = {0, 0, 0.0};
  const double fix = TT == 2 ? 6.0 : 8.0, per = TT == 2 ? 2.5 : TT == 3 ? 2.9 : 3.3;
  const size_t part_bytes = (size_t)16 * TT * 64 * 4;
  auto cols = [&](int P) { return (double)((nb + P - 1) / P) * per / 16.0; };
  auto consider = [&](int T1, int P) {
    const int split = tiles - T1;
    if (P > 1 && (tiles * TG > kSplitCounters || (size_t)split * TG * P * part_bytes > room || nb < kS * P)) return;
    const double t1 = T1 ? fix + cols(1) : 0.0;
    const long r2 = ((long)split * TG * P + cu - 1) / cu;
    const double t = t1 + r2 * (fix + cols(P)) + (P > 1 ? 2.5 : 0.0);
    if (best.P == 0 || t < best.cost) best = {T1, P, t};
  };
  for (int P = 1; P <= kMaxParts; ++P) consider(0, P);
  if (tiles * TG > cu)
    for (int P = 2; P <= kMaxParts; ++P) consider(cu / TG, P);
  if (TT == 2) return launch_t<2, HAS_S, XT>(l, n, best, TG, s, work, off);
  if (TT == 3) return launch_t<3, HAS_S, XT>(l, n, best, TG, s, work, off);
  return launch_t<4, HAS_S, XT>(l, n, best, TG, s, work, off);
}

}  // namespace dwide

// Returns 0 if launched, -1 outside the kernel's range.
int launch_decode_wide_multi(const LinearArgs* l, int n, hipStream_t s, void* work, long long work_bytes) {
  if (n < 1 || n > kMaxLayers) return -1;
  const LinearArgs& a = l[0];
  if (a.B < 1 || a.B > kWideMaxTokens || a.codes_f32 || (a.N & 7) != 0 || a.prep != 0) return -1;
  // y is written in pairs (4-byte stores), g and bias read in pairs.
  if ((a.ldy & 1) != 0) return -1;
  for (int i = 0; i < n; ++i) {
    const LinearArgs& b = l[i];
    if (b.N != a.N || b.B != a.B || b.x != a.x || b.ldx != a.ldx || b.codes != a.codes || b.codes_f32 || b.prep != 0 ||
        b.x_bf16 != a.x_bf16 || (b.S != nullptr) != (a.S != nullptr) || b.res || b.ldy != a.ldy ||
        (((uintptr_t)b.y | (uintptr_t)b.g | (uintptr_t)b.bias) & 3) != 0)
      return -1;
    if (b.S && (b.qb <= 0 || b.qb % 64 != 0)) return -1;   // one scale row per row tile
    if ((long)b.M * b.N * 2 >= (1L << 30)) return -1;       // 32-bit buffer offsets
  }
  if ((long)(a.B + 64) * a.ldx * 2 >= (1L << 30)) return -1;
  if (a.N > 65536) return -1;   // staged columns in 16 bits
  if (a.x_bf16) return a.S ? dwide::launch_tt<true, bf16>(l, n, s, work, work_bytes)
                           : dwide::launch_tt<false, bf16>(l, n, s, work, work_bytes);
  return a.S ? dwide::launch_tt<true, f16>(l, n, s, work, work_bytes)
             : dwide::launch_tt<false, f16>(l, n, s, work, work_bytes);
}

}  // namespace eptq
