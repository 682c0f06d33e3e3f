// Bit-exact dequantization of an EPTQ layer to fp16 W (8M, N).
//
// Device counterpart of dequantize_layer (reference algorithms/eptq.py:406-471).
// Per element, in IEEE fp32 with round-to-nearest-even and no contraction:
//   v = table row (E8-D4: codes[t,i] | codes[t,j]; E8: points[u])
//   v = v * fp32(S_group[row / qb, n])            (if S_group)
//   v = fp32(O[rank])  for critical blocks          (not multiplied by S)
//   W = fp16((v * fp32(g[row])) * fp32(h[n]))
// The table must be the fp32 one the reference's loader produces
// (reconstruct.py:52-62), so the bits match eptq.reconstruct.
//
#include "common.h"
#include "kernels.h"

namespace eptq {

// First CSR slot in [lo, hi) whose column is >= n (columns ascend per row).
__device__ __forceinline__ int csr_lower_bound(const int32_t* __restrict__ col,
                                               int lo, int hi, int n) {
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (col[mid] < n) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// One wave per (Q-row, 512 columns): every lane takes 8 columns (one 16-byte
// index load, one 16-byte store in each of the 8 output rows), and the row's
// critical blocks are found by the wave together.  The row's CSR entries are
// in ascending column order, so the entry of a marker is the number of
// entries left of the segment plus the number of markers before it in the
// segment (ballots); its O vector comes from the lane that loaded it
// (bpermute).  Rows of up to 64 entries load columns and vectors at once with
// the indices, so a marker costs no memory round trip of its own; longer rows
// count their entries left of the segment first.  An entry whose column does
// not match (inconsistent CSR data) falls back to the search by column.
//
// Bound by the W writes (16 bytes out per 2-byte index).  Measured at 1% critical
// blocks, 11008x4096: 41.1 -> 19.5 us (4.6 TB/s of W; a device copy moves 5.1,
// a fill 6.9), 4096x4096: 17.3 -> 9.0 us, against one search by column per
// marker and lane (nearly every wave held one); S_group 14336x4096 at 0.2%:
// 89 -> 24 us (scale rows in 16-byte loads rather than one load per element).
// 2, 8 and 64 workgroups per CU are within 3% of 4; more waves per SIMD through
// fewer registers 20-100% slower; cached in place of streaming stores 18-36%
// slower, but a GEMM that reads W next finds part of it in the last-level
// cache: both passes of 13824x5120 at 2048 tokens 298 -> 280 us (keep).
constexpr int kSegCols = 512;
constexpr int kSegWaves = 8;   // waves per workgroup: one 8 KB table fill per 64 KB or more of W
constexpr int kSegPerCu = 4;   // workgroups per CU (2 resident at this register count, the rest follow)

template <int KIND, bool HAS_S>
__global__ __launch_bounds__(64 * kSegWaves) void k_dequant_seg(DequantArgs a, int segs, int tasks) {
  __shared__ f32x4 tab[KIND == KIND_E8D4 ? 512 : 1];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int N = a.N;
  if (KIND == KIND_E8D4) {
    if (a.table_f16) {   // uniform
      const f16x4 v = ((const f16x4*)a.table)[threadIdx.x];
      tab[threadIdx.x] = (f32x4){(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
    } else {
      tab[threadIdx.x] = ((const f32x4*)a.table)[threadIdx.x];
    }
    static_assert(64 * kSegWaves == 512, "one table row per thread");
    __syncthreads();
  }
  for (int t = (int)blockIdx.x * kSegWaves + wave; t < tasks; t += (int)gridDim.x * kSegWaves) {
    const int m = t / segs;
    const int s0 = (t - m * segs) * kSegCols;   // the segment's first column
    const int n0 = s0 + 8 * lane;
    const bool act = n0 < N;                    // N % 8 == 0: whole chunks
    const int r0 = a.O ? a.O_row_ptr[m] : 0, r1 = a.O ? a.O_row_ptr[m + 1] : 0;
    u16x8 qv = {};
    f16x8 hv = {}, sv = {};
    if (act) {
      qv = *(const u16x8*)(a.Q + (size_t)m * N + n0);
      hv = *(const f16x8*)(a.h + n0);
      if (HAS_S) sv = *(const f16x8*)(a.S + (size_t)(8 * m / a.qb) * N + n0);
    }
    // The row's entries, one per lane: all of them here, or (more than 64)
    // those from the segment's first one on, below.
    int ecol = 0x7fffffff;
    u32x4 eo = {};
    auto load_entries = [&](int first) {
      if (first + lane < r1) {
        ecol = a.O_col[first + lane];
        eo = *(const u32x4*)(a.O + (size_t)(first + lane) * 8);
      }
    };
    const bool whole = r1 - r0 <= 64;
    if (whole) load_entries(r0);
    float gk[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) gk[k] = (float)a.g[8 * m + k];

    uint64_t mk[8], any = 0;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      mk[c] = __ballot(qv[c] == 0x7fffu);
      any |= mk[c];
    }
    int src = 0;   // the lane that holds the entry of this lane's next marker
    if (any) {
      if (whole) {
        src = __popcll(__ballot(ecol < s0));
      } else {
        int first = r0;
        for (int e = r0; e < r1; e += 64) {
          const int left = __popcll(__ballot(e + lane < r1 && a.O_col[e + lane < r1 ? e + lane : r1 - 1] < s0));
          first += left;
          if (left < 64) break;
        }
        load_entries(first);
      }
#pragma unroll
      for (int c = 0; c < 8; ++c)
        src = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mk[c] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mk[c], src));
    }
    // out[k] word c/2: the fp16 pair (column c, column c + 1) of output row
    // 8m + k, converted two at a time (one v_cvt_pk_f16_f32).
    u32x4 out[8];
#pragma unroll
    for (int c = 0; c < 8; c += 2) {
      float v[2][8];
#pragma unroll
      for (int cc = 0; cc < 2; ++cc) {
        unsigned u = (unsigned)qv[c + cc] ^ 0x8000u;   // index + 32768; 65535 marks a critical block
        f32x4 lo, hi;
        if (KIND == KIND_E8D4) {
          lo = tab[u >> 7];
          hi = tab[((u >> 14) << 7) | (u & 127u)];
        } else {
          u = u == 65535u ? 0u : u;   // past the table
          if (a.table_f16) {          // uniform
            const f16x8 v = ((const f16x8*)a.table)[u];
            lo = (f32x4){(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
            hi = (f32x4){(float)v[4], (float)v[5], (float)v[6], (float)v[7]};
          } else {
            const f32x4* p = (const f32x4*)a.table + (size_t)u * 2;
            lo = p[0];
            hi = p[1];
          }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          v[cc][k] = lo[k];
          v[cc][k + 4] = hi[k];
        }
        if (HAS_S) {
          const float s = (float)sv[c + cc];
#pragma unroll
          for (int k = 0; k < 8; ++k) v[cc][k] *= s;
        }
        if (mk[c + cc]) {   // uniform
          const bool mine = qv[c + cc] == 0x7fffu;
          const int n = n0 + c + cc;
          u32x4 o;
#pragma unroll
          for (int d = 0; d < 4; ++d) o[d] = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * src, (int)eo[d]);
          const int oc = __builtin_amdgcn_ds_bpermute(4 * src, ecol);
          const bool found = src < 64 && oc == n;
          if (mine) {
            if (!found) {   // inconsistent data, or over 64 markers in the segment
              const int i = csr_lower_bound(a.O_col, r0, r1, n);
              const bool hit = i < r1 && a.O_col[i] == n;
              o = hit ? *(const u32x4*)(a.O + (size_t)i * 8) : u32x4{};
            }
            const f16x8 of = __builtin_bit_cast(f16x8, o);
#pragma unroll
            for (int k = 0; k < 8; ++k) v[cc][k] = (float)of[k];
            ++src;
          }
        }
      }
      const float h0 = (float)hv[c], h1 = (float)hv[c + 1];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        float w0 = (v[0][k] * gk[k]) * h0;
        float w1 = (v[1][k] * gk[k]) * h1;
        // The reference rounds twice: to fp32 at the multiply, then to fp16.
        // Materialize the fp32 products so the compiler cannot fold multiply
        // and conversion into one single-rounding mix instruction.
        asm volatile("" : "+v"(w0), "+v"(w1));
        out[k][c >> 1] = __builtin_bit_cast(uint32_t, (f16x2){(f16)w0, (f16)w1});
      }
    }
    if (act) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        u32x4* dst = (u32x4*)(a.W + (size_t)(8 * m + k) * N + n0);
        if (a.keep) *dst = out[k];                       // uniform
        else __builtin_nontemporal_store(out[k], dst);   // not re-read here
      }
    }
  }
}

// Element by element, for column counts or pointers that rule the 16-byte
// accesses out: a thread takes (Q-row, 8 columns) items with a grid stride.
constexpr int kDqPerCu = 16;  // resident workgroups per CU

template <int KIND, bool HAS_S>
__global__ __launch_bounds__(256) void k_dequant(DequantArgs a, int chunks_per_row) {
  __shared__ f32x4 tab[KIND == KIND_E8D4 ? 512 : 1];
  auto row4 = [&](size_t r) {   // four table values
    if (!a.table_f16) return ((const f32x4*)a.table)[r];
    const f16x4 v = ((const f16x4*)a.table)[r];
    return (f32x4){(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
  };
  if (KIND == KIND_E8D4) {
    for (int i = threadIdx.x; i < 512; i += 256) tab[i] = row4(i);
    __syncthreads();
  }
  const int M = a.M, N = a.N;
  const int64_t items = (int64_t)M * chunks_per_row;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t it = (int64_t)blockIdx.x * 256 + threadIdx.x; it < items; it += stride) {
    const int m = (int)(it / chunks_per_row);
    const int n0 = (int)(it - (int64_t)m * chunks_per_row) * 8;
    const int r0 = a.O_row_ptr[m], r1 = a.O_row_ptr[m + 1];
    for (int n = n0; n < N && n < n0 + 8; ++n) {
      const unsigned u = (unsigned)((int)a.Q[(size_t)m * N + n] + 32768);
      float v[8];
      if (u == 65535u) {
        const int i = csr_lower_bound(a.O_col, r0, r1, n);
        const bool hit = (i < r1) && (a.O_col[i] == n);
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = hit ? (float)a.O[(size_t)i * 8 + k] : 0.0f;
      } else {
        f32x4 lo, hi;
        if (KIND == KIND_E8D4) {
          lo = tab[u >> 7];
          hi = tab[((u >> 14) << 7) | (u & 127u)];
        } else {
          lo = row4(2 * (size_t)u);
          hi = row4(2 * (size_t)u + 1);
        }
        const float s = HAS_S ? (float)a.S[(size_t)(8 * m / a.qb) * N + n] : 1.0f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          v[k] = HAS_S ? lo[k] * s : lo[k];
          v[k + 4] = HAS_S ? hi[k] * s : hi[k];
        }
      }
      const float hn = (float)a.h[n];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        float w = (v[k] * (float)a.g[8 * m + k]) * hn;
        asm volatile("" : "+v"(w));   // two roundings, as above
        a.W[(size_t)(8 * m + k) * N + n] = (f16)w;
      }
    }
  }
}

template <int KIND>
int launch_dequant(const DequantArgs& a, hipStream_t s) {
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  // 16-byte accesses: whole 8-column chunks, every operand they touch aligned.
  const bool vec = a.N % 8 == 0 &&
                   ((((uintptr_t)a.Q | (uintptr_t)a.h | (uintptr_t)a.W | (uintptr_t)a.S | (uintptr_t)a.O) & 15u) == 0);
  const int segs = (a.N + kSegCols - 1) / kSegCols;
  const int64_t tasks = (int64_t)a.M * segs;
  if (vec && tasks <= 0x3fffffff) {
    int64_t blocks = (tasks + kSegWaves - 1) / kSegWaves;
    if (blocks > (int64_t)cus * kSegPerCu) blocks = (int64_t)cus * kSegPerCu;
    if (a.S) k_dequant_seg<KIND, true><<<(unsigned)blocks, 64 * kSegWaves, 0, s>>>(a, segs, (int)tasks);
    else k_dequant_seg<KIND, false><<<(unsigned)blocks, 64 * kSegWaves, 0, s>>>(a, segs, (int)tasks);
    return 0;
  }
  const int chunks = (a.N + 7) / 8;
  int64_t blocks = ((int64_t)a.M * chunks + 255) / 256;
  if (blocks > (int64_t)cus * kDqPerCu) blocks = (int64_t)cus * kDqPerCu;
  if (blocks < 1) return 0;
  if (a.S) k_dequant<KIND, true><<<(unsigned)blocks, 256, 0, s>>>(a, chunks);
  else k_dequant<KIND, false><<<(unsigned)blocks, 256, 0, s>>>(a, chunks);
  return 0;
}

template int launch_dequant<KIND_E8D4>(const DequantArgs&, hipStream_t);
template int launch_dequant<KIND_E8>(const DequantArgs&, hipStream_t);

}  // namespace eptq
