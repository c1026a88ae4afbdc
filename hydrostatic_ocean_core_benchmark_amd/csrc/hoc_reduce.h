// NumPy-order float64 reductions over a PCG partition (see PcgArgs in
// hoc_kernels.h): per-part pairwise sums and the in-order total.
//
// Both are chains of latencies (load, a few adds, LDS, barrier), so they are
// cut to the fewest links: adds between lanes are DPP moves, the accumulators'
// sixteen LDS reads are issued together, the trees have one shape for every
// length (an absent leaf is -0.0, which adds as nothing), and each has one
// barrier. With the trailing chunk's tree walked from a plan in memory, LDS
// read by read and with a barrier per tree level, the A phase of 131 x 77 took
// 8.3 us and its update 5.8, of 128 x 128 6.5 and 4.4; so they are 5.8 and
// 3.9, 5.2 and 3.5.
#pragma once

#include "hoc_device.h"
#include "hoc_kernels.h"

namespace hoc {

__device__ __forceinline__ double shfl_xor_d(double v, int m) { return __shfl_xor(v, m, 8); }

struct Two {
  double a, b;
};

template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Pairwise sums over groups of 8 and of 16 neighbouring lanes, in every lane:
// lane ^ 1, lane ^ 2, then the mirrored lane of the 8 and of the 16, whose
// value is that of lane ^ 4 and lane ^ 8 once quads and eights agree. All
// lanes of the group must be active.
__device__ __forceinline__ double sum8(double v) {
  v = v + dpp_d<0xB1>(v);
  v = v + dpp_d<0x4E>(v);
  return v + dpp_d<0x141>(v);
}
__device__ __forceinline__ double sum16(double v) {
  v = sum8(v);
  return v + dpp_d<0x140>(v);
}

// The elements of one part: [base, base + nel). Full 8192-element chunks are
// cut into PCG_SUB aligned subtrees of 512 elements (four 128-element leaves).
// The trailing partial chunk is one part per slot of its halving tree filled
// up to a perfect one: a slot whose leaf lies higher up is empty (nel = 0).
struct PartRange {
  long long base;
  int nel;
};

__device__ __forceinline__ PartRange part_range(const PcgArgs& a, int part) {
  const int nfp = (int)a.nfull * PCG_SUB;
  if (part < nfp) return PartRange{(long long)part * PCG_PART, PCG_PART};
  // halve as the pairwise sum does (the left half a multiple of 8)
  int off = 0, len = a.tail;
  for (int bit = a.tail_slots >> 1; bit > 0; bit >>= 1) {
    const bool right = ((part - nfp) & bit) != 0;
    if (len > 128) {
      const int half = (len / 2) & ~7;
      off += right ? half : 0;
      len = right ? len - half : half;
    } else if (right) {
      len = 0;
    }
  }
  return PartRange{a.nfull * PW_CHUNK + off, len};
}

// Where element t of a part is staged in LDS: the leaves 8 values apart from
// a common bank.
__device__ __forceinline__ int stage_at(int t) { return t + (t >> 7) * 8; }

// Pairwise sum(s) in NumPy's order over values staged at lds[stage_at(0..nel)]
// (and lds[PCG_STAGE + ..] for the second sum): the first wave's lanes 0-31
// form the first sum, lanes 32-63 the second, eight lanes per leaf with
// NumPy's eight interleaved accumulators, then the leaves pairwise. Starts with
// a barrier (the staging must be done). The sums are in threads 0 and 32.
template <int NS>
__device__ __forceinline__ double part_reduce(const PartRange& pr, const double* lds) {
  const int tid = threadIdx.x;
  __syncthreads();
  if (tid >= 64) return 0.0;
  const int g = (tid >> 3) & 3, lane = tid & 7;
  const double* v = lds + (NS > 1 ? (tid >> 5) * PCG_STAGE : 0) + g * 136;
  double w[16];
#pragma unroll
  for (int t = 0; t < 16; ++t) w[t] = v[8 * t + lane];
  double s;
  if (pr.nel == PCG_PART) {
    s = w[0];
#pragma unroll
    for (int t = 1; t < 16; ++t) s = s + w[t];
    s = sum8(s);
  } else {
    const int len = min(max(pr.nel - 128 * g, 0), 128), fl = len & ~7;
    double rem[7];
#pragma unroll
    for (int t = 0; t < 7; ++t) rem[t] = v[fl + t];
    s = fl ? w[0] : len ? 0.0 : -0.0;
#pragma unroll
    for (int t = 1; t < 16; ++t) s = 8 * t < fl ? s + w[t] : s;
    s = sum8(s);
#pragma unroll
    for (int t = 0; t < 7; ++t) s = fl + t < len ? s + rem[t] : s;
  }
  s = s + dpp_d<0x140>(s);
  return s + __shfl_xor(s, 16, 64);
}

// This workgroup's part and the pairwise sum over it in NumPy's order (in
// thread 0). Each thread evaluates elements independently (`elem(e)` may store
// per-element results; it runs exactly once per index) and the values are
// staged in LDS for part_reduce; a thread's elements are evaluated before
// any is staged, so their loads are in flight together.
template <class F>
__device__ __forceinline__ double part_sum(const PcgArgs& a, int part, F elem,
                                           double* lds /* [PCG_STAGE] */) {
  const PartRange pr = part_range(a, part);
  double v[PCG_EPT];
#pragma unroll
  for (int k = 0; k < PCG_EPT; ++k) {
    const int t = threadIdx.x + k * PCG_WG;
    v[k] = t < pr.nel ? elem(pr.base + t) : 0.0;
  }
#pragma unroll
  for (int k = 0; k < PCG_EPT; ++k) lds[stage_at(threadIdx.x + k * PCG_WG)] = v[k];
  return part_reduce<1>(pr, lds);
}

// The same, one element after the other: half the registers, for the
// cooperative kernel, whose workgroups must all be resident.
template <class F>
__device__ __forceinline__ double part_sum_each(const PcgArgs& a, int part, F elem, double* lds) {
  const PartRange pr = part_range(a, part);
#pragma unroll 1
  for (int t = threadIdx.x; t < pr.nel; t += PCG_WG) lds[stage_at(t)] = elem(pr.base + t);
  return part_reduce<1>(pr, lds);
}

// In-order float64 sums of whole vectors from their per-part partials: sixteen
// lanes sum a full chunk's subtrees pairwise, the trailing chunk's slots are
// rows of sixteen of its tree, then the chunk sums are added sequentially.
// Every thread forms them identically; NV vectors (1 or 2) are summed in one
// pass. The first rows' loads are apart (totals_load), for a kernel to issue
// before its other loads. cs must not be in use (its last readers a barrier
// ago).
constexpr int PCG_CS = PCG_MAX_CHUNKS + 8;  // rows of one vector
constexpr int PCG_ROWS = PCG_WG / 16;       // rows of one pass, two in flight
template <int NV>
struct TotalsLoads {
  double v[2][NV];
};

// The trailing chunk's first row, behind fillers of -0.0, and all rows.
__device__ __forceinline__ int totals_tail_row(const PcgArgs& a) { return ((int)a.nfull + 7) & ~7; }
__device__ __forceinline__ int totals_rows(const PcgArgs& a) {
  return totals_tail_row(a) + (a.tail_slots + 15) / 16;
}

template <int NV>
__device__ __forceinline__ TotalsLoads<NV> totals_load(const PcgArgs& a,
                                                       const double* const* part, int c0 = 0) {
  const int nfull = (int)a.nfull, trow = totals_tail_row(a), rows = totals_rows(a);
  const int row = threadIdx.x >> 4, lane = threadIdx.x & 15;
  TotalsLoads<NV> L;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int c = c0 + k * PCG_ROWS + row;
    const int slot = c < trow ? c * 16 + lane : (nfull + c - trow) * 16 + lane;
    const bool on = c < rows && (c < trow ? c < nfull : slot < a.nparts);
#pragma unroll
    for (int q = 0; q < NV; ++q) L.v[k][q] = on ? part[q][slot] : -0.0;
  }
  return L;
}

template <int NV, int CS = PCG_CS>
__device__ __forceinline__ void totals_finish(const PcgArgs& a, const double* const* part,
                                              TotalsLoads<NV> L, double* cs /* [NV][CS] */,
                                              double* out) {
  const int trow = totals_tail_row(a), rows = totals_rows(a);
  const int row = threadIdx.x >> 4, lane = threadIdx.x & 15;
  for (int c0 = 0; c0 < rows; c0 += 2 * PCG_ROWS) {
    if (c0) L = totals_load<NV>(a, part, c0);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int c = c0 + k * PCG_ROWS + row;
      if (c0 + k * PCG_ROWS >= rows) break;
#pragma unroll
      for (int q = 0; q < NV; ++q) {
        const double s = sum16(L.v[k][q]);
        if (lane == 0 && c < rows) cs[q * CS + c] = s;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    const double* v = cs + q * CS;
    double s = 0.0;
    for (int c = 0; c < trow; c += 8) {
      double w[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) w[k] = v[c + k];
#pragma unroll
      for (int k = 0; k < 8; ++k) s = s + w[k];
    }
    if (a.tail) {
      double w[8];
      const int n = rows - trow;
#pragma unroll
      for (int k = 0; k < 8; ++k) w[k] = k < n ? v[trow + k] : -0.0;
      s = s + (((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7])));
    }
    out[q] = s;
  }
}

template <int NV, int CS = PCG_CS>
__device__ __forceinline__ void totals_from_parts(const PcgArgs& a, const double* const* part,
                                                  double* cs, double* out) {
  totals_finish<NV, CS>(a, part, totals_load<NV>(a, part), cs, out);
}

__device__ __forceinline__ double total_from_parts(const PcgArgs& a, const double* part,
                                                   double* cs) {
  const double* p[1] = {part};
  double out[1];
  totals_from_parts<1>(a, p, cs, out);
  return out[0];
}

}  // namespace hoc
