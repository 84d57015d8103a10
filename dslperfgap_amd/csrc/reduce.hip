// Mean, max (value + index) and argmax over one axis, for gfx950.
//
// The tensor is viewed as contiguous [outer, n, inner] and reduced over n.
//   inner == 1 (last axis): `tpr` lanes own one row and stream it with 16-byte
//   loads (nothing per element is written, so the row is never held in
//   registers and any n works), then all-reduce across the group.
//   inner > 1: column tiles (col_lane): each lane owns the columns of one
//   16-byte vector and takes every 2^ty_log2-th row, the lines of lanes are
//   combined through LDS; few columns split the axis over workgroups; short
//   axes of small launches or narrow slabs run one lane per column.
// Each input element is read once; one value (and/or index) per output is
// written.
//
// Semantics (torch): mean accumulates in fp32 and divides by n
// (ViperBench/mean_reduction/pytorch_impl.py:4-8); max returns (values, int64
// indices) (ViperBench/max_reduction/pytorch_impl.py:4-11); argmax returns
// int64 indices (ViperBench/argmax/pytorch_impl.py:4-8).  NaN counts as the
// largest value and ties resolve to the smallest index, so the first maximal
// (or first NaN) position is returned.
#include <limits.h>

#include "vbh_device.h"
#include "vbh_launch.h"

namespace vbh {

namespace {

constexpr float kNegInf = -__builtin_huge_valf();

// true when (av, ai) should win over (bv, bi): a total order, so every lane of
// a butterfly picks the same pair.
__device__ __forceinline__ bool better(float av, int ai, float bv, int bi) {
  const bool an = av != av, bn = bv != bv;
  if (an || bn) return an && (!bn || ai < bi);
  return av > bv || (av == bv && ai < bi);
}

struct ValIdx {
  float v;
  int i;
};

__device__ __forceinline__ ValIdx pick(ValIdx a, ValIdx b) {
  return better(a.v, a.i, b.v, b.i) ? a : b;
}

template <int Ctrl>
__device__ __forceinline__ ValIdx dpp_vi(ValIdx a) {
  return ValIdx{dpp<Ctrl>(a.v),
                __builtin_amdgcn_update_dpp(0, a.i, Ctrl, 0xF, 0xF, false)};
}

__device__ __forceinline__ int swap16_partner_i(int v) {
  auto p = __builtin_amdgcn_permlane16_swap(static_cast<unsigned>(v), static_cast<unsigned>(v),
                                            false, false);
  return static_cast<int>((threadIdx.x & 16) ? p[0] : p[1]);
}
__device__ __forceinline__ int swap32_partner_i(int v) {
  auto p = __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(v), static_cast<unsigned>(v),
                                            false, false);
  return static_cast<int>((threadIdx.x & 32) ? p[0] : p[1]);
}

// All-reduce of (value, index) pairs over the tpr lanes of one row (see
// group_allreduce for the lane layout and the LDS contract; `lds` holds
// 2 * kMaxWaves words).
__device__ __forceinline__ ValIdx group_allreduce_vi(ValIdx a, int tpr, float* lds) {
  const int width = tpr < kWave ? tpr : kWave;
  if (width >= 2) a = pick(a, dpp_vi<0xB1>(a));
  if (width >= 4) a = pick(a, dpp_vi<0x4E>(a));
  if (width >= 8) a = pick(a, dpp_vi<0x141>(a));
  if (width >= 16) a = pick(a, dpp_vi<0x140>(a));
  if (width >= 32) a = pick(a, ValIdx{swap16_partner(a.v), swap16_partner_i(a.i)});
  if (width >= 64) a = pick(a, ValIdx{swap32_partner(a.v), swap32_partner_i(a.i)});
  if (tpr <= kWave) return a;
  const int wave = threadIdx.x / kWave;
  const int nwaves = tpr / kWave;
  const int first = (wave / nwaves) * nwaves;
  int* ldsi = reinterpret_cast<int*>(lds + kMaxWaves);
  if ((threadIdx.x & (kWave - 1)) == 0) {
    lds[wave] = a.v;
    ldsi[wave] = a.i;
  }
  __syncthreads();
  ValIdx r{lds[first], ldsi[first]};
  for (int w = first + 1; w < first + nwaves; ++w) r = pick(r, ValIdx{lds[w], ldsi[w]});
  return r;
}

// IEEE maximum of a 16-byte vector's values: NaN if one of them is NaN
// (fp16 pairs go to v_pk_maximum3_f16, fp32 values to v_maximum3_f32).
template <typename T, int V>
__device__ __forceinline__ float vec_max_nan(const typename Raw<T, V>::type& r) {
  float m = raw_at<T, V>(r, 0);
#pragma unroll
  for (int k = 1; k < V; ++k) m = max_nan(m, raw_at<T, V>(r, k));
  return m;
}

// The first element of `r` equal to `m` (the vector's maximum, so one
// exists), or its first NaN when `m` is NaN: (its value, its position in `r`).
// A NaN comes back as the canonical quiet NaN.
template <typename T, int V>
__device__ __forceinline__ ValIdx first_max_at(const typename Raw<T, V>::type& r, float m) {
  const bool nan = m != m;
  ValIdx f{m, V - 1};
#pragma unroll
  for (int k = V - 1; k >= 0; --k) {
    const float v = raw_at<T, V>(r, k);
    if (nan ? v != v : v == m) f = ValIdx{v, k};
  }
  if (nan) f.v = __builtin_nanf("");
  return f;
}

// An element as a (value, position) candidate, a NaN as the canonical one.
__device__ __forceinline__ ValIdx candidate(float v, int i) {
  return ValIdx{v != v ? __builtin_nanf("") : v, i};
}

template <typename T, int V, int OP>
__device__ __forceinline__ void write_result(void* vals, int64_t* idx, int64_t o, float sum_or_v,
                                             int i, int n, const Span& sv, const Span& si) {
  if constexpr (OP == 0) {
    const float m = sum_or_v / static_cast<float>(n);
    store_from_f32<T, 1>(static_cast<T*>(vals) + o, &m, sv);
  } else {
    if constexpr (OP == 1) store_from_f32<T, 1>(static_cast<T*>(vals) + o, &sum_or_v, sv);
    if (VBH_IN_SPAN(si, idx + o, sizeof(int64_t))) idx[o] = i;
  }
}

// OP: 0 = mean (To = output type), 1 = max values + indices, 2 = argmax.
// MIS: rows not a multiple of V long start at varying offsets within a
// 16-byte vector; each row is read as a scalar head up to the first 16-byte
// boundary (lanes g < head, element g), whole aligned vectors, and a scalar
// tail (lanes g < tail); the launcher makes tpr >= V.  A lane visits its head
// element first and its tail element last, so its positions still increase.
template <typename Ti, typename To, int V, int OP, bool MIS>
__global__ __launch_bounds__(kMaxBlock) void reduce_rows(const Ti* __restrict__ x,
                                                         void* __restrict__ vals,
                                                         int64_t* __restrict__ idx,
                                                         int64_t rows, int n, int tpr) {
  __shared__ float lds[2 * kMaxWaves];
  const GroupShape gs = group_shape(tpr);
  const int g = gs.g;
  int64_t row = static_cast<int64_t>(blockIdx.x) * gs.per_block + gs.sub;
  const bool live = row < rows;
  if (!live) row = rows - 1;
  const Span sx = VBH_SPAN(x, rows * n);
  const Span sv = VBH_SPAN(static_cast<To*>(vals), rows), si = VBH_SPAN(idx, rows);
  const int64_t start = row * n;
  int head = 0, nvec = n / V, tail = 0;
  if constexpr (MIS) {
    head = static_cast<int>((V - start % V) % V);
    if (head > n) head = n;
    nvec = (n - head) / V;
    tail = n - head - nvec * V;
  }
  const Ti* xr = x + start + head;  // 16-byte aligned body; element j * V + k is head + j * V + k
  const bool hv = MIS && g < head, tv = MIS && g < tail;
  const int tail0 = head + nvec * V;  // row index of the first tail element
  typedef typename Raw<Ti, V>::type RT;
  // Each lane loads kChunk vectors (kChunk * tpr apart... j, j + tpr, ...) before
  // processing any of them, so a chunk's loads are in flight together whatever
  // the data-dependent branches below do.
  constexpr int kChunk = 4;
  // (unsigned vector numbers: in a row of almost 2^31 vectors of one element the
  // last chunk passes 2^31)
  const uint32_t nv = nvec;
  if constexpr (OP == 0) {
    float acc[V];
#pragma unroll
    for (int k = 0; k < V; ++k) acc[k] = 0.f;
    for (uint32_t base = g; base < nv; base += kChunk * tpr) {
      RT r[kChunk];
#pragma unroll
      for (int c = 0; c < kChunk; ++c) {
        const uint32_t j = base + c * tpr;
        r[c] = j < nv ? load_raw<Ti, V, true>(xr + static_cast<int64_t>(j) * V, sx) : RT{};
      }
#pragma unroll
      for (int c = 0; c < kChunk; ++c)
#pragma unroll
        for (int k = 0; k < V; ++k) acc[k] += raw_at<Ti, V>(r[c], k);  // padding is zero
    }
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < V; ++k) s += acc[k];
    if (hv) {
      float v;
      load_f32<Ti, 1>(x + start + g, &v, sx);
      s += v;
    }
    if (tv) {
      float v;
      load_f32<Ti, 1>(x + start + tail0 + g, &v, sx);
      s += v;
    }
    s = group_allreduce<Sum>(s, tpr, lds);
    if (live && g == 0) write_result<To, V, OP>(vals, idx, row, s, 0, n, sv, si);
  } else {
    ValIdx best;
    if (nvec >= kChunk * tpr) {  // uniform: every lane holds a chunk of vectors or more
      // The lane's vectors are visited in increasing position order.  Per vector
      // only its IEEE maximum (NaN if it holds one) is formed and compared with
      // the lane's best; the winning vector is kept raw, and the position of its
      // first maximal (or first NaN) element is looked up once, after the loop.
      // A later vector wins only with a strictly larger maximum, or with the
      // first NaN, so the lane's result is its first maximal position.
      float bv = kNegInf;  // best vector's maximum
      int bj = -1;         // its vector index (-1: none yet)
      RT braw = RT{};
      for (uint32_t base = g; base < nv; base += kChunk * tpr) {
        RT r[kChunk];
#pragma unroll
        for (int c = 0; c < kChunk; ++c) {
          const uint32_t j = base + c * tpr;
          r[c] = j < nv ? load_raw<Ti, V, true>(xr + static_cast<int64_t>(j) * V, sx) : RT{};
        }
#pragma unroll
        for (int c = 0; c < kChunk; ++c) {
          const uint32_t j = base + c * tpr;
          if (j >= nv) break;  // the lane's later vectors are past the row too
          const float m = vec_max_nan<Ti, V>(r[c]);
          const bool win = bj < 0 || m > bv || (m != m && bv == bv);
          bv = win ? m : bv;
          bj = win ? static_cast<int>(j) : bj;
          braw = win ? r[c] : braw;
        }
      }
      best = ValIdx{kNegInf, n};  // an empty lane loses to any element
      if (bj >= 0) {
        const ValIdx f = first_max_at<Ti, V>(braw, bv);
        best = ValIdx{f.v, head + bj * V + f.i};
      }
      // the head element precedes every body position and the tail element
      // follows them; pick() orders by value (NaN largest), then position
      if (hv) {
        float v;
        load_f32<Ti, 1>(x + start + g, &v, sx);
        best = pick(candidate(v, g), best);
      }
      if (tv) {
        float v;
        load_f32<Ti, 1>(x + start + tail0 + g, &v, sx);
        best = pick(best, candidate(v, tail0 + g));
      }
    } else {
      // Short rows (fewer than kChunk vectors per lane), visited in
      // increasing position order: head element, body vectors, tail element.
      // Per vector an fmax tree and a NaN test; the index search runs where
      // the vector beats the lane's best (a later value only wins when it is
      // strictly larger, or the first NaN).  With one or two vectors per lane
      // this is 3-8% faster than the search after the loop (fp16, 64, 100 and
      // 255 columns).
      best = ValIdx{kNegInf, n};  // an empty lane loses to any element
      bool done = false;        // a NaN was found: nothing later can win
      if (hv) {
        float v;
        load_f32<Ti, 1>(x + start + g, &v, sx);
        if (v != v) {
          best = ValIdx{__builtin_nanf(""), g};
          done = true;
        } else {
          best = ValIdx{v, g};
        }
      }
      for (uint32_t base = g; base < nv; base += kChunk * tpr) {
        RT r[kChunk];
#pragma unroll
        for (int c = 0; c < kChunk; ++c) {
          const uint32_t j = base + c * tpr;
          r[c] = j < nv ? load_raw<Ti, V, true>(xr + static_cast<int64_t>(j) * V, sx) : RT{};
        }
#pragma unroll
        for (int c = 0; c < kChunk; ++c) {
          const uint32_t j = base + c * tpr;
          if (done || j >= nv) continue;
          float v[V];
#pragma unroll
          for (int k = 0; k < V; ++k) v[k] = raw_at<Ti, V>(r[c], k);
          float m = v[0];
          bool nan = v[0] != v[0];
#pragma unroll
          for (int k = 1; k < V; ++k) {
            m = fmaxf(m, v[k]);
            nan |= v[k] != v[k];
          }
          if (nan) {  // first NaN of the vector (unrolled selects, no indexed registers)
            int kk = V - 1;
#pragma unroll
            for (int k = V - 1; k >= 0; --k)
              if (v[k] != v[k]) kk = k;
            best = ValIdx{__builtin_nanf(""), head + static_cast<int>(j) * V + kk};
            done = true;
          } else if (m > best.v || best.i == n) {  // first position of the vector max
            int kk = V - 1;
#pragma unroll
            for (int k = V - 1; k >= 0; --k)
              if (v[k] == m) kk = k;
            best = ValIdx{m, head + static_cast<int>(j) * V + kk};
          }
        }
      }
      if (tv && !done) {
        float v;
        load_f32<Ti, 1>(x + start + tail0 + g, &v, sx);
        if (v != v) best = ValIdx{__builtin_nanf(""), tail0 + g};
        else if (v > best.v || best.i == n) best = ValIdx{v, tail0 + g};
      }
    }
    best = group_allreduce_vi(best, tpr, lds);
    if (live && g == 0) write_result<To, V, OP>(vals, idx, row, best.v, best.i, n, sv, si);
  }
}

// Second stage of a row reduction split into `segs` segments of `segn`
// elements (max / argmax): one lane per row picks the winner of the segments'
// (value, index) results, which the first stage wrote as values of type T and
// int64 segment-local indices, under the same order as the row kernel (NaN
// largest, then the smaller global index).
template <typename T, int OP>
__global__ __launch_bounds__(256) void reduce_combine_vi(const T* __restrict__ pvals,
                                                         const int64_t* __restrict__ pidx,
                                                         void* __restrict__ vals,
                                                         int64_t* __restrict__ idx, int64_t rows,
                                                         int segs, int segn) {
  const int64_t row = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (row >= rows) return;
  const int64_t base = row * segs;
  const Span spv = VBH_SPAN(pvals, rows * segs), spi = VBH_SPAN(pidx, rows * segs);
  const Span sv = VBH_SPAN(static_cast<T*>(vals), rows), si = VBH_SPAN(idx, rows);
  ValIdx best{VBH_IN_SPAN(spv, pvals + base, sizeof(T)) ? static_cast<float>(pvals[base]) : 0.f,
              VBH_IN_SPAN(spi, pidx + base, sizeof(int64_t)) ? static_cast<int>(pidx[base]) : 0};
  for (int s = 1; s < segs; ++s) {
    const ValIdx c{
        VBH_IN_SPAN(spv, pvals + base + s, sizeof(T)) ? static_cast<float>(pvals[base + s]) : 0.f,
        s * segn + (VBH_IN_SPAN(spi, pidx + base + s, sizeof(int64_t))
                        ? static_cast<int>(pidx[base + s])
                        : 0)};
    best = pick(best, c);
  }
  if constexpr (OP == 1) store_from_f32<T, 1>(static_cast<T*>(vals) + row, &best.v, sv);
  if (VBH_IN_SPAN(si, idx + row, sizeof(int64_t))) idx[row] = best.i;
}

// Middle axis: column tiles (col_lane in vbh_device.h) of kColBlock lanes.
// PART (first stage of a split axis, grid.y segments of seg_n rows): each
// column's fp32 sum or value goes to pv[seg * columns + column] and its row to
// pi; else the result to vals / idx.
//
// Bound by memory: every element is read once, eight rows (128 bytes of loads)
// per lane in flight.  The kernel it replaced ran one lane per column with one
// element in flight and left most CUs idle.  MI355X, time per call before ->
// after (the bytes at the copy's rate): max fp16 64 x 512 x 768 149 -> 12.1 us
// (7.0), mean fp32 512 x 32 x 4096 77 -> 44 (38), max fp16 20 x 200 x 20000 111
// -> 36 (23), mean fp32 8192 x 64 x 49 34 -> 16.8 (14), max bf16 4096 x 2 x 4096
// 78 -> 38 (32).  Max and argmax stay up to 2 us behind the mean: five VALU
// instructions per element (convert, two compares, two selects).  Results go
// through LDS to the lanes that write them, so that stores of consecutive
// columns coalesce (straight from the lanes, the int64 indices of one lane are
// 64 bytes apart: max fp32 3375 x 3 x 512 12.9 against 8.7 us).
template <typename Ti, typename To, int V, int OP, bool PART, bool NT>
__global__ __launch_bounds__(kColBlock) void reduce_cols(
    const Ti* __restrict__ x, void* __restrict__ vals, int64_t* __restrict__ idx,
    float* __restrict__ pv, int* __restrict__ pi, int64_t outer, int n, int64_t inner, int cx,
    int ty_log2, uint32_t tiles, int seg_n) {
  typedef typename Raw<Ti, V>::type RT;
  constexpr int U = 8;  // rows in flight per lane
  constexpr int B = kColBlock;
  // a workgroup's columns side by side, line after line
  __shared__ __align__(16) float lds_v[V * B];
  __shared__ __align__(16) int lds_i[OP == 0 ? 4 : V * B];
  // per vector of the workgroup: its first output times 8, plus how many of its
  // columns the vector before it writes
  __shared__ int64_t lds_out[B];
  const ColLane L = col_lane<V>(outer, inner, cx, ty_log2, tiles);
  const int64_t cols = outer * inner;
  const Span sx = VBH_SPAN(x, outer * n * inner);
  const int seg = static_cast<int>(blockIdx.y);
  const int r0 = PART ? seg * seg_n : 0;
  const int len = PART ? min(n - r0, seg_n) : n;  // rows of this segment
  const int rows = L.live && L.ty < len ? ((len - L.ty - 1) >> ty_log2) + 1 : 0;  // the lane's
  const int64_t step = inner << ty_log2;
  const Ti* p = x + (L.o * n + r0 + L.ty) * inner + L.col;

  float a[V];  // the lane's sums, or its best values
  int at[OP == 0 ? 1 : V];
#pragma unroll
  for (int k = 0; k < V; ++k) a[k] = OP == 0 ? 0.f : kNegInf;
  if constexpr (OP != 0) {
    // a lane whose values are all -inf has its first row, one without rows none
#pragma unroll
    for (int k = 0; k < V; ++k) at[k] = rows > 0 ? r0 + L.ty : INT_MAX;
  }
  auto take = [&](const RT& v, int r) {
#pragma unroll
    for (int k = 0; k < V; ++k) {
      const float f = raw_at<Ti, V>(v, k);
      if constexpr (OP == 0) {
        a[k] += f;
      } else {
        // larger, or the column's first NaN
        const bool win = !(f <= a[k]) && a[k] == a[k];
        a[k] = win ? f : a[k];
        at[k] = win ? r : at[k];
      }
    }
  };
  int i = 0;
  for (; rows - i >= U; i += U, p += U * step) {
    RT v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = load_any<Ti, V, NT>(p + u * step, sx);
#pragma unroll
    for (int u = 0; u < U; ++u) take(v[u], r0 + L.ty + ((i + u) << ty_log2));
  }
  if (i < rows) {
    RT v[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i + u < rows) v[u] = load_any<Ti, V, NT>(p + u * step, sx);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i + u < rows) take(v[u], r0 + L.ty + ((i + u) << ty_log2));
  }
  // Through LDS, so that consecutive lanes write consecutive columns: each of
  // the workgroup's W columns is combined by `parts` lanes over its lines,
  // then by one over their results.
  const int W = L.per_block * cx * V;
  const int TY = 1 << ty_log2;
  const int t = static_cast<int>(threadIdx.x);
  if (L.sub < L.per_block) {
    const int vec = L.sub * cx + L.c;
    const int j = L.ty * W + vec * V;
#pragma unroll
    for (int k = 0; k < V; ++k) {
      lds_v[j + k] = a[k];
      if constexpr (OP != 0) lds_i[j + k] = at[k];
    }
    if (L.ty == 0) lds_out[vec] = L.live ? (L.o * inner + L.col) * 8 + L.shared : -1;
  }
  __syncthreads();
  auto gather = [&](int j, int stride, int count) {  // over lds[j], lds[j + stride], ...
    ValIdx r{lds_v[j], OP == 0 ? 0 : lds_i[OP == 0 ? 0 : j]};
    for (int s = 1; s < count; ++s) {
      j += stride;
      if constexpr (OP == 0) r.v += lds_v[j];
      else r = pick(r, ValIdx{lds_v[j], lds_i[j]});
    }
    return r;
  };
  int lines = TY;
  if (TY > 2 && W * 2 <= B) {
    int parts = TY >> 1;  // at least two lines each
    while (parts * W > B) parts >>= 1;
    const int part = t / W, j = t - part * W;
    ValIdx r{0.f, 0};
    const int per = TY / parts;  // powers of two
    if (part < parts) r = gather(part * per * W + j, W, per);
    __syncthreads();
    if (part < parts) {
      lds_v[part * W + j] = r.v;
      if constexpr (OP != 0) lds_i[part * W + j] = r.i;
    }
    __syncthreads();
    lines = parts;
  }
  const Span sv = VBH_SPAN(static_cast<To*>(vals), PART ? 0 : cols),
             si = VBH_SPAN(idx, PART ? 0 : cols);
  const Span spv = VBH_SPAN(pv, PART ? cols * gridDim.y : 0),
             spi = VBH_SPAN(pi, PART ? cols * gridDim.y : 0);
  for (int j = t; j < W; j += B) {
    const int64_t base = lds_out[j / V];
    const int k = j & (V - 1);
    if (base < 0 || k < static_cast<int>(base & 7)) continue;
    const int64_t out = (base >> 3) + k;
    const ValIdx r = gather(j, W, lines);
    if constexpr (PART) {
      const int64_t q = static_cast<int64_t>(seg) * cols + out;
      store_from_f32<float, 1>(pv + q, &r.v, spv);
      if constexpr (OP != 0)
        if (VBH_IN_SPAN(spi, pi + q, sizeof(int))) pi[q] = r.i;
    } else {
      write_result<To, 1, OP>(vals, idx, out, r.v, r.i, n, sv, si);
    }
  }
}

// Short middle axes: one lane per column and no exchange between lanes; bound by
// latency in the launches that take it (reduce_short_axis in capi.hip has both
// sides measured).  Consecutive lanes take consecutive columns and a slab's rows
// lie together, so that the lanes' narrow loads of several rows share lines; they
// are plain loads, which keep those.  Eight guarded loads in flight per lane were
// slower (mean bf16 16384 x 2 x 64: 0.77 of the speed, the guards' branches).
template <typename Ti, typename To, int OP>
__global__ __launch_bounds__(kColBlock) void reduce_short_cols(const Ti* __restrict__ x,
                                                               void* __restrict__ vals,
                                                               int64_t* __restrict__ idx,
                                                               uint32_t cols, int n,
                                                               uint32_t inner) {
  const uint32_t col = blockIdx.x * kColBlock + threadIdx.x;
  if (col >= cols) return;
  const uint32_t o = col / inner;
  const int64_t row = inner;
  const Ti* xc = x + o * (n * row) + (col - o * inner);
  const Span sx = VBH_SPAN(x, int64_t(cols) * n);
  const Span sv = VBH_SPAN(static_cast<To*>(vals), cols), si = VBH_SPAN(idx, cols);
  auto at = [&](int r) {
    float f;
    load_f32<Ti, 1>(xc + r * row, &f, sx);
    return f;
  };
  ValIdx best{OP == 0 ? 0.f : kNegInf, n};
  for (int r = 0; r < n; ++r) {
    const float f = at(r);
    if constexpr (OP == 0) best.v += f;
    else if (better(f, r, best.v, best.i)) best = ValIdx{f, r};
  }
  write_result<To, 1, OP>(vals, idx, col, best.v, best.i, n, sv, si);
}

// Second stage of a split middle axis: kCombineParts lanes per column, each
// over every kCombineParts-th of its `segs` (<= 64) partial results, then one.
constexpr int kCombineParts = 8;
constexpr int kCombineCols = kColBlock / kCombineParts;

template <typename To, int OP>
__global__ __launch_bounds__(kColBlock) void reduce_cols_combine(
    const float* __restrict__ pv, const int* __restrict__ pi, void* __restrict__ vals,
    int64_t* __restrict__ idx, int64_t cols, int n, int segs) {
  constexpr int M = kColMaxSegs / kCombineParts;
  __shared__ float lds_v[kColBlock];
  __shared__ int lds_i[kColBlock];
  const int t = static_cast<int>(threadIdx.x);
  const int j = t % kCombineCols, part = t / kCombineCols;
  const int64_t col = static_cast<int64_t>(blockIdx.x) * kCombineCols + j;
  const Span sp = VBH_SPAN(pv, cols * segs), spi = VBH_SPAN(pi, cols * segs);
  const Span sv = VBH_SPAN(static_cast<To*>(vals), cols), si = VBH_SPAN(idx, cols);
  ValIdx w[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const int s = part + m * kCombineParts;
    w[m] = ValIdx{OP == 0 ? 0.f : kNegInf, INT_MAX};
    if (s < segs && col < cols) {
      const int64_t q = s * cols + col;
      load_f32<float, 1>(pv + q, &w[m].v, sp);
      if constexpr (OP != 0) w[m].i = VBH_IN_SPAN(spi, pi + q, sizeof(int)) ? pi[q] : 0;
    }
  }
  auto fold = [](ValIdx a, ValIdx b) {
    if constexpr (OP == 0) return ValIdx{a.v + b.v, 0};
    else return pick(a, b);
  };
#pragma unroll
  for (int m = 1; m < M; ++m) w[0] = fold(w[0], w[m]);
  lds_v[t] = w[0].v;
  lds_i[t] = w[0].i;
  __syncthreads();
  if (part != 0 || col >= cols) return;
#pragma unroll
  for (int q = 1; q < kCombineParts; ++q)
    w[0] = fold(w[0], ValIdx{lds_v[q * kCombineCols + j], lds_i[q * kCombineCols + j]});
  write_result<To, 1, OP>(vals, idx, col, w[0].v, w[0].i, n, sv, si);
}

}  // namespace

hipError_t launch_reduce(const void* x, void* vals, int64_t* idx, int64_t outer, int n, int idt,
                         int odt, int op, const Geometry& g, hipStream_t s) {
  hipError_t err = hipErrorInvalidValue;
  auto body = [&](auto ti, auto to) {
    using Ti = typename decltype(ti)::type;
    using To = typename decltype(to)::type;
    constexpr int VN = Vec<Ti>::n;
    auto go = [&](auto opc) {
      constexpr int OP = decltype(opc)::value;
      auto launch = [&](auto kern) {
        launch_kernel(kern, dim3(grid_for(outer, g)), dim3(g.block), 0, s,
                           static_cast<const Ti*>(x), vals, idx, outer, n, g.tpr);
      };
      if (g.v == 1) launch(reduce_rows<Ti, To, 1, OP, false>);
      else if (g.mis) launch(reduce_rows<Ti, To, VN, OP, true>);
      else launch(reduce_rows<Ti, To, VN, OP, false>);
      err = hipGetLastError();
    };
    if (op == 0) go(std::integral_constant<int, 0>{});
    else if (op == 1) go(std::integral_constant<int, 1>{});
    else go(std::integral_constant<int, 2>{});
  };
  if (idt == odt) {
    dispatch_float_type(idt, [&](auto t) { body(t, t); });
  } else if (op == 0 && odt == kF32 && (idt == kF16 || idt == kBF16)) {
    dispatch_float_type(idt, [&](auto t) { body(t, TypeTag<float>{}); });
  } else if (op == 0 && idt == kF32 && (odt == kF16 || odt == kBF16)) {
    // second stage of a split mean: fp32 segment means in, the output type out
    dispatch_float_type(odt, [&](auto t) { body(TypeTag<float>{}, t); });
  }
  return err;
}

hipError_t launch_reduce_cols(const void* x, void* vals, int64_t* idx, void* parts,
                              int64_t outer, int n, int64_t inner, int idt, int odt, int op,
                              const ColGeometry& c, hipStream_t s) {
  hipError_t err = hipErrorInvalidValue;
  const int64_t cols = outer * inner;
  float* pv = static_cast<float*>(parts);
  int* pi = pv == nullptr ? nullptr : reinterpret_cast<int*>(pv + cols * c.segs);
  auto body = [&](auto ti, auto to) {
    using Ti = typename decltype(ti)::type;
    using To = typename decltype(to)::type;
    auto go = [&](auto opc, auto vc) {
      constexpr int OP = decltype(opc)::value;
      constexpr int V = decltype(vc)::value;
      auto launch = [&](auto kern) {
        launch_kernel(kern, dim3(static_cast<uint32_t>(c.grid), static_cast<uint32_t>(c.segs)),
                      dim3(kColBlock), 0, s, static_cast<const Ti*>(x), vals, idx, pv, pi, outer,
                      n, inner, c.cx, c.ty_log2, static_cast<uint32_t>(c.tiles), c.seg_n);
      };
      auto tiles = [&](auto nt) {
        constexpr bool NT = decltype(nt)::value;
        if (c.segs > 1) launch(reduce_cols<Ti, To, V, OP, true, NT>);
        else launch(reduce_cols<Ti, To, V, OP, false, NT>);
      };
      if (c.short_axis) {
        launch_kernel((reduce_short_cols<Ti, To, OP>), dim3(static_cast<uint32_t>(c.grid)),
                      dim3(kColBlock), 0, s, static_cast<const Ti*>(x), vals, idx,
                      static_cast<uint32_t>(cols), n, static_cast<uint32_t>(inner));
      } else {
        if (V > 1 && c.nt) tiles(std::bool_constant<(V > 1)>{});
        else tiles(std::false_type{});
        if (c.segs > 1)
          launch_kernel((reduce_cols_combine<To, OP>),
                        dim3(static_cast<uint32_t>((cols + kCombineCols - 1) / kCombineCols)),
                        dim3(kColBlock), 0, s, pv, pi, vals, idx, cols, n, c.segs);
      }
      err = hipGetLastError();
    };
    auto by_op = [&](auto vc) {
      if (op == 0) go(std::integral_constant<int, 0>{}, vc);
      else if (op == 1) go(std::integral_constant<int, 1>{}, vc);
      else go(std::integral_constant<int, 2>{}, vc);
    };
    if (c.v == 1) by_op(std::integral_constant<int, 1>{});
    else by_op(std::integral_constant<int, Vec<Ti>::n>{});
  };
  if (idt == odt) {
    dispatch_float_type(idt, [&](auto t) { body(t, t); });
  } else if (op == 0 && odt == kF32 && (idt == kF16 || idt == kBF16)) {
    dispatch_float_type(idt, [&](auto t) { body(t, TypeTag<float>{}); });
  }
  return err;
}

hipError_t launch_reduce_combine(const void* pvals, const int64_t* pidx, void* vals, int64_t* idx,
                                 int64_t rows, int segs, int segn, int dt, int op,
                                 hipStream_t s) {
  hipError_t err = hipErrorInvalidValue;
  const int64_t grid = (rows + 255) / 256;
  dispatch_float_type(dt, [&](auto t) {
    using T = typename decltype(t)::type;
    if (op == 1)
      launch_kernel((reduce_combine_vi<T, 1>), dim3(grid), dim3(256), 0, s,
                         static_cast<const T*>(pvals), pidx, vals, idx, rows, segs, segn);
    else
      launch_kernel((reduce_combine_vi<T, 2>), dim3(grid), dim3(256), 0, s,
                         static_cast<const T*>(pvals), pidx, vals, idx, rows, segs, segn);
    err = hipGetLastError();
  });
  return err;
}

}  // namespace vbh
