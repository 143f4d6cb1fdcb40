// Top-p alone over few rows: each row split over several workgroups (included by
// filter.hip; the definitions and the exact selection are stated there).
//
// filter_rows_kernel and filter_deferred_kernel give a row one 256-thread workgroup: 64
// rows of 128256 logits fill a quarter of the compute units and each row's statistics,
// histogram and listing passes are bound by one unit's vector arithmetic (86 + 100 us of a
// 225 us draw).  Here every pass of a row runs on P workgroups and the passes meet at
// kernel boundaries:
//   nucleus_stats_kernel: part p takes the canonical threads [T p, T (p+1)), T = 256 / P;
//     each of its threads runs 8 / P lanes of canon.h over their groups in order, so the
//     lane states are those of the one-workgroup pass, bit for bit;
//   nucleus_hist_kernel: every part evaluates the row's (M, Z) from the lane states (the
//     canonical tree; 16 KB from L2) and the fixed-point masses of its slice per
//     exponent bin (1024 bins in LDS);
//   nucleus_list_kernel: every part sums the parts' histograms, finds the bin that holds
//     t* and lists its slice's elements in it;
//   nucleus_finish_kernel: the walk over the listed keys gives t* and Z_K.  For sample()
//     (no draft position) every part runs it and then sums its share of the draw tiles;
//     otherwise one workgroup per row writes the row info;
//   nucleus_draw_kernel (sample()): the tile, lane and element of the draw point.
// bf16 rows skip the histogram and list kernels.  Their values are 16-bit keys, and a
// threshold with a nucleus worth the name lies within kNucWin of them below the row
// maximum (8 binades: down to a 256th of it).  So the statistics kernel also counts its
// part's elements per key, in a window of kNucWin keys below the part's own maximum (the
// slice is read again, from L2); the windows of the parts line up by absolute key, the
// mass at or above a key is a sum of count * mass, and t* and Z_K come from one scan.
// Measured on MI355X, sample() over 64 rows of 128256 bf16 logits, top_p = 0.95: 229 us with
// one workgroup per row, 69 us through the histogram and the list, 41 us this way
// (statistics 14, threshold and tiles 18, draw 7); fp32 rows 218 -> 64 us.
// A row whose bin does not list (ties), or whose threshold is not found in the bins or the
// window, takes the exact search of filter_deferred_kernel (large_threshold), in one
// workgroup.
// Rows outside canon.h's domain (+inf, all -inf, scores past 2^31) give what one workgroup
// per row gives; a row with a NaN has no defined result on either path.
// P = 8 up to 128 rows, 4 up to 256, 2 up to 512: at most four workgroups per compute unit
// (256 rows: 262 -> 76 us, 512 rows: 300 -> 125 us).
#pragma once

namespace bsx {
namespace filt {

constexpr int kNucMaxRows = 512;
constexpr int kNucMaxParts = 8;
constexpr int64_t kNucMaxWgs = 1024;  // rows * parts
constexpr int kNucList = 512;         // keys a part lists
constexpr int64_t kNucMinVocab = 8 * kLanes;
constexpr int kNucWin = 1024;         // bf16: keys counted below a part's maximum
static_assert(kNucWin * 4 <= kYBins * 8 && kNucWin % kThreads == 0, "counts fit hist");

inline int nucleus_parts(int64_t rows) { return rows <= 128 ? 8 : rows <= 256 ? 4 : 2; }

struct NucRec {
  float m, z;       // row statistics
  uint64_t base;    // mass above the bin that holds t*
  int32_t bin;      // that bin, or -1: not found among the bins
  int32_t pad;
};

struct NucArgs {
  const void* a;  // rows [0, n_a)
  int64_t n_a;
  const void* b;  // rows [n_a, ...)
  int64_t V;
  float c, top_p;
  RowInfo* info;
  float* lane_s;    // [rows][8][kThreads]: lane 8 t + i at [i][t]
  float* lane_r;    // [rows][8][kThreads]
  float* part_m;    // [rows][P]
  uint64_t* hist;   // [rows][P][kYBins]
  NucRec* rec;      // [rows]
  uint32_t* cnt;    // bf16: [rows][P][kNucWin], in place of hist
  uint32_t* top;    // bf16: [rows][P] the part's largest key >> 16
  uint32_t* keys;   // [rows][P][kNucList]
  int32_t* counts;  // [rows][P], -1: does not list
};

template <int DT>
__device__ __forceinline__ const char* nuc_row(const NucArgs& a, int64_t r) {
  const size_t esz = DT == BSX_DTYPE_FP32 ? 4 : 2;
  return r < a.n_a ? static_cast<const char*>(a.a) + r * a.V * esz
                   : static_cast<const char*>(a.b) + (r - a.n_a) * a.V * esz;
}

template <int DT>
__device__ __forceinline__ bool nuc_vec(const char* row, int64_t V) {
  return (V * (DT == BSX_DTYPE_FP32 ? 4 : 2)) % 16 == 0 && ((uintptr_t)row) % 16 == 0;
}

// Calls f(x) for the elements of the groups [g0, g1) of the row.
template <int DT, typename F>
__device__ __forceinline__ void for_each_in_groups(const void* row, int64_t V, bool vec,
                                                   int64_t g0, int64_t g1, F&& f) {
  const int t = threadIdx.x;
  const int64_t gw = vec ? min(g1, V / kGroup) : g0;  // whole groups in 16-byte loads
  constexpr int U = 4;
  for (int64_t g = g0 + t; g < gw; g += kThreads * U) {
    float x[U][8];
#pragma unroll
    for (int u = 0; u < U; ++u) load8<DT>(row, g + kThreads * u < gw ? g + kThreads * u : g, x[u]);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (g + kThreads * u < gw) {
#pragma unroll
        for (int e = 0; e < 8; ++e) f(x[u][e]);
      }
  }
  for (int64_t v = max(g0, gw) * kGroup + t; v < min(g1 * kGroup, V); v += kThreads)
    f(load_one<DT>(row, v));
}

// The 8 elements of a group from its 16-byte words.
template <int DT, int W>
__device__ __forceinline__ void unpack8(const u32x4 (&w)[W], float (&x)[8]) {
  if constexpr (DT == BSX_DTYPE_FP32) {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = __uint_as_float(w[e >> 2][e & 3]);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = (e & 1) ? hi_f32<DT>(w[0][e >> 1]) : lo_f32<DT>(w[0][e >> 1]);
  }
}

template <int DT, int P>
__global__ void __launch_bounds__(kThreads) nucleus_stats_kernel(NucArgs a) {
  __shared__ float s_max[kThreads / 64];
  constexpr int T = kThreads / P;                  // canonical threads of a part
  constexpr int LPT = 8 * T / kThreads;            // lanes per thread
  const int64_t r = blockIdx.x / P;
  const int p = (int)(blockIdx.x % P);
  const int64_t V = a.V;
  const char* row = nuc_row<DT>(a, r);
  const bool vec = nuc_vec<DT>(row, V);
  const int64_t G = ceil_div(V, kGroup), G_whole = V / kGroup;
  float mx = -INFINITY;
  // Groups loaded at once: all of a lane's whole rounds for the usual vocabularies (the
  // pass is a few memory round trips long, not bandwidth).
  constexpr int U = DT == BSX_DTYPE_FP32 ? 4 : 8;
  u32x4 held[U];  // bf16 rows, one lane per thread: its first U groups, counted below
#pragma unroll
  for (int u = 0; u < LPT; ++u) {
    const int q = (int)threadIdx.x + kThreads * u;
    const int t = T * p + q % T, i = q / T;  // canonical thread and lane slot
    LaneState st;
    st.m = -INFINITY;
    st.s = 0.f;
    st.r = canon::kRefStart;
    // rounds that are whole for the canonical thread (row_stats' whole rounds)
    int64_t j = 0;
    const int64_t whole = vec ? max((int64_t)0, (G_whole - 1 - t - 256 * 7 + kLanes) / kLanes) : 0;
    for (; j < whole; j += U) {
      u32x4 raw[U][DT == BSX_DTYPE_FP32 ? 2 : 1];
#pragma unroll
      for (int h = 0; h < U; ++h) {
        const int64_t g = t + 256 * i + kLanes * min(j + h, whole - 1);
#pragma unroll
        for (int w = 0; w < (DT == BSX_DTYPE_FP32 ? 2 : 1); ++w)
          raw[h][w] = reinterpret_cast<const u32x4*>(row)[(DT == BSX_DTYPE_FP32 ? 2 : 1) * g + w];
      }
#pragma unroll
      for (int h = 0; h < U; ++h) {
        if (LPT == 1 && DT == BSX_DTYPE_BF16 && j == 0) held[h] = raw[h][0];
        if (j + h < whole) {
          float x[8];
          unpack8<DT>(raw[h], x);
          float gm = x[0];
#pragma unroll
          for (int e = 1; e < 8; ++e) gm = __builtin_elementwise_maximum(gm, x[e]);
          const float rr = canon::lane_reference(st, gm, a.c);
          float gs = canon::weight(x[0], a.c, -rr);
#pragma unroll
          for (int e = 1; e < 8; ++e) gs = gs + canon::weight(x[e], a.c, -rr);
          st.s = st.s + gs;
        }
      }
    }
    for (j = whole; t + 256 * i + kLanes * j < G; ++j) {
      float x[8];
      const int n = load_group<DT>(row, t + 256 * i + kLanes * j, V, vec, x);
      float gm = x[0];
#pragma unroll
      for (int e = 1; e < 8; ++e)
        if (e < n) gm = fmaxf(gm, x[e]);
      canon::lane_update(st, x, n, gm, a.c);
    }
    a.lane_s[(r * 8 + i) * kThreads + t] = st.s;
    a.lane_r[(r * 8 + i) * kThreads + t] = st.r;
    mx = fmaxf(mx, st.m);
  }
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) mx = fmaxf(mx, __shfl_xor(mx, m));
  if ((threadIdx.x & 63) == 0) s_max[threadIdx.x >> 6] = mx;
  __syncthreads();
  const float pm = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
  if (threadIdx.x == 0) a.part_m[r * P + p] = pm;
  if constexpr (DT == BSX_DTYPE_BF16) {
    // counts of the part's groups (t + 256 i + 2048 j, t in [T p, T (p + 1))) per key
    __shared__ uint32_t cnt[kNucWin];
    const uint32_t top = okey(pm) >> 16;
    for (int w = threadIdx.x; w < kNucWin; w += kThreads) cnt[w] = 0u;
    __syncthreads();
    auto count = [&](float x) {
      const uint32_t d = top - (okey(x) >> 16);
      if (d < (uint32_t)kNucWin) atomicAdd(&cnt[d], 1u);
    };
    int64_t j0 = 0;
    if constexpr (LPT == 1) {
      // this thread's first groups are in registers
      const int t = T * p + (int)threadIdx.x % T;
      const int64_t whole =
          vec ? max((int64_t)0, (G_whole - 1 - t - 256 * 7 + kLanes) / kLanes) : 0;
#pragma unroll
      for (int h = 0; h < U; ++h)
        if (h < whole) {
          const u32x4 w[1] = {held[h]};
          float x[8];
          unpack8<DT>(w, x);
#pragma unroll
          for (int e = 0; e < 8; ++e) count(x[e]);
        }
      j0 = min(whole, (int64_t)U);
    }
    // the other groups of its lanes, read again (from L2)
#pragma unroll
    for (int u = 0; u < LPT; ++u) {
      const int q = (int)threadIdx.x + kThreads * u;
      const int64_t g0 = T * p + q % T + 256 * (q / T);
      constexpr int R = 4;
      for (int64_t j = j0; g0 + kLanes * j < G; j += R) {
        float x[R][8];
        int n[R];
#pragma unroll
        for (int h = 0; h < R; ++h) {
          const int64_t g = g0 + kLanes * (j + h);
          n[h] = 0;
          if (vec && g < G_whole) {
            load8<DT>(row, g, x[h]);
            n[h] = 8;
          } else if (g < G) {
            n[h] = load_group<DT>(row, g, V, vec, x[h]);
          }
        }
#pragma unroll
        for (int h = 0; h < R; ++h)
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (e < n[h]) count(x[h][e]);
      }
    }
    __syncthreads();
    for (int w = threadIdx.x; w < kNucWin; w += kThreads)
      a.cnt[(r * P + p) * kNucWin + w] = cnt[w];
    if (threadIdx.x == 0) a.top[r * P + p] = top;
  }
}

// (M, Z) of row r from its lane states: row_stats' epilogue.  Every thread calls it.
template <int P>
__device__ __forceinline__ void nuc_row_stats(const NucArgs& a, int64_t r, float* M, float* Z) {
  __shared__ float wave_val[kThreads / 64];
  const int t = threadIdx.x;
  float ls[8], lr[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    ls[i] = a.lane_s[(r * 8 + i) * kThreads + t];
    lr[i] = a.lane_r[(r * 8 + i) * kThreads + t];
  }
  float mx = a.part_m[r * P];
#pragma unroll
  for (int q = 1; q < P; ++q) mx = fmaxf(mx, a.part_m[r * P + q]);
  const float rho_m = mx * a.c;
  float w[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) w[i] = canon::lane_rescaled(LaneState{0.f, ls[i], lr[i]}, rho_m);
  float s = ((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7]));
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) s = s + __shfl_xor(s, m);
  if ((t & 63) == 0) wave_val[t >> 6] = s;
  __syncthreads();
  *M = mx;
  *Z = (wave_val[0] + wave_val[1]) + (wave_val[2] + wave_val[3]);
}

__device__ __forceinline__ bool finite_f(float x) { return x > -INFINITY && x < INFINITY; }

template <int DT, int P>
__global__ void __launch_bounds__(kThreads) nucleus_hist_kernel(NucArgs a) {
  __shared__ uint64_t hist[kYBins];
  const int64_t r = blockIdx.x / P;
  const int p = (int)(blockIdx.x % P);
  for (int i = threadIdx.x; i < kYBins; i += kThreads) hist[i] = 0ull;
  float M, Z;
  nuc_row_stats<P>(a, r, &M, &Z);  // (its barrier also orders the cleared histogram)
  const float neg = -(M * a.c);
  if (p == 0 && threadIdx.x == 0) {
    a.rec[r].m = M;
    a.rec[r].z = Z;
  }
  const char* row = nuc_row<DT>(a, r);
  const int64_t G = ceil_div(a.V, kGroup);
  if (finite_f(neg))
    for_each_in_groups<DT>(row, a.V, nuc_vec<DT>(row, a.V), G * p / P, G * (p + 1) / P,
                           [&](float x) {
                             const float y = fmaf(x, a.c, neg);
                             const float q = -y * kYScale;  // ypos(x, c, neg)
                             if (!(q < (float)(kYBins - 1))) return;
                             atomicAdd(reinterpret_cast<unsigned long long*>(
                                           &hist[(int)fmaxf(q, 0.0f)]),
                                       (unsigned long long)mass_of_exponent(y));
                           });
  __syncthreads();
  for (int i = threadIdx.x; i < kYBins; i += kThreads)
    a.hist[(r * P + p) * kYBins + i] = hist[i];
}

__device__ __forceinline__ uint64_t nuc_target(const NucArgs& a, float Z) {
  return (uint64_t)ceilf((a.top_p * Z) * 0x1p40f);
}

template <int DT, int P>
__global__ void __launch_bounds__(kThreads) nucleus_list_kernel(NucArgs a) {
  __shared__ __align__(16) RowsLds L;
  const int t = threadIdx.x;
  const int64_t r = blockIdx.x / P;
  const int p = (int)(blockIdx.x % P);
  const float M = a.rec[r].m, Z = a.rec[r].z;
  const float neg = -(M * a.c);
  uint64_t* mass = reinterpret_cast<uint64_t*>(L.hist);
  constexpr int PER = kYBins / kThreads;
  uint64_t h[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) h[i] = 0ull;
#pragma unroll
  for (int q = 0; q < P; ++q)
#pragma unroll
    for (int i = 0; i < PER; ++i) h[i] += a.hist[(r * P + q) * kYBins + kThreads * i + t];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    mass[kThreads * i + t] = h[i];
    L.ckey[kThreads * i + t] = 0u;
  }
  if (t == 0) L.count = 0;
  __syncthreads();
  const int b0 = finite_f(neg) ? ybin_first(L, L.ckey, mass, kYBins - 1, 0u, 0ull, false, true, 0,
                                            nuc_target(a, Z))
                               : -1;
  if (p == 0 && t == 0) {
    a.rec[r].base = b0 < 0 ? 0ull : L.above_m;
    a.rec[r].bin = b0;
  }
  if (b0 < 0) {
    if (t == 0) a.counts[r * P + p] = -1;
    return;
  }
  float xlo, xhi;
  ybin_range(L, b0, -1, a.c, neg, &xlo, &xhi);
  const char* row = nuc_row<DT>(a, r);
  const int64_t G = ceil_div(a.V, kGroup);
  uint32_t* keys = a.keys + (r * P + p) * kNucList;
  for_each_in_groups<DT>(row, a.V, nuc_vec<DT>(row, a.V), G * p / P, G * (p + 1) / P,
                         [&](float x) {
                           if (x >= xlo && x <= xhi) {
                             const int slot = atomicAdd(&L.count, 1);
                             if (slot < kNucList) keys[slot] = okey(x);
                           }
                         });
  __syncthreads();
  if (t == 0) a.counts[r * P + p] = L.count <= kNucList ? L.count : -1;
}

// bf16: t* and Z_K of row r from the parts' counts; false when t* is not in the window.
// Every thread calls it.
template <int P>
__device__ __forceinline__ bool nucleus_count_threshold(const NucArgs& a, int64_t r, RowsLds& L,
                                                        NucRec& rec) {
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  constexpr int PER = kNucWin / kThreads;
  uint32_t tops[P], top = 0u;
#pragma unroll
  for (int q = 0; q < P; ++q) {
    tops[q] = a.top[r * P + q];
    top = max(top, tops[q]);
  }
  // thread t: the keys top - (PER t + i); the part's window starts at its own top
  // (unconditional loads, all in flight together)
  uint32_t raw[P][PER], c[PER];
#pragma unroll
  for (int q = 0; q < P; ++q)
#pragma unroll
    for (int i = 0; i < PER; ++i)
      raw[q][i] = a.cnt[(r * P + q) * kNucWin + max(PER * t + i - (int)(top - tops[q]), 0)];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    c[i] = 0u;
#pragma unroll
    for (int q = 0; q < P; ++q)
      c[i] += PER * t + i >= (int)(top - tops[q]) ? raw[q][i] : 0u;
  }
  nuc_row_stats<P>(a, r, &rec.m, &rec.z);
  const float neg = -(rec.m * a.c);
  const uint64_t target = nuc_target(a, rec.z);
  if (t == 0) {
    L.bin = INT_MAX;
    L.nk = -1;
  }
  uint64_t m[PER], mine = 0ull;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    uint32_t key = (top - (uint32_t)(PER * t + i)) << 16;
    if (!(key & 0x80000000u)) key |= 0xffffu;  // (images of negative values end in ones)
    m[i] = c[i] ? (uint64_t)c[i] * fx40(canon::weight(key_value(key), a.c, neg)) : 0ull;
    mine += m[i];
  }
  const uint64_t incl = wave_prefix_u64(mine);
  uint64_t* wt = reinterpret_cast<uint64_t*>(L.part);
  if (lane == 63) wt[wave] = incl;
  __syncthreads();
  uint64_t run = incl - mine;
  for (int w = 0; w < wave; ++w) run += wt[w];
  int first = -1;
  uint64_t zk = 0ull;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    run += m[i];
    if (first < 0 && c[i] != 0u && run >= target) {
      first = PER * t + i;
      zk = run;
    }
  }
  if (first >= 0) atomicMin(&L.bin, first);
  __syncthreads();
  const int d = L.bin;
  if (d == INT_MAX || !finite_f(neg)) return false;
  if (first == d) {
    uint32_t key = (top - (uint32_t)d) << 16;
    if (!(key & 0x80000000u)) key |= 0xffffu;
    L.tk = key;
    L.zk = zk;
  }
  __syncthreads();
  return true;
}

// t* and Z_K of row r into L.tk and L.zk (L.nk = -1: no list) from what the parts left, or
// false (in every thread).  rec: the row's record (bf16: filled here).
template <int DT, int P>
__device__ __forceinline__ bool nucleus_threshold(const NucArgs& a, int64_t r, RowsLds& L,
                                                  NucRec& rec) {
  if constexpr (DT == BSX_DTYPE_BF16) return nucleus_count_threshold<P>(a, r, L, rec);
  rec = a.rec[r];
  const int t = threadIdx.x;
  const float neg = -(rec.m * a.c);
  const uint64_t target = nuc_target(a, rec.z);
  int cnt[P], n = 0;
  bool ok = rec.bin >= 0;
#pragma unroll
  for (int q = 0; q < P; ++q) {
    cnt[q] = a.counts[r * P + q];
    ok &= cnt[q] >= 0;
    n += cnt[q];
  }
  ok &= n <= kCands;
  if (ok) {
    int base = 0;
#pragma unroll
    for (int q = 0; q < P; ++q) {
      for (int s = t; s < cnt[q]; s += kThreads)
        L.ckey[base + s] = a.keys[(r * P + q) * kNucList + s];
      base += cnt[q];
    }
    __syncthreads();
    ok = walk_listed_bin(L, n, rec.bin, a.c, neg, false, true, 0, target, 0u, rec.base);
  }
  return ok;
}

template <int DT>
__device__ __forceinline__ void nucleus_exact(const NucArgs& a, int64_t r, RowsLds& L,
                                              const NucRec& rec) {
  const char* row = nuc_row<DT>(a, r);
  __syncthreads();
  large_threshold<DT>(L, row, a.V, nuc_vec<DT>(row, a.V), a.c, -(rec.m * a.c), false, true, 0,
                      nuc_target(a, rec.z));
}

template <int DT, int P>
__global__ void __launch_bounds__(kThreads) nucleus_finish_kernel(NucArgs a) {
  __shared__ __align__(16) RowsLds L;
  const int64_t r = blockIdx.x;
  NucRec rec;
  if (!nucleus_threshold<DT, P>(a, r, L, rec)) nucleus_exact<DT>(a, r, L, rec);
  write_info(L, a.info + r, rec.m);
}

// sample(): the threshold in every part of the row (the same in each), then the part's
// share of the draw tiles (filter_tiles_kernel's sums without a draft).
template <int DT, int P>
__global__ void __launch_bounds__(kThreads, 4) nucleus_tiles_kernel(NucArgs a, ChainArgs ca) {
  __shared__ __align__(16) RowsLds L;
  const int64_t r = blockIdx.x / P;
  const int p = (int)(blockIdx.x % P);
  const int E = draw_tile_elems(a.V), ntiles = draw_tiles(a.V);
  int T0 = ntiles * p / P, T1 = ntiles * (p + 1) / P;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  constexpr int W = kThreads / 64, U = DT == BSX_DTYPE_FP32 ? 4 : 8;
  const char* row = nuc_row<DT>(a, r);
  const bool vec = nuc_vec<DT>(row, a.V);
  const bool groups = vec && E == kGroup && a.V % kGroup == 0;  // one whole group per lane
  const int first = T0 + wave;
  u32x4 pre[U][DT == BSX_DTYPE_FP32 ? 2 : 1];
  auto load_tile = [&](int T, u32x4 (&w)[DT == BSX_DTYPE_FP32 ? 2 : 1]) {
    const int64_t g = min((int64_t)T * 64 + lane, a.V / kGroup - 1);
#pragma unroll
    for (int h = 0; h < (DT == BSX_DTYPE_FP32 ? 2 : 1); ++h)
      w[h] = reinterpret_cast<const u32x4*>(row)[(DT == BSX_DTYPE_FP32 ? 2 : 1) * g + h];
  };
  if (groups) {
#pragma unroll
    for (int u = 0; u < U; ++u) load_tile(first + W * u, pre[u]);
  }
  NucRec rec;
  if (!nucleus_threshold<DT, P>(a, r, L, rec)) {
    // (rare) one workgroup finds the threshold and sums all the tiles
    if (p != 0) return;
    nucleus_exact<DT>(a, r, L, rec);
    T0 = 0;
    T1 = ntiles;
  }
  __syncthreads();
  RowInfo ri;
  ri.m = rec.m;
  ri.inv_k = 1.0f / (canon::u64_to_f32(L.zk) * 0x1p-40f);
  ri.t_key = L.tk;
  ri.n_list = -1;
  if (p == 0 && threadIdx.x == 0) a.info[r] = ri;
  DrawRow<DT> R;
  R.V = a.V;
  R.P = filtered_row<DT>(a.a, r, a.V, ri, a.c);
  R.Q = Filtered<DT>{};
  R.has_q = R.qlog = false;
  R.xj = -1;
  R.vec8 = vec;
  if (groups) {
    // the first ones were loaded ahead of the threshold
    for (int Tb = T0 + wave; Tb < T1; Tb += W * U) {
      if (Tb != first) {
#pragma unroll
        for (int u = 0; u < U; ++u) load_tile(Tb + W * u, pre[u]);
      }
      uint64_t sp[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float x[8];
        unpack8<DT>(pre[u], x);
        sp[u] = 0ull;
        const int64_t v0 = ((int64_t)(Tb + W * u) * 64 + lane) * kGroup;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float pe = okey(x[e]) >= ri.t_key ? canon::weight(x[e], a.c, R.P.nmc) * ri.inv_k : 0.0f;
          sp[u] += fx40(pe);
        }
        if (v0 >= a.V) sp[u] = 0ull;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint64_t s = wave_sum_u64(sp[u]);
        if (lane == 0 && Tb + W * u < T1) ca.tiles[r * ntiles + Tb + W * u] = s;
      }
    }
    return;
  }
  for (int T = T0 + wave; T < T1; T += W) {
    uint64_t sq, sp;
    R.sums((int64_t)T * 64 * E + (int64_t)lane * E, E, sq, sp);
    const uint64_t s = wave_sum_u64(sp);
    if (lane == 0) ca.tiles[r * ntiles + T] = s;
  }
}

// sample(): the draw of row r over its tile sums, as chain_request without a list or a
// draft: the first tile, lane and element whose running sum exceeds the draw point (the
// last non-zero one if none does).
template <int DT>
__global__ void __launch_bounds__(kThreads) nucleus_draw_kernel(ChainArgs ca) {
  __shared__ uint64_t s_wave[kThreads / 64];
  __shared__ uint64_t s_base;
  __shared__ int s_tile, s_last;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const int64_t r = blockIdx.x;
  const int64_t V = ca.V;
  const int E = draw_tile_elems(V), ntiles = draw_tiles(V);
  constexpr int PER = kMaxTiles / kThreads;
  const uint64_t* ts = ca.tiles + r * ntiles;
  // thread t: tiles [n t, n t + n)
  const int n = (ntiles + kThreads - 1) / kThreads;
  uint64_t x[PER], mine = 0ull;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int T = t * n + i;
    x[i] = ts[min(T, ntiles - 1)];
    if (i >= n || T >= ntiles) x[i] = 0ull;
    mine += x[i];
  }
  const RowInfo ri = ca.info[r];
  const float u = ca.uniforms[r];
  if (t == 0) {
    s_tile = -1;
    s_last = -1;
    s_base = 0ull;
  }
  const uint64_t incl = wave_prefix_u64(mine);
  if (lane == 63) s_wave[wave] = incl;
  __syncthreads();
  uint64_t base = incl - mine, total = 0ull;
  for (int w = 0; w < kThreads / 64; ++w) {
    if (w < wave) base += s_wave[w];
    total += s_wave[w];
  }
  const uint64_t tp = canon::draw_point(u, total);
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    if (x[i] != 0ull) {
      if (tp >= base && tp < base + x[i]) {
        s_tile = t * n + i;
        s_base = base;
      }
      atomicMax(&s_last, t * n + i);
    }
    base += x[i];
  }
  __syncthreads();
  if (wave != 0) return;
  const bool found = s_tile >= 0;
  const int tile = found ? s_tile : s_last;
  int tok = -1;
  if (tile >= 0) {
    DrawRow<DT> R;
    R.V = V;
    R.P = filtered_row<DT>(ca.t_logits, r, V, ri, ca.c);
    R.Q = Filtered<DT>{};
    R.has_q = R.qlog = false;
    R.xj = -1;
    R.vec8 = nuc_vec<DT>(static_cast<const char*>(R.P.row), V);
    const int64_t v0 = (int64_t)tile * 64 * E + (int64_t)lane * E;
    uint64_t sq, ls;
    R.sums(v0, E, sq, ls);
    const uint64_t li = wave_prefix_u64(ls), le = li - ls;
    const uint64_t tt = tp - s_base;
    const uint64_t nz = __builtin_amdgcn_ballot_w64(ls != 0ull);
    const bool my_lane = found ? (ls != 0ull && tt >= le && tt < li)
                               : (nz != 0ull && lane == 63 - __builtin_clzll(nz));
    if (my_lane) {
      uint64_t cum = le;
      bool done = false;
      for (int e0 = 0; e0 < E && v0 + e0 < V && !done; e0 += 8) {
        uint64_t rq[8], rp[8];
        R.at8(v0 + e0, rq, rp);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          cum += rp[e];
          if (!done && rp[e] != 0ull) {
            tok = (int)(v0 + e0 + e);  // the last non-zero element so far
            done = found && cum > tt;
          }
        }
      }
    }
    const uint64_t who = __builtin_amdgcn_ballot_w64(my_lane);
    tok = __shfl(tok, who != 0ull ? __builtin_ctzll(who) : 0);
  }
  if (lane == 0) {
    const int32_t id = tok;
    ca.out_ids[r] = id;
    ca.accepted[r] = 0;
    ca.emitted[r] = 0;
    write_verdict(ca.verdict, (int)r, &id, 0, 0);
  }
}

}  // namespace filt
}  // namespace bsx
