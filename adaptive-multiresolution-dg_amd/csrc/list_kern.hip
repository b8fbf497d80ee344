// Source lists of the fibers and the sweeps that run on them; see list.hpp.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <stdexcept>

#include "list.hpp"

namespace adg {
namespace {

constexpr int kBlock = 256;
constexpr int kWave = 64;

inline unsigned nblocks(int64_t n) { return static_cast<unsigned>((n + kBlock - 1) / kBlock); }

// Sources requested together: four on small grids, where a launch waits for
// the longest lists of its few wavefronts, two on large ones, where the
// registers of four cost more resident wavefronts than the overlap saves
// (4D sparse grid of 10,496 elements: 9.3 ms a run with two, 8.0 with four;
// 512 2D instances, 90 to 165 thousand elements: 18.9 and 20.0 ms).
constexpr int64_t kFewElements = 16384;

// ---------------------------------------------------------------------------
// build

// Whether the cells of two slots are nested (their supports overlap).
__device__ __forceinline__ bool nested(int a, int b) {
  const int la = slot_level(a), lb = slot_level(b);
  if (la <= 1 || lb <= 1) return true;
  return la >= lb ? (a >> (la - lb)) == b : (b >> (lb - la)) == a;
}

__global__ __launch_bounds__(kBlock) void k_list_nz(uint32_t* nz, const double* M, int ns, int nw, int block,
                                                    int in_support) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= static_cast<int64_t>(ns) * ns) return;
  const int st = static_cast<int>(i / ns), s = static_cast<int>(i % ns);
  bool any = M == nullptr;
  if (M)
    for (int j = 0; j < block; ++j) any = any || M[i * block + j] != 0.;
  if (any && (!in_support || nested(st, s))) atomicOr(&nz[st * nw + (s >> 5)], 1u << (s & 31));
}

__global__ __launch_bounds__(kBlock) void k_list_clear(uint32_t* nz, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) nz[i] = 0;
}

__global__ void k_list_zero(int32_t* p, int n) {
  if (static_cast<int>(threadIdx.x) < n) p[threadIdx.x] = 0;
}

// G threads per (dimension, target) for up to three kinds of lists at once.
// The sources of a target are the set bits of (occupancy of its fiber) AND (the
// target slot's row of nonzero pairs), in slot order; each thread counts and
// later writes those of its run of 16-cell pieces, so the threads of a block in
// order hold the block's entries in order.  The block takes room for them with
// one atomic add per list.  Where a target's entries lie differs from run to
// run, what they hold does not.
// Bound: latency of the bit words and the fiber map.  Walking the relation a
// cell at a time, a thread per (list, target): 590 us for 237 thousand elements
// of the rotating wave at level 9 (the coarse targets' walks), 168 us for 90 to
// 165 thousand of 512 Burgers solves, 68 us for 145 elements; a thread per
// target over words 747, 54 and 24 us; now 249, 53 and 13 us.
constexpr int kPiece = 16;

template <int G>
__global__ __launch_bounds__(kBlock) void k_list_build(ListBuildArgs a, int kind0, int nkind) {
  constexpr int NK = 3;
  __shared__ int s_wave[NK][kBlock / kWave];
  __shared__ int s_base[NK];
  const int d = blockIdx.y;
  const int64_t e = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / G;
  const int g = threadIdx.x % G, lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int32_t* fmap = a.fmap[d];
  const int nw = (a.ns + 31) / 32;
  int st = 0, fb = 0, maxl = -1, lt = 0;
  if (e < a.E) {
    st = a.slot[d][e];
    lt = slot_level(st);
    fb = a.fbase[d][e];
    maxl = a.fmaxl[d][e];
    if (a.level_cap >= 0) {  // coarse grid (FastMultiplyLU::transform_1D_coarse_grid)
      const int ls = a.lsum[e];
      maxl = ls > a.level_cap ? -1 : min(maxl, a.level_cap - ls + lt);
    }
  }
  // the cells of levels 0 .. maxl are the slots below 2^maxl
  const int cells = maxl < 0 ? 0 : 1 << maxl;
  const int per = ((cells + kPiece - 1) / kPiece + G - 1) / G;  // pieces of a thread
  const int p0 = g * per, p1 = min(p0 + per, (cells + kPiece - 1) / kPiece);
  const uint32_t* occ = a.fbits[d] + (fb >> 5);
  const int64_t row = static_cast<int64_t>(st) * nw;
  // present cells of piece p (a fiber of fewer than 32 cells shares its word)
  auto present = [&](int p) {
    const uint32_t m = (occ[p >> 1] >> (fb & 31)) >> (p & 1) * kPiece & 0xffffu;
    return cells < (p + 1) * kPiece ? m & ((1u << max(cells - p * kPiece, 0)) - 1u) : m;
  };
  auto pairs = [&](int q, int p) { return a.nz[kind0 + q][row + (p >> 1)] >> (p & 1) * kPiece; };
  int n[NK] = {0, 0, 0}, nu[NK] = {0, 0, 0};
  for (int p = p0; p < p1; ++p) {
    const uint32_t m = present(p);
    // slots of levels up to lt: below 2^lt
    const int up_cells = (1 << lt) - p * kPiece;
    const uint32_t up = up_cells >= kPiece ? 0xffffu : (up_cells <= 0 ? 0u : (1u << up_cells) - 1u);
#pragma unroll
    for (int q = 0; q < NK; ++q)
      if (q < nkind) {
        const uint32_t mq = m & pairs(q, p);
        n[q] += __popc(mq);
        nu[q] += __popc(mq & up);
      }
  }
  int beg[NK], all[NK];
#pragma unroll
  for (int q = 0; q < NK; ++q) {
    int inc = n[q];  // inclusive sum over the wavefront
    for (int o = 1; o < kWave; o <<= 1) {
      const int v = __shfl_up(inc, o);
      if (lane >= o) inc += v;
    }
    if (lane == kWave - 1) s_wave[q][wave] = inc;
    beg[q] = inc - n[q];
    all[q] = __shfl(inc, lane - g + G - 1) - __shfl(beg[q], lane - g);
    for (int o = 1; o < G; o <<= 1) nu[q] += __shfl_xor(nu[q], o);
  }
  __syncthreads();
  if (static_cast<int>(threadIdx.x) < nkind) {
    const int q = threadIdx.x;
    int sum = 0;
    for (int w = 0; w < kBlock / kWave; ++w) {
      const int v = s_wave[q][w];
      s_wave[q][w] = sum;
      sum += v;
    }
    s_base[q] = atomicAdd(&a.total[(kind0 + q) * a.D + d], sum);
  }
  __syncthreads();
  if (e >= a.E) return;
  for (int q = 0; q < nkind; ++q) {
    const int list = (kind0 + q) * a.D + d;
    int at = beg[q] + s_base[q] + s_wave[q][wave], left = n[q];
    if (static_cast<int64_t>(at) + left > a.cap[list]) {  // (the host's bound is exceeded: never)
      atomicOr(a.err, ERR_LIST);
      left = all[q] = 0;
    }
    if (g == 0) a.meta[list][e] = make_int4(all[q] ? at : 0, all[q] ? nu[q] | all[q] << 16 : 0, st, a.inst[e]);
    int2* ent = a.ent[list];
    int p = p0;
    uint32_t m = left > 0 ? present(p) & pairs(q, p) : 0;
    for (; left > 0; left -= 4, at += 4) {  // four sources at a time
      int s[4], src[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s[j] = s[0];
        if (j < left) {
          while (!m) {
            ++p;
            m = present(p) & pairs(q, p);
          }
          s[j] = kPiece * p + __builtin_ctz(m);
          m &= m - 1;
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) src[j] = fmap[fb + s[j]];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j < left) ent[at + j] = make_int2(src[j], s[j]);
    }
  }
}

// ---------------------------------------------------------------------------
// sweeps
//
// A thread evaluates one rest index of a target (the PT outputs of the swept
// dimension): per source it takes an 8-byte entry, the PF values of the source
// and its PF*PT table block.  Bound: the vector memory unit, which takes a
// wavefront's load in 16 cycles or more whatever its width (busy 73 % of the
// time; table and value loads about a third each).  Hence in the phases of
// large grids the R lanes of a target fetch a table block once between them and
// read it from LDS (7 of 12 loads less), and the phases lay their outputs out
// so that the next sweep's values are one run (2 loads instead of 4).  The last
// sweeps keep their own table loads: sharing costs their term values LDS, and
// they lose more wavefronts than it saves (1984 us against 1812).  More rest
// indices per thread (2, 4) save table loads but scatter the value loads and
// lose wavefronts; copying the blocks of several sources to LDS in rounds was
// 1.2 to 3 times slower (lists are 3 to 5 sources long).
// 256 3D instances, 213 thousand elements, k = 2, m = 3, us per launch: the two
// right-hand-side phases 1597 plain, 1142 with shared blocks, 1061 with runs
// (walking the fibers: 2300); last sweeps 1950, 1739 with runs (2900); 23
// rotating-wave instances: phase 580, 447, 412, last sweeps 880, 800.

// Loads through the global address space at a uniform base plus a 32-bit byte
// offset (list_stage_fits() keeps every array a sweep reads below 4 GiB).
template <class T>
__device__ __forceinline__ T gl(const void* base, uint32_t bytes, int i = 0) {
  return ((const __attribute__((address_space(1))) T*)((const __attribute__((address_space(1))) char*)base + bytes))[i];
}
typedef int vi2 __attribute__((ext_vector_type(2)));
typedef int vi4 __attribute__((ext_vector_type(4)));

// Input and table of a term for values of type T.  x[k]: values k of a source
// (the swept dimension has stride sdd; RUN: 1, one run of values) at the offset
// of its element and rest index; m: the N values of the table block of (target slot, source slot).
template <class T, int PF, bool RUN>
struct ListIn;
template <int PF, bool RUN>
struct ListIn<double, PF, RUN> {
  const double* x[PF];
  const double* m;
  __device__ __forceinline__ ListIn(const ListTerm& t, const double* u, int64_t E) : m(t.M) {
    const double* b = (t.in ? t.in : u) + t.comp * (E * t.comp_size);
    for (int k = 0; k < PF; ++k) x[k] = b + k * t.sdd;
  }
  __device__ __forceinline__ void values(uint32_t at, double (&v)[PF]) const {
#pragma unroll
    for (int k = 0; k < PF; ++k) v[k] = RUN ? gl<double>(x[0], at * 8, k) : gl<double>(x[k], at * 8);
  }
  template <int N>
  struct Block { double w[N]; };
  template <int N>
  __device__ __forceinline__ Block<N> block(uint32_t at) const {
    Block<N> b;
#pragma unroll
    for (int i = 0; i < N; ++i) b.w[i] = gl<double>(m, at * 8, i);
    return b;
  }
  template <int N>
  static __device__ __forceinline__ void madd(double& acc, double v, const Block<N>& b, int j) { acc += v * b.w[j]; }
  // piece p of block number b, and the product with a block in LDS
  template <int N, class Piece>
  __device__ __forceinline__ Piece piece(uint32_t b, int p) const {
    return gl<Piece>(m, b * (N * 8) + p * static_cast<int>(sizeof(Piece)));
  }
  template <int N>
  static __device__ __forceinline__ void madd_lds(double& acc, double v, const double* w, int j) { acc += v * w[j]; }
};
template <int PF, bool RUN>
struct ListIn<float, PF, RUN> {
  const double* x[PF];
  const float* x32[PF];
  const float *mh, *ml;
  bool f32;
  __device__ __forceinline__ ListIn(const ListTerm& t, const double* u, int64_t E) : mh(t.Mh), ml(t.Ml), f32(t.in32) {
    const double* b = (t.in ? t.in : u) + t.comp * (E * t.comp_size);
    const float* b32 = t.in32 + t.comp * (E * t.comp_size);
    for (int k = 0; k < PF; ++k) {
      x[k] = b + k * t.sdd;
      x32[k] = b32 + k * t.sdd;
    }
  }
  __device__ __forceinline__ void values(uint32_t at, float (&v)[PF]) const {
#pragma unroll
    for (int k = 0; k < PF; ++k)
      v[k] = f32 ? (RUN ? gl<float>(x32[0], at * 4, k) : gl<float>(x32[k], at * 4))
                 : static_cast<float>(RUN ? gl<double>(x[0], at * 8, k) : gl<double>(x[k], at * 8));
  }
  template <int N>
  struct Block { float h[N], l[N]; };
  template <int N>
  __device__ __forceinline__ Block<N> block(uint32_t at) const {
    Block<N> b;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      b.h[i] = gl<float>(mh, at * 4, i);
      b.l[i] = gl<float>(ml, at * 4, i);
    }
    return b;
  }
  template <int N>
  static __device__ __forceinline__ void madd(float& acc, float v, const Block<N>& b, int j) {
    acc = fmaf(v, b.l[j], acc);
    acc = fmaf(v, b.h[j], acc);
  }
  // the high parts of a block, then its low parts
  template <int N, class Piece>
  __device__ __forceinline__ Piece piece(uint32_t b, int p) const {
    constexpr int half = N * 4 / static_cast<int>(sizeof(Piece));
    const float* q = p < half ? mh : ml;
    return gl<Piece>(q, b * (N * 4) + (p < half ? p : p - half) * static_cast<int>(sizeof(Piece)));
  }
  template <int N>
  static __device__ __forceinline__ void madd_lds(float& acc, float v, const float* w, int j) {
    acc = fmaf(v, w[N + j], acc);
    acc = fmaf(v, w[j], acc);
  }
};

// acc[i] = sum over the sources of a target, ascending, k inner, of
// in[source][bin + k*sdd] * M(k, i).  NB sources are requested together.
template <int PF, int PT, class T, int NB, bool RUN>
__device__ __forceinline__ void list_sum(const ListTerm& t, const ListIn<T, PF, RUN>& src, const vi4 meta, uint32_t bin,
                                         T (&acc)[PT]) {
  constexpr int N = PF * PT;
#pragma unroll
  for (int i = 0; i < PT; ++i) acc[i] = T(0);
  const uint32_t nu = meta.y & 0xffff, na = static_cast<uint32_t>(meta.y) >> 16;
  const uint32_t lo = t.lu == LU_L ? nu : 0, hi = t.lu == LU_U ? nu : na;
  const uint32_t Mst = __umul24(meta.z, t.ns) * N;
  const uint32_t Tin = t.Tin;
  const uint32_t end = (meta.x + hi) * 8;
  for (uint32_t i = (meta.x + lo) * 8; i < end; i += 8 * NB) {
    vi2 en[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) en[j] = gl<vi2>(t.ent, j == 0 ? i : min(i + 8 * j, end - 8));
    typename ListIn<T, PF, RUN>::template Block<N> m[NB];
    T x[NB][PF];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      m[j] = src.template block<N>(Mst + en[j].y * N);
      src.values(__umul24(en[j].x, Tin) + bin, x[j]);
    }
#pragma unroll
    for (int j = 0; j < NB; ++j)
      if (j == 0 || i + 8 * j < end) {
#pragma unroll
        for (int q = 0; q < PT; ++q)
#pragma unroll
          for (int k = 0; k < PF; ++k) ListIn<T, PF, RUN>::template madd<N>(acc[q], x[j][k], m[j], k * PT + q);
      }
  }
}

// The same with the lanes of a target (rest indices c of R, side by side in the
// wavefront) loading each source's table block once between them: a lane
// fetches every R-th 16-byte piece and passes it through LDS.
template <int BYTES>
struct PieceOf;
template <>
struct PieceOf<16> { typedef unsigned int type __attribute__((ext_vector_type(4))); };
template <>
struct PieceOf<8> { typedef unsigned int type __attribute__((ext_vector_type(2))); };
template <>
struct PieceOf<4> { using type = unsigned int; };

template <class T, int N>
constexpr int piece_bytes() {
  if (sizeof(T) == 8) return N % 2 == 0 ? 16 : 8;
  return N % 4 == 0 ? 16 : (N % 2 == 0 ? 8 : 4);
}

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// lds: this target's N 8-byte words; pieces a lane fetches at most: MP
template <int PF, int PT, class T, int MP, bool RUN>
__device__ __forceinline__ void list_sum_shared(const ListTerm& t, const ListIn<T, PF, RUN>& src, const vi4 meta,
                                                uint32_t bin, int c, int R, unsigned char* lds, T (&acc)[PT]) {
  constexpr int N = PF * PT, PB = piece_bytes<T, N>(), NP = N * 8 / PB;
  using Piece = typename PieceOf<PB>::type;
#pragma unroll
  for (int i = 0; i < PT; ++i) acc[i] = T(0);
  const uint32_t nu = meta.y & 0xffff, na = static_cast<uint32_t>(meta.y) >> 16;
  const uint32_t lo = t.lu == LU_L ? nu : 0, hi = t.lu == LU_U ? nu : na;
  const uint32_t Mst = __umul24(meta.z, t.ns), Tin = t.Tin;
  uint32_t i = (meta.x + lo) * 8;
  const uint32_t end = (meta.x + hi) * 8;
  Piece m[MP];
  T x[PF];
  auto fetch = [&](const vi2 en) {
#pragma unroll
    for (int u = 0; u < MP; ++u)
      if (c + u * R < NP) m[u] = src.template piece<N, Piece>(Mst + en.y, c + u * R);
    src.values(__umul24(en.x, Tin) + bin, x);
  };
  bool on = i < end;
  vi2 next = {0, 0};
  if (on) {
    const vi2 en = gl<vi2>(t.ent, i);
    if (i + 8 < end) next = gl<vi2>(t.ent, i + 8);
    fetch(en);
  }
  while (__any(on)) {
    wave_lds_fence();  // the last block's reads are done
    if (on) {
#pragma unroll
      for (int u = 0; u < MP; ++u)
        if (c + u * R < NP) reinterpret_cast<Piece*>(lds)[c + u * R] = m[u];
    }
    wave_lds_fence();
    T xc[PF];
#pragma unroll
    for (int k = 0; k < PF; ++k) xc[k] = x[k];
    const bool was = on;
    i += 8;
    on = i < end;
    if (on) {
      const vi2 en = next;
      if (i + 8 < end) next = gl<vi2>(t.ent, i + 8);
      fetch(en);
    }
    if (was) {
      const T* w = reinterpret_cast<const T*>(lds);
#pragma unroll
      for (int q = 0; q < PT; ++q)
#pragma unroll
        for (int k = 0; k < PF; ++k) ListIn<T, PF, RUN>::template madd_lds<N>(acc[q], xc[k], w, k * PT + q);
    }
  }
}

// Pieces of a block a lane fetches when R lanes share it (0: not shared: few
// lanes, or more than a wavefront).
template <class T, int N>
inline int shared_pieces(int R) {
  const int np = N * 8 / piece_bytes<T, N>();
  if (R > kWave) return 0;
  const int mp = (np + R - 1) / R;
  return 2 * mp <= np ? (mp <= 1 ? 1 : (mp <= 2 ? 2 : 0)) : 0;
}

// Term t for rest index c of element e, to out (the element's values).  MP > 0:
// table blocks shared by the R lanes of a target; live lanes only otherwise.
template <int PF, int PT, class T, int NB, int MP, bool RUN, class O>
__device__ __forceinline__ void list_item_run(const ListTerm& t, const double* u, int64_t E, uint32_t e, uint32_t c,
                                              bool live, int R, unsigned char* lds, double coef, O* out) {
  const ListIn<T, PF, RUN> src(t, u, E);
  vi4 meta = {0, 0, 0, 0};
  if (MP == 0 || live) meta = gl<vi4>(t.meta, e * 16);
  const vi2 o = gl<vi2>(t.rofs, c * 8);
  T acc[PT];
  if constexpr (MP > 0) list_sum_shared<PF, PT, T, MP, RUN>(t, src, meta, o.x, c, R, lds, acc);
  else list_sum<PF, PT, T, NB, RUN>(t, src, meta, o.x, acc);
  if (MP > 0 && !live) return;
  const T cf = T(t.coef_inst ? gl<double>(t.coef_inst, meta.w * 8) : coef);
  const int sod = t.sod;
#pragma unroll
  for (int i = 0; i < PT; ++i) out[o.y + i * sod] = O(acc[i] * cf);
}
template <int PF, int PT, class T, int NB, int MP, class O>
__device__ __forceinline__ void list_item(const ListTerm& t, const double* u, int64_t E, uint32_t e, uint32_t c,
                                          bool live, int R, unsigned char* lds, double coef, O* out) {
  if (t.sdd == 1) list_item_run<PF, PT, T, NB, MP, true>(t, u, E, e, c, live, R, lds, coef, out);
  else list_item_run<PF, PT, T, NB, MP, false>(t, u, E, e, c, live, R, lds, coef, out);
}

// Sweeps of one phase: thread per (element, rest index), a row of blocks per
// term; with shared table blocks whole targets per wavefront (TW of them).
template <int PF, int PT, class T, int NB, int MP>
__global__ __launch_bounds__(kBlock) void k_list_phase(const ListTerm* terms, uint32_t E, uint32_t R, uint32_t TW,
                                                       const double* u) {
  const ListTerm& t = terms[blockIdx.y];
  if constexpr (MP == 0) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    const uint32_t e = i / R, c = i - e * R;
    if (e >= E) return;
    list_item<PF, PT, T, NB, 0>(t, u, E, e, c, true, R, nullptr, t.coef,
                                static_cast<T*>(t.out) + static_cast<int64_t>(e) * t.Tout);
  } else {
    extern __shared__ __align__(16) unsigned char smem[];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const uint32_t tl = lane / R, c = lane - tl * R;
    const uint32_t e = (blockIdx.x * (kBlock / kWave) + wave) * TW + tl;
    const bool live = tl < TW && e < E;
    list_item<PF, PT, T, NB, MP>(t, u, E, e, c, live, R, smem + (wave * TW + min(tl, TW - 1)) * (PF * PT * 8), t.coef,
                                 static_cast<T*>(t.out) + static_cast<int64_t>(e) * t.Tout);
  }
}

// Last sweep of every eval_up partial sum, added in order into the point
// value, and the point flux.  A block holds EB elements; each of its
// wavefronts takes every W-th term for all of them.
template <int PF, int PT, class T, int NB>
__global__ __launch_bounds__(NB == 4 ? 1024 : 512) void k_list_up_final(const ListTerm* terms, int nterm, int EB, int nch, int64_t E,
                                                        int P, const double* u, T* up, T* fp, const double* vcoef,
                                                        int kind, double s, int ncomp) {
  extern __shared__ double vals[];  // [nterm][EB][P]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), W = blockDim.x / kWave;
  const int lane = threadIdx.x % kWave;
  const int64_t e0 = static_cast<int64_t>(xcd_block()) * EB;
  const int ne = static_cast<int>(min(static_cast<int64_t>(EB), E - e0));
  for (int t = wave; t < nterm; t += W) {
    for (int it = lane; it < ne * nch; it += kWave) {
      const int el = it / nch, c = it - el * nch;
      list_item<PF, PT, T, NB, 0>(terms[t], u, E, static_cast<uint32_t>(e0) + el, c, true, nch, nullptr, terms[t].coef,
                                  vals + (t * EB + el) * P);
    }
  }
  __syncthreads();
  const int64_t n = E * P;
  for (int o = threadIdx.x; o < ne * P; o += blockDim.x) {
    double v = 0.;
    for (int j = 0; j < nterm; ++j) v += vals[j * EB * P + o];
    const int64_t gid = e0 * P + o;
    const T uu = T(v);
    up[gid] = uu;
    flux_point<T>(kind, uu, s, vcoef, fp, gid, n, ncomp);
  }
}

// Last sweep of every right-hand-side partial sum and the penalty sweeps,
// added in order, then the RK stage update.  Blocks as above.
template <int PFM, int PFK, class T, int NB>
__global__ __launch_bounds__(NB == 4 ? 1024 : 512) void k_list_rhs_final(const ListTerm* terms, int nterm, int npen, int EB, int nch,
                                                        int64_t E, int K, ListRhs a) {
  extern __shared__ double vals[];  // [nterm + npen][EB][K]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), W = blockDim.x / kWave;
  const int lane = threadIdx.x % kWave;
  const int64_t e0 = static_cast<int64_t>(xcd_block()) * EB;
  const int ne = static_cast<int>(min(static_cast<int64_t>(EB), E - e0));
  for (int t = wave; t < nterm + npen; t += W) {
    for (int it = lane; it < ne * nch; it += kWave) {
      const int el = it / nch, c = it - el * nch;
      double* out = vals + (t * EB + el) * K;
      const uint32_t e = static_cast<uint32_t>(e0) + el;
      if (t < nterm) list_item<PFM, PFK, T, NB, 0>(terms[t], a.u, E, e, c, true, nch, nullptr, terms[t].coef, out);
      else list_item<PFK, PFK, double, NB, 0>(terms[t], a.u, E, e, c, true, nch, nullptr, a.coef[t - nterm], out);
    }
  }
  __syncthreads();
  const int4* meta = terms[0].meta;
  for (int o = threadIdx.x; o < ne * K; o += blockDim.x) {
    const int64_t gid = e0 * K + o;
    double r = a.add ? a.rhs[gid] : 0.;
    for (int j = 0; j < nterm + npen; ++j) r += vals[j * EB * K + o];
    a.rhs[gid] = r;
    if (!a.u_next) continue;
    const double dte = a.dtv ? a.dtv[meta[e0 + o / K].w] : a.dt;
    const double t = a.tn[gid];
    if (a.tn_store) a.tn_store[gid] = t;
    const double un = rk_combine(a.scheme, a.stage, dte, t, a.u[gid], r);
    a.u_next[gid] = un;
    if (!isfinite(un)) atomicOr(a.err, ERR_NONFINITE);
  }
}

// Elements and wavefronts of a block of a final kernel with nt terms of nch
// chunks and `outs` outputs per element: one wavefront's lanes full of
// (element, chunk) pairs when the term values fit in 64 KB of LDS.
struct FinalShape { int eb, waves; };
inline FinalShape final_shape(int nt, int nch, int outs, int64_t E) {
  const int fit = kFinalValues / (nt * outs);
  if (fit < 1) throw std::runtime_error("final kernel: block too large");
  int eb = std::max(1, std::min(kWave / std::min(nch, kWave), fit));
  eb = static_cast<int>(std::min<int64_t>(eb, std::max<int64_t>(E, 1)));
  // up to eight wavefronts with equally many terms each (27 terms of three
  // dimensions on 7, 10 of two on 5: 1740 and 795 us on eight, 1655 and 772 so;
  // ten wavefronts leave a compute unit fewer blocks: 1883 and 833); sixteen on
  // small grids, whose time is the terms in turn of the block with the longest
  // lists (4D, 68 terms: 407 us with eight, 171 with sixteen)
  const int most = E <= kFewElements ? 16 : 8;
  const int rounds = (nt + most - 1) / most;
  return {eb, (nt + rounds - 1) / rounds};
}

template <int PF, int PT, class T>
void phase_t(const ListTerm* terms, int ntask, int64_t E, int R, const double* u, hipStream_t s) {
  const dim3 block(kBlock);
  const uint32_t e = static_cast<uint32_t>(E), r = static_cast<uint32_t>(R);
  // (small grids wait for latency, not for the vector memory unit: 4D, 10,496
  // elements: 171 us plain, 179 shared)
  const int mp = E <= kFewElements ? 0 : shared_pieces<T, PF * PT>(R);
  if (mp > 0) {
    const uint32_t TW = kWave / R;
    const int per = TW * (kBlock / kWave);
    const dim3 grid(static_cast<unsigned>((E + per - 1) / per), ntask);
    const size_t lds = static_cast<size_t>(per) * PF * PT * 8;
    if (mp == 1) hipLaunchKernelGGL((k_list_phase<PF, PT, T, 1, 1>), grid, block, lds, s, terms, e, r, TW, u);
    else hipLaunchKernelGGL((k_list_phase<PF, PT, T, 1, 2>), grid, block, lds, s, terms, e, r, TW, u);
    return;
  }
  const dim3 grid(nblocks(E * R), ntask);
  if (E <= kFewElements) hipLaunchKernelGGL((k_list_phase<PF, PT, T, 4, 0>), grid, block, 0, s, terms, e, r, 0u, u);
  else hipLaunchKernelGGL((k_list_phase<PF, PT, T, 2, 0>), grid, block, 0, s, terms, e, r, 0u, u);
}

template <int PF, int PT, class T>
void up_final_t(const ListTerm* terms, int nterm, int64_t E, int P, const double* u, T* up, T* fp, const double* vcoef,
                int kind, double fs, int ncomp, hipStream_t s) {
  const int R = P / PT;
  const FinalShape f = final_shape(nterm, R, P, E);
  const dim3 grid(static_cast<unsigned>((E + f.eb - 1) / f.eb)), block(f.waves * kWave);
  const size_t lds = sizeof(double) * nterm * f.eb * P;
  if (E <= kFewElements)
    hipLaunchKernelGGL((k_list_up_final<PF, PT, T, 4>), grid, block, lds, s, terms, nterm, f.eb, R, E, P, u, up, fp,
                       vcoef, kind, fs, ncomp);
  else
    hipLaunchKernelGGL((k_list_up_final<PF, PT, T, 2>), grid, block, lds, s, terms, nterm, f.eb, R, E, P, u, up, fp,
                       vcoef, kind, fs, ncomp);
}

template <int PFM, int PFK, class T>
void rhs_final_t(const ListTerm* terms, int nterm, int npen, int64_t E, int K, const ListRhs& r, hipStream_t s) {
  const int R = K / PFK;
  const FinalShape f = final_shape(nterm + npen, R, K, E);
  const dim3 grid(static_cast<unsigned>((E + f.eb - 1) / f.eb)), block(f.waves * kWave);
  const size_t lds = sizeof(double) * (nterm + npen) * f.eb * K;
  if (E <= kFewElements)
    hipLaunchKernelGGL((k_list_rhs_final<PFM, PFK, T, 4>), grid, block, lds, s, terms, nterm, npen, f.eb, R, E, K, r);
  else
    hipLaunchKernelGGL((k_list_rhs_final<PFM, PFK, T, 2>), grid, block, lds, s, terms, nterm, npen, f.eb, R, E, K, r);
}

}  // namespace

void list_nonzero(uint32_t* nz, const double* M, int ns, int block, bool in_support, bool clear, hipStream_t s) {
  const int64_t n = static_cast<int64_t>(ns) * ns;
  const int nw = (ns + 31) / 32;
  if (clear) hipLaunchKernelGGL(k_list_clear, dim3(nblocks(int64_t{ns} * nw)), dim3(kBlock), 0, s, nz, int64_t{ns} * nw);
  hipLaunchKernelGGL(k_list_nz, dim3(nblocks(n)), dim3(kBlock), 0, s, nz, M, ns, nw, block, in_support ? 1 : 0);
}

void list_fill_totals(int32_t* total, int n, hipStream_t s) {
  hipLaunchKernelGGL(k_list_zero, dim3(1), dim3(kWave), 0, s, total, n);
}

void list_build(const ListBuildArgs& a, int kind0, int nkind, int lmax, hipStream_t s) {
  if (a.E == 0) return;
  // more threads a target where fibers are long, or where the grid is small and
  // a thread's chain of loads is the launch's time
  if (lmax <= 7 && a.E > kFewElements)
    hipLaunchKernelGGL(k_list_build<2>, dim3(nblocks(a.E * 2), a.D), dim3(kBlock), 0, s, a, kind0, nkind);
  else if (lmax <= 8)
    hipLaunchKernelGGL(k_list_build<4>, dim3(nblocks(a.E * 4), a.D), dim3(kBlock), 0, s, a, kind0, nkind);
  else
    hipLaunchKernelGGL(k_list_build<8>, dim3(nblocks(a.E * 8), a.D), dim3(kBlock), 0, s, a, kind0, nkind);
}

template <class T>
void list_phase(int pf1, int pt1, const ListTerm* terms, int ntask, int64_t E, int R, const double* u,
                hipStream_t s) {
#define ADG_LP(F, P) if (pf1 == F && pt1 == P) { phase_t<F, P, T>(terms, ntask, E, R, u, s); return; }
  ADG_LP(2, 2) ADG_LP(2, 3) ADG_LP(2, 4) ADG_LP(2, 5) ADG_LP(3, 2) ADG_LP(3, 3) ADG_LP(3, 4) ADG_LP(3, 5)
  ADG_LP(4, 2) ADG_LP(4, 3) ADG_LP(4, 4) ADG_LP(4, 5) ADG_LP(5, 2) ADG_LP(5, 3) ADG_LP(5, 4)
#undef ADG_LP
  throw std::runtime_error("list phase: unsupported basis sizes");
}

template <class T>
void list_up_final(int k1, int m1, const ListTerm* terms, int nterm, int64_t E, int P, const double* u, T* up,
                   T* fp, const double* vcoef, int kind, double fs, int ncomp, hipStream_t s) {
#define ADG_LU(F, Q)                                                                          \
  if (k1 == F && m1 == Q) {                                                                   \
    up_final_t<F, Q, T>(terms, nterm, E, P, u, up, fp, vcoef, kind, fs, ncomp, s);        \
    return;                                                                                   \
  }
  ADG_LU(2, 2) ADG_LU(2, 3) ADG_LU(2, 4) ADG_LU(2, 5) ADG_LU(3, 2) ADG_LU(3, 3) ADG_LU(3, 4) ADG_LU(3, 5)
  ADG_LU(4, 2) ADG_LU(4, 3) ADG_LU(4, 4) ADG_LU(4, 5)
#undef ADG_LU
  throw std::runtime_error("list up final: unsupported basis sizes");
}

template <class T>
void list_rhs_final(int m1, int k1, const ListTerm* terms, int nterm, int npen, int64_t E, int K, const ListRhs& r,
                    hipStream_t s) {
#define ADG_LR(F, Q)                                                \
  if (m1 == F && k1 == Q) {                                         \
    rhs_final_t<F, Q, T>(terms, nterm, npen, E, K, r, s);           \
    return;                                                         \
  }
  ADG_LR(2, 2) ADG_LR(2, 3) ADG_LR(2, 4) ADG_LR(3, 2) ADG_LR(3, 3) ADG_LR(3, 4) ADG_LR(4, 2) ADG_LR(4, 3)
  ADG_LR(4, 4) ADG_LR(5, 2) ADG_LR(5, 3) ADG_LR(5, 4)
#undef ADG_LR
  throw std::runtime_error("list rhs final: unsupported basis sizes");
}

#define ADG_LIST_INST(T)                                                                                              \
  template void list_phase<T>(int, int, const ListTerm*, int, int64_t, int, const double*, hipStream_t);              \
  template void list_up_final<T>(int, int, const ListTerm*, int, int64_t, int, const double*, T*, T*,            \
                                 const double*, int, double, int, hipStream_t);                                       \
  template void list_rhs_final<T>(int, int, const ListTerm*, int, int, int64_t, int, const ListRhs&, hipStream_t);
ADG_LIST_INST(double)
ADG_LIST_INST(float)

}  // namespace adg
