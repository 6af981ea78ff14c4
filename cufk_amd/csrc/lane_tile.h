// Rows between HBM and a wave's registers through a wave-private LDS tile.
//
// A wave owns a window of 64 N consecutive elements of a row, lane t the run [tN, tN + N).  HBM
// wants the window as 16-byte vectors, vector v in lane v % 64 (coalesced); the scan wants each
// lane's run in its own registers.  The tile turns one form into the other: vectors are written
// in one order and read in the other, all as 16-byte (8-byte) LDS accesses at constant offsets
// from one address per lane, so moving a row costs next to no VALU.  Only the wave itself touches
// its tile, LDS serves a wave's accesses in order, and so no barrier and no wait is needed between
// one row's reads and the next row's writes: one tile serves all rows of the wave in turn, and
// the rows live in registers (512 KB per CU) instead of LDS (160 KB per CU).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "chain_ops.h"
#include "staging.h"

namespace cufk_amd {

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4a8 __attribute__((ext_vector_type(4), aligned(8)));
typedef unsigned int u32x4a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned int u32x4a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef unsigned int u32x2a4 __attribute__((ext_vector_type(2), aligned(4)));
typedef unsigned int u32x2a2 __attribute__((ext_vector_type(2), aligned(2)));

// A vector of Bytes bytes, and the same at the alignment of a row of Elem-byte elements.
template <int Bytes, int Elem> struct TileVec;
template <> struct TileVec<16, 8> { typedef u32x4 Local; typedef u32x4a8 Global; };
template <> struct TileVec<16, 4> { typedef u32x4 Local; typedef u32x4a4 Global; };
template <> struct TileVec<16, 2> { typedef u32x4 Local; typedef u32x4a2 Global; };
template <> struct TileVec<8, 4> { typedef u32x2 Local; typedef u32x2a4 Global; };
template <> struct TileVec<8, 2> { typedef u32x2 Local; typedef u32x2a2 Global; };
// Runs of N elements of T per lane.  Vectors are 16 bytes, or 8 where a run is no multiple of 16
// (half types, N = 4 or 12).  A run's first vector sits at kStride vectors per lane, kStride odd:
// 16 lanes reading one 16-byte vector each (32 reading 8 bytes) then cover all 64 banks once.
template <typename T, int N> struct LaneTile {
  static constexpr int kBytes = N * static_cast<int>(sizeof(T));
  static constexpr int kVecBytes = kBytes % 16 == 0 ? 16 : 8;
  static_assert(kBytes % kVecBytes == 0, "a lane's run is whole vectors");
  static constexpr int E = kVecBytes / static_cast<int>(sizeof(T));  // elements per vector
  static constexpr int NV = kBytes / kVecBytes;                     // vectors per run
  static constexpr int kStride = NV | 1;
  using Vec = typename TileVec<kVecBytes, sizeof(T)>::Local;
  using GVec = typename TileVec<kVecBytes, sizeof(T)>::Global;
  static constexpr int tile_bytes(int lanes) { return lanes * kStride * kVecBytes; }

  // Where vector v of the window lies in the tile.
  __device__ __forceinline__ static int slot(int v) { return (NV & 1) ? v : v + v / NV; }
};

// Keeps the three values in registers here: nothing computed from them moves above, and what they
// are computed from need not live on below.
template <typename R> __device__ __forceinline__ void hold(R& a, R& b, R& c) {
  asm volatile("" : "+v"(a), "+v"(b), "+v"(c));
}

// The elements of E-element vector v as the compute type.
template <typename T, typename Vec> __device__ __forceinline__ compute_t<T> vec_element(const Vec& v, int e) {
  struct Elems {
    T x[sizeof(Vec) / sizeof(T)];
  };
  return widen(__builtin_bit_cast(Elems, v).x[e]);
}

// A lane's K points (coordinate c of point i in P[c][i]) as the vectors of its run of a (points, 3)
// row, rounded to T.
template <typename T, int K, typename R, typename Vec, int NV>
__device__ __forceinline__ void pack_points(const R (&P)[3][K], Vec (&run)[NV]) {
  constexpr int E = sizeof(Vec) / sizeof(T);
  static_assert(E * NV == 3 * K, "the run holds the lane's points");
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    struct Elems {
      T x[E];
    } el;
#pragma unroll
    for (int e = 0; e < E; ++e) el.x[e] = narrow<T>(P[(E * j + e) % 3][(E * j + e) / 3]);
    run[j] = __builtin_bit_cast(Vec, el);
  }
}

// A lane's N values as the vectors of its run of a row, rounded to T.
template <typename T, typename R, int N, typename Vec, int NV>
__device__ __forceinline__ void pack_run(const R (&v)[N], Vec (&run)[NV]) {
  constexpr int E = sizeof(Vec) / sizeof(T);
  static_assert(E * NV == N, "the run holds the lane's values");
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    struct Elems {
      T x[E];
    } el;
#pragma unroll
    for (int e = 0; e < E; ++e) el.x[e] = narrow<T>(v[E * j + e]);
    run[j] = __builtin_bit_cast(Vec, el);
  }
}

// A window of one row on its way from HBM to the lanes' runs: elements [start, end) of the row (end
// - start may be 64 runs and more, or <= 0).  fetch() issues the loads, to_runs() hands every lane its
// run.  Every lane issues every load, those past the row's end at its last whole vector instead: with
// no branch around them, what is loaded before the rows need not wait for the rows (with an exec mask
// around each load the compiler waits for all of them at once: at B = 4096, N = 2049, whose last wave
// is not full, the forward took 55 us against 48 us at N = 2051).  The vector that `end` cuts comes
// element by element from the low lanes, so no access leaves the row: with Whole the row's `elements`
// are E or more, without it fewer than E.  Stream: nontemporal loads, for rows whose step reads other
// rows from the last-level cache.
template <typename T, typename Tile> struct WindowLoad {
  static constexpr int E = Tile::E, NV = Tile::NV;
  using Vec = typename Tile::Vec;
  struct Elems {
    T x[E];
  };
  Vec vec[NV];
  T tail;  // this lane's element of the cut vector

  template <bool Whole, bool Stream>
  __device__ __forceinline__ void fetch(const T* __restrict__ row, int start, int end, int elements, int lane) {
    if constexpr (Whole) {
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const unsigned at = min(start + (lane + 64 * j) * E, elements - E);
        const auto* const g = reinterpret_cast<const typename Tile::GVec*>(row + at);
        if constexpr (Stream)
          vec[j] = __builtin_nontemporal_load(g);
        else
          vec[j] = *g;
      }
    } else {
#pragma unroll
      for (int j = 0; j < NV; ++j) vec[j] = Vec{};
    }
    const unsigned at = min(start + max(end - start, 0) / E * E + lane, end - 1);
    tail = row[at];
  }

  // n = end - start; elements past them are `pad`.  `full` (uniform): n holds 64 whole runs.
  __device__ __forceinline__ void to_runs(void* tile, Vec (&run)[NV], int n, bool full, T pad, int lane) const {
    Vec* const t = static_cast<Vec*>(tile);
    wave_lds_order();
    if (full) {
#pragma unroll
      for (int j = 0; j < NV; ++j) t[Tile::slot(lane + 64 * j)] = vec[j];
    } else {
      Elems el;
#pragma unroll
      for (int e = 0; e < E; ++e) el.x[e] = pad;
      const Vec none = __builtin_bit_cast(Vec, el);
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const int v = lane + 64 * j;
        const bool in = (v + 1) * E <= n;
        Vec x;
#pragma unroll
        for (int k = 0; k < static_cast<int>(sizeof(Vec) / 4); ++k) x[k] = in ? vec[j][k] : none[k];
        t[Tile::slot(v)] = x;
      }
      wave_lds_order();
      const int cut = max(n, 0) / E;
      if (lane < n - cut * E) static_cast<T*>(tile)[Tile::slot(cut) * E + lane] = tail;
    }
    wave_lds_order();
#pragma unroll
    for (int j = 0; j < NV; ++j) run[j] = t[lane * Tile::kStride + j];
    wave_lds_order();
  }
};

// A wave's lane runs to dst[0, n): the runs of Part lanes at a time go through the tile (Part = 32
// halves the tile of a long run) and leave as contiguous vectors, the elements past the last whole
// one from the low lanes.
template <typename Tile, int Part, bool Stream, typename T>
__device__ __forceinline__ void store_window(T* __restrict__ dst, void* tile, const typename Tile::Vec (&run)[Tile::NV],
                                             int n, bool full, int lane) {
  constexpr int E = Tile::E, NV = Tile::NV;
  using Vec = typename Tile::Vec;
  using GVec = typename Tile::GVec;
  Vec* const t = static_cast<Vec*>(tile);
  constexpr int kVecs = Part * NV;  // vectors per part
  constexpr int kPer = (kVecs + 63) / 64;
#pragma unroll
  for (int p = 0; p < 64 / Part; ++p) {
    wave_lds_order();
    if (Part == 64 || lane / Part == p) {
#pragma unroll
      for (int j = 0; j < NV; ++j) t[(lane % Part) * Tile::kStride + j] = run[j];
    }
    wave_lds_order();
    T* const d = dst + p * kVecs * E;
    const int left = n - p * kVecs * E;
    const int whole = full ? kVecs : max(min(left / E, kVecs), 0);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int v = lane + 64 * j;
      if (64 * (j + 1) <= kVecs ? full || v < whole : v < whole) {
        GVec* const g = reinterpret_cast<GVec*>(d + E * v);
        const GVec x = t[Tile::slot(v)];
        if constexpr (Stream)
          __builtin_nontemporal_store(x, g);
        else
          *g = x;
      }
    }
    if (!full && whole < kVecs && lane < left - E * whole) {
      const T* const e = reinterpret_cast<const T*>(t + Tile::slot(whole)) + lane;
      global_store<Stream>(d + E * whole + lane, *e);
    }
  }
}

}  // namespace cufk_amd
