// Position-based-fluids substep kernels for gfx950.
//
// Particles live in two orders.  The canonical state (x_can, v_can) is in
// particle-id order, like the reference's arrays.  After the neighbour search
// the substep works on copies reordered into (cell key, id) order, so that a
// particle's 27-cell neighbourhood is nine contiguous index ranges and the
// neighbour gathers of one wavefront hit the same cache lines.  The commit
// kernel scatters x* and v back to id order at the end of the substep.
//
// Vector fields are float4.  pos.w carries lambda between the density/lambda
// pass and the delta-p pass, and rho afterwards; aux.w carries |omega|.
//
// Neighbour lists are stored per 64-particle group in 16-byte quads: lane
// s%64's quad q is at word (s/64)*64*60 + q*256 + (s%64)*4, so a wave's load
// of one quad per lane covers 1 KB contiguously.  In (dz, dy, dx, id) order a
// particle's neighbours have strictly increasing sorted indices, and those of
// one dz layer lie within a few grid rows of the layer's first candidate, so
// a compact list stores 16-bit offsets from the three layer bases held in the
// particle's list head (8 neighbours per quad); a wide list stores the 32-bit
// indices (4 per quad).
#include <type_traits>

#include "sph_internal.h"
#include "sph_mlp_dev.h"

namespace sph {

// Logical block index for a launch of nb blocks so that each XCD (blocks are
// dispatched round-robin over 8 XCDs) walks one contiguous range of particles
// and keeps its neighbourhood in its own L2.
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t nb) {
  const uint32_t q = nb >> 3, r = nb & 7u;
  const uint32_t x = b & 7u, idx = b >> 3;
  return x * q + min(x, r) + idx;
}

__device__ __forceinline__ uint32_t particle_index(uint32_t n_blocks) {
  return xcd_block(blockIdx.x, n_blocks) * blockDim.x + threadIdx.x;
}

// Depth of the gather kernels that give a particle four lanes (sum_neighbors).
constexpr int kQuad = 4;

// The particle of a gather kernel's lane, and whether the lane stores its results.
template <int NB>
__device__ __forceinline__ uint32_t gather_index(uint32_t n_blocks) {
  return NB == kQuad ? particle_index(n_blocks) >> 2 : particle_index(n_blocks);
}

template <int NB>
__device__ __forceinline__ bool gather_lead() {
  return NB != kQuad || (threadIdx.x & 3u) == 0u;
}

__device__ __forceinline__ const uint32_t *list_ptr(const uint32_t *list, uint32_t s) {
  return list + (size_t)(s >> 6) * kListStride + (s & 63u) * 4u;
}

// One particle's list: its first quad, its head and the wave's format.
struct NbList {
  const uint32_t *L;
  uint4 h;      // layer bases (x, y, z) and counts (w)
  int c;        // neighbours
  int e0, e1;   // neighbours in layer 0, in layers 0 and 1
  bool wide;    // uniform over the wavefront
};

__device__ __forceinline__ NbList nb_list(const uint32_t *list, const uint4 *head, uint32_t s) {
  NbList r;
  r.L = list_ptr(list, s);
  r.h = head[s];
  r.c = (int)(r.h.w & kHeadCount);
  r.e0 = (int)((r.h.w >> 8) & kHeadCount);
  r.e1 = (int)((r.h.w >> 16) & kHeadCount);
  // every lane of a wavefront holds the same format bit
  r.wide = (__builtin_amdgcn_readfirstlane(r.h.w) & kHeadWide) != 0u;
  return r;
}

// Launch bounds of the delta-p, density, colour and confinement kernels: at
// up to 16 gathers in flight at most 128 VGPRs, i.e. 4 waves per SIMD, which density
// and delta p meet without spilling, colour and confinement with 15 spilled (at 3 waves delta p measured 7% slower, colour
// and confinement 2-3%).  Five waves (96 VGPRs) would spill 164-220 bytes.
#define GATHER_BOUNDS(NB) __launch_bounds__(kBlock, (NB) <= 16 ? 4 : 1)

// Visits the c neighbours of a particle in list order, NB at a time: the
// batch's list quads (raw, as stored), their decoding to indices, the NB gathers
// in one burst, then the arithmetic.  NB gathers in flight per wave: 16 was
// 13-22% faster than 8 in every gather pass on MI355X; the autotuner chooses 8,
// 16 or 32 per kernel.
//
// What bounds it: the vector L1's return path is 93-96% busy in every pass.  A
// gather of 16-byte records costs it 1, 1.5 or 2.3 cycles per four lanes whose
// records lie in 1, 2 or 4 cache lines (16, 24, 38 cycles per wave, measured on a
// resident window), and here four neighbouring lanes touch three lines on
// average, 31 cycles; the 16-byte passes are at the same time 80-90% VALU-busy.
//
// The first batch's quads are loaded together with the particle and its head
// (their place does not depend on it), which takes one memory round trip off
// every pass.  With kRaw the quads of batch k+1 are issued right after the
// gathers of batch k and stay raw until their batch: 8 registers, where decoded
// indices took 16 and spilled (20 bytes in delta p), and a last half batch
// decodes only its own half.  Decoding in a block of its own, before the first
// gather issues, keeps the gathers together: interleaved with it, the surface
// pass took 643 us against 551 and every other pass 1-7% more.  Measured at 8.4M
// particles against decoded prefetch (kIndices): density+lambda 358 -> 323 us, delta p
// 317 -> 303, surface 562 -> 551, vorticity within 1%.  Colour, confinement and XSPH at
// 16 gathers, whose arithmetic is shortest, decode the next batch beside it (kIndices):
// 309, 336 and 500 us against 317, 343 and 504 with raw quads (XSPH: without a
// prefetch, as with raw quads it is slower still), and 397, 476 and 712 against 414,
// 490 and 729 where lists are longer (33 on average for 28).  The same made surface
// 630 us for 499 and vorticity 561 for 530.
// Slots past c are never used; their gathers load a valid index (the particle
// itself in a wide list, the layer-2 base in a compact one, which the build sets
// to the particle itself when that layer has no candidates), which costs less
// than it seems: an index past the records instead, which touches no line, made
// no pass faster.
constexpr uint32_t kQuadStride = kWave * 4;  // list words between a lane's quads
// Hits the list build buffers in LDS per thread (16 bits each) for the
// coalesced write-out; later hits of a compact list are stored directly.  At
// 40 a 256-thread block holds 20 KB, so LDS admits 7 waves per SIMD, which the
// kernel's launch bound (70 VGPRs, no spill) also fits: measured at 8M
// particles 0.855 -> 0.842 ms against 48 slots at 6 waves (60 slots, 30 KB,
// admitted 5).
constexpr int kLdsHits = 40;
static_assert(kLdsHits % 8 == 0 && kLdsHits <= kMaxNb, "whole quads in LDS");

// Entry e of a lane's compact list (16-bit offset v), stored on its own: quad
// e / 8 (kQuadStride words apart), 32-bit word (e % 8) / 2, low half first.
__device__ __forceinline__ void store_entry16(uint32_t *out, int e, uint32_t v) {
  uint16_t *w = reinterpret_cast<uint16_t *>(out + (size_t)(e >> 3) * kQuadStride + ((e & 7) >> 1));
  w[e & 1] = (uint16_t)v;
}

// Raw quads of the NB entries from k0 on; those past the last quad stay as they
// were (decode does not use them).
template <int NB, bool WIDE>
struct Quads {
  static constexpr int kPer = WIDE ? 4 : 8, kCount = NB / kPer;
  uint4 q[kCount];
  __device__ __forceinline__ void load(const NbList &nl, int k0) {
    const uint4 *Q = reinterpret_cast<const uint4 *>(nl.L) + (size_t)(k0 / kPer) * kWave;
#pragma unroll
    for (int u = 0; u < kCount; ++u)
      if (k0 + kPer * u < nl.c) q[u] = Q[(size_t)u * kWave];
  }
};

// Sorted indices of entries [k0, k0 + M) from their quads.  Wide: as stored, the
// particle itself past c.  Compact: base of the entry's layer + 16-bit offset;
// past the last quad, offset 0 from the layer-2 base.
template <int M, int NB, bool WIDE>
__device__ __forceinline__ void decode(const NbList &nl, const Quads<NB, WIDE> &r, int k0,
                                       uint32_t self, uint32_t (&j)[M]) {
  // values, not member lvalues: a select between member addresses would
  // keep the struct in memory (and the compiler moves such memory to LDS)
  const uint32_t b0 = nl.h.x, b1 = nl.h.y, b2 = nl.h.z;
  const int e0 = nl.e0, e1 = nl.e1, c = nl.c;
  if (WIDE) {
#pragma unroll
    for (int t = 0; t < M; ++t) {
      const uint4 a = r.q[t / 4];
      const uint32_t w[4] = {a.x, a.y, a.z, a.w};
      j[t] = k0 + t < c ? w[t & 3] : self;
    }
  } else {
#pragma unroll
    for (int u = 0; u < M / 8; ++u) {
      const bool in = k0 + 8 * u < c;
      const uint4 a = r.q[u];
      const uint32_t w[4] = {in ? a.x : 0u, in ? a.y : 0u, in ? a.z : 0u, in ? a.w : 0u};
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const int k = k0 + 8 * u + t;
        const uint32_t off = (t & 1) ? (w[t >> 1] >> 16) : (w[t >> 1] & 0xFFFFu);
        const uint32_t lb = k < e1 ? b1 : b2;
        j[8 * u + t] = (k < e0 ? b0 : lb) + off;
      }
    }
  }
}

// What a batch fetches of the next one's list before its arithmetic.
enum Prefetch { kNone, kRaw, kIndices };

// A wavefront runs each batch for its longest list.  Batches in which no lane's
// list ends skip the per-neighbour count test, and a last batch in which every
// lane ends within NB/2 neighbours runs only NB/2 of them (the wave's longest
// list, not the mean, sets the work: half batches cut the padding slots).
template <typename T, int NB, int PREFETCH, bool WIDE, typename Load, typename Body>
__device__ __forceinline__ void gather_loop(const NbList &nl, const uint4 *first, uint32_t self,
                                            Load &load, Body &body) {
  Quads<NB, WIDE> r;
  const int c = nl.c;
  if (WIDE) {
    r.load(nl, 0);
  } else {
#pragma unroll
    for (int u = 0; u < Quads<NB, WIDE>::kCount; ++u) r.q[u] = first[u];
  }
  uint32_t j[NB];
  if (PREFETCH == kIndices) decode<NB>(nl, r, 0, self, j);
  for (int k0 = 0; k0 < c; k0 += NB) {
    // the lanes still in the loop have c > k0
    if (PREFETCH == kNone && k0 > 0) r.load(nl, k0);
    if (NB >= 16 && __ballot(k0 + NB / 2 < c) == 0ull) {
      uint32_t h[NB / 2];
      if (PREFETCH != kIndices) {
        decode<NB / 2>(nl, r, k0, self, h);
        __builtin_amdgcn_sched_barrier(0);
      }
      T q[NB / 2];
#pragma unroll
      for (int b = 0; b < NB / 2; ++b) q[b] = load(PREFETCH == kIndices ? j[b] : h[b]);
#pragma unroll
      for (int b = 0; b < NB / 2; ++b)
        if (k0 + b < c) body(q[b]);
    } else {
      if (PREFETCH != kIndices) {
        decode<NB>(nl, r, k0, self, j);
        __builtin_amdgcn_sched_barrier(0);
      }
      T q[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) q[b] = load(j[b]);
      if (PREFETCH == kRaw) r.load(nl, k0 + NB);
      if (PREFETCH == kIndices) {
        Quads<NB, WIDE> next;  // not r, which would be held over the loop
        next.load(nl, k0 + NB);
        decode<NB>(nl, next, k0 + NB, self, j);
      }
      if (__ballot(k0 + NB > c) == 0ull) {
#pragma unroll
        for (int b = 0; b < NB; ++b) body(q[b]);
      } else {
#pragma unroll
        for (int b = 0; b < NB; ++b)
          if (k0 + b < c) body(q[b]);
      }
    }
  }
}

template <typename T, int NB, int PREFETCH, typename Load, typename Body>
__device__ __forceinline__ void for_neighbors(const uint32_t *list, const uint4 *head, uint32_t s,
                                              int *count, Load load, Body body) {
  uint4 first[NB / 8];
#pragma unroll
  for (int u = 0; u < NB / 8; ++u)
    first[u] = reinterpret_cast<const uint4 *>(list_ptr(list, s))[(size_t)u * kWave];
  const NbList nl = nb_list(list, head, s);
  *count = nl.c;
  if (nl.wide)
    gather_loop<T, NB, PREFETCH, true>(nl, first, s, load, body);
  else
    gather_loop<T, NB, PREFETCH, false>(nl, first, s, load, body);
}

struct Pair4 {
  float4 a, b;
};

// What a neighbour adds to a particle's NA sums: acc[a] = fma(w, d, acc[a]) for the
// P pairs (w, d) of each, in order.
template <int NA, int P = 1>
struct Terms {
  float w[NA * P], d[NA * P];
};

// Value of lane K of each four lanes, in all of them.
template <int K>
__device__ __forceinline__ float quad_lane(float v) {
  return __int_as_float(
      __builtin_amdgcn_mov_dpp(__float_as_int(v), K * 0x55, 0xF, 0xF, true));
}

// Sum over each four lanes, in all of them.
__device__ __forceinline__ uint32_t quad_sum(uint32_t v) {
  v += (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true);        // 1 0 3 2
  return v + (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true);  // 2 3 0 1
}

// The sums over a particle's neighbours with four lanes for each particle: lane q
// of the four gathers and evaluates entries 8 q .. 8 q + 7 of each 32, and the sums
// pass from lane to lane, so that they are the ones a single lane makes in list
// order, bit for bit.  An entry past the list adds 0 * 0.
template <typename T, int NA, int P, bool WIDE, typename Load, typename Term>
__device__ __forceinline__ void quad_loop(const NbList &nl, const uint4 &first, uint32_t self,
                                          Load &load, Term &term, float (&acc)[NA]) {
  constexpr int E = 8;  // entries per lane and round
  const int sub = threadIdx.x & 3;
  Quads<E, WIDE> r;
  if (WIDE)
    r.load(nl, E * sub);
  else
    r.q[0] = first;
  for (int base = 0; base < nl.c; base += 4 * E) {
    const int k0 = base + E * sub;
    uint32_t j[E];
    decode<E>(nl, r, k0, self, j);
    __builtin_amdgcn_sched_barrier(0);
    T q[E];
    if (k0 < nl.c) {
#pragma unroll
      for (int b = 0; b < E; ++b) q[b] = load(j[b]);
    }
    r.load(nl, k0 + 4 * E);
    Terms<NA, P> t[E];
#pragma unroll
    for (int b = 0; b < E; ++b) {
      t[b] = {};
      if (k0 + b < nl.c) t[b] = term(q[b]);
    }
    const auto pass = [&](auto lane) {
#pragma unroll
      for (int b = 0; b < E; ++b)
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
          for (int i = 0; i < P; ++i)
            acc[a] = fmaf(t[b].w[a * P + i], t[b].d[a * P + i], acc[a]);
#pragma unroll
      for (int a = 0; a < NA; ++a) acc[a] = quad_lane<decltype(lane)::value>(acc[a]);
      // whether the next lane has an entry in any particle of the wave
      return __ballot(base + E * (decltype(lane)::value + 1) < nl.c) != 0ull;
    };
    if (pass(std::integral_constant<int, 0>{}) && pass(std::integral_constant<int, 1>{}) &&
        pass(std::integral_constant<int, 2>{}))
      pass(std::integral_constant<int, 3>{});
  }
}

// acc = the sums of term(load(j)) over the neighbours j of particle s, in list
// order, with NB gathers in flight or (kQuad) four lanes a particle.
template <typename T, int NB, int PREFETCH, int NA, int P, typename Load, typename Term>
__device__ __forceinline__ void sum_neighbors(const uint32_t *list, const uint4 *head, uint32_t s,
                                              int *count, float (&acc)[NA], Load load,
                                              Term term) {
#pragma unroll
  for (int a = 0; a < NA; ++a) acc[a] = 0.0f;
  if constexpr (NB == kQuad) {
    const uint4 first =
        reinterpret_cast<const uint4 *>(list_ptr(list, s))[(size_t)(threadIdx.x & 3u) * kWave];
    const NbList nl = nb_list(list, head, s);
    *count = nl.c;
    if (nl.wide)
      quad_loop<T, NA, P, true>(nl, first, s, load, term, acc);
    else
      quad_loop<T, NA, P, false>(nl, first, s, load, term, acc);
  } else {
    for_neighbors<T, NB, PREFETCH>(list, head, s, count, load, [&](const T &q) {
      const Terms<NA, P> t = term(q);
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int i = 0; i < P; ++i) acc[a] = fmaf(t.w[a * P + i], t.d[a * P + i], acc[a]);
    });
  }
}

// Gathers of 16-byte records through a buffer resource with a 16-byte stride
// (`buffer_load ... idxen`): the texture addresser forms base + 16 j from the
// index itself, so a gather costs no VALU (a 64-bit address costs two, the
// zero high word and the shift-add) and needs no address registers.  At 16
// gathers in flight colour and confinement took 138-140 -> 130-133 VGPRs, XSPH
// at 8 gathers 112 -> 90 VGPRs (5 waves per SIMD instead of 4), and the autotuner
// picked 16 gathers in flight for XSPH and vorticity instead of 8 (measured
// at 8M particles: vorticity 0.70 -> 0.58 ms, XSPH 0.67 -> 0.60, delta p,
// colour and confinement 3% faster, density+lambda unchanged).  An index at or
// past `records` reads zeros instead of leaving the array.
typedef float sph_v4f __attribute__((ext_vector_type(4)));
__device__ sph_v4f sph_struct_load_v4f32(__amdgpu_buffer_rsrc_t rsrc, int vindex, int voffset,
                                         int soffset, int aux)
    __asm("llvm.amdgcn.struct.ptr.buffer.load.v4f32");
// Word 3 of a gfx9-family buffer descriptor: 32-bit data format, no swizzle.
constexpr int kBufferWord3 = 0x00020000;

struct Records16 {
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ Records16(const float4 *a, uint32_t records)
      : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<float4 *>(a), (short)16, (int)records,
                                            kBufferWord3)) {}
  __device__ __forceinline__ float4 operator[](uint32_t j) const {
    const sph_v4f v = sph_struct_load_v4f32(r, (int)j, 0, 0, 0);
    return make_float4(v.x, v.y, v.z, v.w);
  }
};

__device__ __forceinline__ float fast_rsq(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }

// x^2 + y^2 + z^2 with two fused multiply-adds (this file is compiled without
// implicit contraction, so every fma is written out).
__device__ __forceinline__ float sq3(float x, float y, float z) {
  return fmaf(z, z, fmaf(y, y, x * x));
}

// ApplyBoundaryConditions (particles.c:842-867).
__device__ __forceinline__ float clamp_axis(float x, float lo, float hi, float hi_clamp) {
  if (x < lo) return lo;
  if (x >= hi) return hi_clamp;
  return x;
}

// Box and hash grid of the scene a particle belongs to (the context's own for
// a single scene; the scene table's in a batch).  Boxes start at the origin.
struct Geo {
  uint32_t base, nx, ny, nz, nxy;
  float hi[3], hi_clamp[3];
};

template <bool BATCH>
__device__ __forceinline__ Geo geo_of(uint32_t i, const DevParams &P, const BatchDev &B) {
  Geo g;
  if (!BATCH) {
    g.base = 0u;
    g.nx = P.nx; g.ny = P.ny; g.nz = P.nz; g.nxy = P.nxy;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      g.hi[a] = P.box_hi[a];
      g.hi_clamp[a] = P.box_hi_clamp[a];
    }
  } else {
    const SceneDev &d = B.scenes[B.scene_of[i]];
    g.base = d.cell_base;
    g.nx = d.nx; g.ny = d.ny; g.nz = d.nz; g.nxy = d.nxy;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      g.hi[a] = d.box_hi[a];
      g.hi_clamp[a] = d.box_hi_clamp[a];
    }
  }
  return g;
}

// Obstacle of particle i's scene.
template <bool BATCH>
__device__ __forceinline__ const SdfDev &sdf_of(uint32_t i, const SdfDev &o, const BatchDev &B) {
  if (!BATCH) return o;
  return B.scenes[B.scene_of[i]].sdf;
}

__device__ __forceinline__ void apply_boundary(float &x, float &y, float &z, const Geo &g,
                                               const DevParams &P) {
  x = clamp_axis(x, P.box_lo[0], g.hi[0], g.hi_clamp[0]);
  y = clamp_axis(y, P.box_lo[1], g.hi[1], g.hi_clamp[1]);
  z = clamp_axis(z, P.box_lo[2], g.hi[2], g.hi_clamp[2]);
}

__device__ __forceinline__ void apply_boundary(float &x, float &y, float &z,
                                               const DevParams &P) {
  x = clamp_axis(x, P.box_lo[0], P.box_hi[0], P.box_hi_clamp[0]);
  y = clamp_axis(y, P.box_lo[1], P.box_hi[1], P.box_hi_clamp[1]);
  z = clamp_axis(z, P.box_lo[2], P.box_hi[2], P.box_hi_clamp[2]);
}

// Exact floor(x / h) for float x, h: a float estimate corrected with the sign
// of the exactly rounded residual fma(-k, h, x).  Equals the reference's
// floor of the double quotient (neighbors.c:86-88), which never rounds across
// an integer for float operands.
__device__ __forceinline__ uint32_t cell_coord(float x, float h, float inv_h, uint32_t dim,
                                               uint32_t *clamped) {
  float k = floorf(x * inv_h);
  if (fmaf(-k, h, x) < 0.0f)
    k -= 1.0f;
  else if (fmaf(-(k + 1.0f), h, x) >= 0.0f)
    k += 1.0f;
  if (!(k >= 0.0f)) {  // negative or NaN: keep the index inside the grid
    *clamped += 1u;
    return 0u;
  }
  if (k > (float)(dim - 1)) {
    *clamped += 1u;
    return dim - 1;
  }
  return (uint32_t)k;
}

// HashVal (neighbors.c:79-98), offset by the scene's first cell key.
__device__ __forceinline__ uint32_t hash_key(float x, float y, float z, const DevParams &P,
                                             const Geo &g, uint32_t *clamped) {
  const uint32_t gx = cell_coord(x, P.h, P.inv_h, g.nx, clamped);
  const uint32_t gy = cell_coord(y, P.h, P.inv_h, g.ny, clamped);
  const uint32_t gz = cell_coord(z, P.h, P.inv_h, g.nz, clamped);
  return g.base + (g.nxy * gz + (gy * g.nx + gx));
}

__device__ __forceinline__ void add_counter64(uint32_t *stats, int slot, uint32_t v) {
  if (v) atomicAdd(reinterpret_cast<unsigned long long *>(stats + slot), (unsigned long long)v);
}

// The same with one atomic per wavefront (its lanes' sum); every lane of the
// wave must call it.  The list build's drop count is nonzero for every
// particle at the 60-neighbour cap (tens of thousands in a late dam-break
// substep), and per-lane atomics on one word serialise.
__device__ __forceinline__ void add_counter64_wave(uint32_t *stats, int slot, uint32_t v) {
  if (__ballot(v != 0u) == 0ull) return;
  uint32_t t = v;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) t += __shfl_xor(t, o, 64);
  if ((threadIdx.x & 63) == 0)
    atomicAdd(reinterpret_cast<unsigned long long *>(stats + slot), (unsigned long long)t);
}

// Block sum of v written to partial[blockIdx.x] (no atomics; the host adds the
// partials when it reads the statistics).  All threads of the block call it.
__device__ __forceinline__ void block_sum_to(uint32_t *partial, uint32_t v) {
  __shared__ uint32_t wsum[kBlock / kWave];
  uint32_t t = v;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) t += __shfl_xor(t, o, 64);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t s = 0;
    for (uint32_t w = 0; w < blockDim.x / kWave; ++w) s += wsum[w];
    partial[blockIdx.x] = s;
  }
}

// ---------------------------------------------------------------------------
// Elementwise stages before the neighbour search
// ---------------------------------------------------------------------------
// ApplyGravity (particles.c:516-527).
__global__ __launch_bounds__(kBlock) void k_gravity(uint32_t n, float4 *__restrict__ v,
                                                    DevParams P) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  v[i].z = v[i].z + P.g_dt;
}

// PredictPositions (particles.c:748-784).
template <bool BATCH>
__global__ __launch_bounds__(kBlock) void k_predict(uint32_t n, const float4 *__restrict__ x,
                                                    const float4 *__restrict__ v,
                                                    float4 *__restrict__ xs, DevParams P,
                                                    BatchDev B) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const float4 a = x[i], u = v[i];
  float px = a.x + u.x * P.dt, py = a.y + u.y * P.dt, pz = a.z + u.z * P.dt;
  apply_boundary(px, py, pz, geo_of<BATCH>(i, P, B), P);
  xs[i] = make_float4(px, py, pz, 0.0f);
}

// Counts a particle into its cell: its place among the cell's particles in the
// order they happen to be counted.  Lanes of a run of equal keys (particles in
// id order lie along a lattice row, two to a cell) share one atomic: with an
// atomic per lane the runs serialise, 183 us at 8.4M particles against 26.
// Every lane of the wave calls it; the key of one past the end is not counted.
__device__ __forceinline__ uint32_t count_into_cell(uint32_t *__restrict__ cell_count,
                                                    uint32_t key, bool valid) {
  const int lane = threadIdx.x & 63;
  const uint32_t k = valid ? key : 0xFFFFFFFFu;
  const uint32_t left = __shfl_up(k, 1, 64);
  const bool first = lane == 0 || left != k;
  const uint64_t firsts = __ballot(first);
  const int head = 63 - __builtin_clzll(firsts & (~0ull >> (63 - lane)));
  const uint64_t after = lane == 63 ? 0ull : firsts >> (lane + 1);
  const int next = after ? lane + 1 + __builtin_ctzll(after) : 64;
  uint32_t old = 0u;
  if (first && valid) old = atomicAdd(&cell_count[k], (uint32_t)(next - lane));
  return __shfl(old, head, 64) + (uint32_t)(lane - head);
}

// Substep bookkeeping: clears the flags and the error words of iterations up to
// `last`, from the search's first kernel (nothing of it uses them).  No
// hipMemsetAsync, so that the substep can be captured in a graph.
__device__ __forceinline__ void clear_substep_stats(uint32_t *stats, uint32_t last) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= STAT_ITERS && i < STAT_ERR0) stats[i] = 0u;
  for (uint32_t e = i; e < (last + 1u) * kErrSlots; e += gridDim.x * kBlock)
    stats[err_word(0u, e)] = 0u;
}

// HashParticles (neighbors.c:101-125).
template <bool BATCH>
__global__ __launch_bounds__(kBlock) void k_hash(uint32_t n, const float4 *__restrict__ xs,
                                                 uint32_t *__restrict__ keys,
                                                 uint32_t *__restrict__ cell_rank,
                                                 uint32_t *__restrict__ cell_count, DevParams P,
                                                 uint32_t *__restrict__ stats,
                                                 uint32_t last_error, BatchDev B) {
  clear_substep_stats(stats, last_error);
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  const bool valid = i < n;
  uint32_t clamped = 0, key = 0;
  if (valid) {
    const float4 a = xs[i];
    key = hash_key(a.x, a.y, a.z, P, geo_of<BATCH>(i, P, B), &clamped);
  }
  const uint32_t rank = count_into_cell(cell_count, key, valid);
  if (!valid) return;
  keys[i] = key;
  cell_rank[i] = rank;
  add_counter64(stats, STAT_CLAMPS, clamped);
}

// Fused ApplyGravity + PredictPositions + HashParticles for the fused
// substep: v after gravity is only read by the prediction (UpdateVelocities
// overwrites it), so it is not stored.
template <bool BATCH>
__global__ __launch_bounds__(kBlock) void k_predict_hash(uint32_t n,
                                                         const float4 *__restrict__ x,
                                                         const float4 *__restrict__ v,
                                                         float4 *__restrict__ xs,
                                                         uint32_t *__restrict__ keys,
                                                         uint32_t *__restrict__ cell_rank,
                                                         uint32_t *__restrict__ cell_count,
                                                         DevParams P,
                                                         uint32_t *__restrict__ stats,
                                                         uint32_t last_error, BatchDev B) {
  clear_substep_stats(stats, last_error);
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  const bool valid = i < n;
  uint32_t clamped = 0, key = 0;
  if (valid) {
    const float4 a = x[i], u = v[i];
    const float vz = u.z + P.g_dt;
    float px = a.x + u.x * P.dt, py = a.y + u.y * P.dt, pz = a.z + vz * P.dt;
    const Geo g = geo_of<BATCH>(i, P, B);
    apply_boundary(px, py, pz, g, P);
    xs[i] = make_float4(px, py, pz, 0.0f);
    key = hash_key(px, py, pz, P, g, &clamped);
  }
  const uint32_t rank = count_into_cell(cell_count, key, valid);
  if (!valid) return;
  keys[i] = key;
  cell_rank[i] = rank;
  add_counter64(stats, STAT_CLAMPS, clamped);
}

// The stable (cell key, id) sort of the reference (thrust_c.cu:86-91) as a
// counting sort: the cells are counted while the keys are made, their exclusive
// scan is the cell table, and a particle's (id, key) goes to its cell's range
// here, in the order the counting happened to give.  k_reorder puts the cell's
// few particles into id order.  Also zeroes the counts it has used (every
// particle of a cell writes the same zero).  From the hash to the sorted
// positions, against three radix passes of five launches each: 8.4M particles
// 467 -> 319 us, 1M 138 -> 54, 4k 49 (two passes) -> 14.
__global__ __launch_bounds__(kBlock) void k_place(uint32_t n, const uint32_t *__restrict__ keys,
                                                  const uint32_t *__restrict__ cell_rank,
                                                  const uint32_t *__restrict__ cell_start,
                                                  uint2 *__restrict__ slots,
                                                  uint32_t *__restrict__ cell_count) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const uint32_t key = keys[i];
  slots[cell_start[key] + cell_rank[i]] = make_uint2(i, key);
  cell_count[key] = 0u;
}

// Each particle's place in (cell key, id) order, from the ids of its cell that
// are below its own (8 or so, read by the cell's lanes together), and x*, x,
// key and id gathered there.
// Also x* as the list build reads it, in 16-bit coordinates: x and y in one word, z
// in an array of its own.
__device__ __forceinline__ uint32_t fixed16(float x, double scale) {
  const double t = (double)x * scale;
  return x == x ? (uint32_t)(t - 65536.0 * floor(t * (1.0 / 65536.0))) & 0xFFFFu : kFixedNaN;
}

// Eight (id, key) slots, as the hash-ordered array holds them.
typedef uint32_t Slots8 __attribute__((ext_vector_type(16), aligned(8)));

__global__ __launch_bounds__(kBlock) void k_reorder(uint32_t n, const uint2 *__restrict__ slots,
                                                    const uint32_t *__restrict__ cell_start,
                                                    const float4 *__restrict__ xs_can,
                                                    const float4 *__restrict__ x_can,
                                                    uint32_t *__restrict__ key_s,
                                                    uint32_t *__restrict__ id_s,
                                                    float4 *__restrict__ pos,
                                                    float4 *__restrict__ xold,
                                                    uint32_t *__restrict__ fixed_xy,
                                                    uint16_t *__restrict__ fixed_z,
                                                    double fixed_scale) {
  const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= n) return;
  const uint2 me = slots[t];
  const uint32_t a = cell_start[me.y], b = cell_start[me.y + 1];
  const float4 q = xs_can[me.x], o = x_can[me.x];
  uint32_t s = a, m = a;
  // Crowded cells (compressed fluid, a scene fallen into a corner or no longer a number):
  // a wave all of one cell reads its slots as scalars, others sixteen at a time.  With
  // 100,000 particles in one cell this kernel takes 7.8 ms with four ids in flight, 2.6
  // with sixteen, 2.1 with scalars (the list build 4.7); with 250,000 21.2, 9.7 and 4.9
  // (29.2).
  if (__ballot(b - a > 16u) != 0ull) {
    const uint32_t wave_a = (uint32_t)__builtin_amdgcn_readfirstlane((int)a);
    if (__ballot(a != wave_a) == 0ull) {
      const uint32_t wave_b = (uint32_t)__builtin_amdgcn_readfirstlane((int)b);
      uint32_t k = wave_a;
      for (; wave_b - k > 16u; k += 16) {
        const Slots8 lo = *reinterpret_cast<const Slots8 *>(slots + k);
        const Slots8 hi = *reinterpret_cast<const Slots8 *>(slots + k + 8);
#pragma unroll
        for (int u = 0; u < 16; u += 2) s += lo[u] < me.x ? 1u : 0u;
#pragma unroll
        for (int u = 0; u < 16; u += 2) s += hi[u] < me.x ? 1u : 0u;
      }
      m = k;
    }
    for (; b - m > 16u; m += 16) {
      uint32_t id[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) id[u] = slots[m + u].x;
#pragma unroll
      for (int u = 0; u < 16; ++u) s += id[u] < me.x ? 1u : 0u;
    }
  }
  for (; m < b; m += 4) {  // four ids in flight
    uint32_t id[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) id[u] = m + u < b ? slots[m + u].x : 0xFFFFFFFFu;
#pragma unroll
    for (int u = 0; u < 4; ++u) s += id[u] < me.x ? 1u : 0u;
  }
  key_s[s] = me.y;
  id_s[s] = me.x;
  pos[s] = q;
  fixed_xy[s] = fixed16(q.x, fixed_scale) | fixed16(q.y, fixed_scale) << 16;
  fixed_z[s] = (uint16_t)fixed16(q.z, fixed_scale);
  xold[s] = o;
}

// ---------------------------------------------------------------------------
// Neighbour lists: FillNeighbors (neighbors.c:217-298)
// ---------------------------------------------------------------------------
// r^2 < h^2 evaluated exactly as the reference does it, in double with the
// reference's association and no contraction (neighbors.c:278-285).
__device__ __noinline__ bool inside_exact(float px, float py, float pz, float qx, float qy,
                                          float qz, double h2d) {
#pragma clang fp contract(off)
  const double dx = (double)px - (double)qx;
  const double dy = (double)py - (double)qy;
  const double dz = (double)pz - (double)qz;
  const double r2 = dx * dx + dy * dy + dz * dz;
  return r2 < h2d;
}

// Appends the bits of N candidates, from the 16-bit coordinates at XY and Z, to the
// masks of hits (r^2 < h^2) and of those that the rounding leaves to be decided
// exactly, one for every 20 particles; candidate t ends at bit t, so the last are fed
// first.  With w = r^2 - h^2 + kFixedBand in steps^2, negative is a hit, and 0 to below
// 2 kFixedBand (unsigned) to be decided.  16-byte loads of consecutive candidates: a
// wave's lanes (about 8 cells) then touch 2-3 cache lines per load instead of about 8
// for 16-byte records.  Reads up to 7 entries past a range, which kPosPad allows.
//
// The walk is bounded by the bytes its loads return through the vector L1 and, close
// behind, by the VALU.  This takes 6 bytes and 5 instructions a candidate: the squares
// in one dot product and one multiply-add, the bit from the sign, and one min3 for two
// candidates to see whether the wave has any to decide.  With float arrays it was 12
// bytes and 10 instructions, later 7.8.  k_build_lists (us), 12 bytes and 10 / 7.8 and
// the halves of test32 / this: 8.4M particles 876 / 840 / 741, 1M 103 / 98 / 88.6,
// 442k 50.3 / 48.0 / 43.8; k_build_rows at 131k 20.2 / 20.2 / 19.1, at 4k 7.4 / 7.4 /
// 7.5; the reorder, which writes half the bytes, 174 / 174 / 163 at 8.4M.
typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4_2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x2_2 __attribute__((ext_vector_type(2), aligned(2)));

// z.lo^2 + c or z.hi^2 + c, signed.
__device__ __forceinline__ int square_lo(s16x2 z, int c) {
  int w;
  asm("v_mad_i32_i16 %0, %1, %1, %2" : "=v"(w) : "v"(z), "s"(c));
  return w;
}
__device__ __forceinline__ int square_hi(s16x2 z, int c) {
  int w;
  asm("v_mad_i32_i16 %0, %1, %1, %2 op_sel:[1,1,0,0]" : "=v"(w) : "v"(z), "s"(c));
  return w;
}

template <int N>
__device__ __forceinline__ void test(s16x2 pxy, s16x2 pzz, const uint32_t *XY,
                                     const uint16_t *Z, uint32_t &hits, uint32_t &exact) {
  uint32_t xy[N], zz[N / 2];
#pragma unroll
  for (int v = 0; v < N / 4; ++v) {
    const u32x4 a = *reinterpret_cast<const u32x4 *>(XY + 4 * v);
#pragma unroll
    for (int t = 0; t < 4; ++t) xy[4 * v + t] = a[t];
  }
  if constexpr (N == 8) {
    const u32x4_2 a = *reinterpret_cast<const u32x4_2 *>(Z);
#pragma unroll
    for (int t = 0; t < 4; ++t) zz[t] = a[t];
  } else {
    static_assert(N == 4, "one load of z");
    const u32x2_2 a = *reinterpret_cast<const u32x2_2 *>(Z);
    zz[0] = a[0];
    zz[1] = a[1];
  }
  constexpr int c = kFixedBand - kFixedH * kFixedH;
  uint32_t w[N], nearest = 0xFFFFFFFFu;
#pragma unroll
  for (int t = N - 1; t >= 0; --t) {
    const s16x2 d = pxy - __builtin_bit_cast(s16x2, xy[t]);
    const s16x2 z = pzz - __builtin_bit_cast(s16x2, zz[t / 2]);
    w[t] = (uint32_t)__builtin_amdgcn_sdot2(d, d, t & 1 ? square_hi(z, c) : square_lo(z, c),
                                            false);
    hits = __builtin_amdgcn_alignbit(hits, w[t], 31);
  }
#pragma unroll
  for (int t = 0; t < N; t += 2) nearest = min(min(nearest, w[t]), w[t + 1]);
  exact <<= N;
  if (__ballot(nearest < 2u * kFixedBand) != 0ull) {
#pragma unroll
    for (int t = 0; t < N; ++t) exact |= w[t] < 2u * kFixedBand ? 1u << t : 0u;
  }
}

// The masks of up to 32 candidates.  Groups last to first: a lane skips a suffix of
// the groups, which then come first, while its masks are still 0.  A row of three
// cells holds 24 particles or a few more, so the last 8 go in two halves.
__device__ __forceinline__ void test32(s16x2 pxy, s16x2 pzz, const uint32_t *XY,
                                       const uint16_t *Z, uint32_t len, uint32_t &hits,
                                       uint32_t &exact) {
#pragma unroll
  for (int g = 28; g >= 24; g -= 4)
    if ((uint32_t)g < len) test<4>(pxy, pzz, XY + g, Z + g, hits, exact);
#pragma unroll
  for (int g = 16; g >= 0; g -= 8)
    if ((uint32_t)g < len) test<8>(pxy, pzz, XY + g, Z + g, hits, exact);
}

// One thread per sorted particle.  The 3 cells (dx = -1..1) of each (dz, dy)
// row are consecutive keys, so each row is one contiguous range of sorted
// indices; walking rows in (dz, dy) order and indices upward reproduces the
// reference's (dz, dy, dx, id) order and therefore its 60-cap truncation.
//
// Hits are buffered in LDS as 16-bit offsets from the first candidate of
// their dz layer and written out after the scan as compact quads (8 entries
// each): a wave then stores 1 KB of the list contiguously per instruction.
// Written as found, lanes store their k-th neighbour at different times and
// partially written lines are written back several times.  A wavefront in
// which some particle's layer spans more than kCompactSpan indices (never
// near rest density: a layer holds about two grid rows of particles), or
// every wavefront when `force_wide` is set, writes 32-bit indices directly.
// The head records the layer bases (the particle itself for a layer without
// candidates, so that padding entries decode to a valid index) and counts.
template <bool BATCH>
__global__ __launch_bounds__(kBlock, 7) void k_build_lists(
    uint32_t n, uint32_t nblocks, const float4 *__restrict__ pos,
    const uint32_t *__restrict__ XY, const uint16_t *__restrict__ Z,
    const uint32_t *__restrict__ key_s, const uint32_t *__restrict__ cstart, DevParams P,
    uint32_t *__restrict__ list, uint4 *__restrict__ head, uint32_t *__restrict__ stats,
    uint32_t *__restrict__ pair_partial, int force_wide, BatchDev B) {
  extern __shared__ uint16_t sbuf[];  // [kLdsHits][blockDim.x]
  const uint32_t s = particle_index(nblocks);
  int c = 0;
  uint32_t dropped = 0;
  bool wide = false;
  uint32_t *out = list + (size_t)(s >> 6) * kListStride + (s & 63u) * 4u;
  if (s < n) {
    const float4 p = pos[s];
    const s16x2 pxy = __builtin_bit_cast(s16x2, XY[s]), pzz = {(short)Z[s], (short)Z[s]};
    // a NaN has no neighbours (two of one cell share their 16-bit coordinate)
    const bool nan = !(p.x == p.x && p.y == p.y && p.z == p.z);
    const Geo G = geo_of<BATCH>(s, P, B);
    const uint32_t key = key_s[s] - G.base;
    const uint32_t cz = key / G.nxy;
    const uint32_t rem = key - cz * G.nxy;
    const uint32_t cy = rem / G.nx;
    const uint32_t cx = rem - cy * G.nx;
    const uint32_t x0 = cx > 0 ? cx - 1 : 0;
    const uint32_t x1 = cx + 1 < G.nx ? cx + 1 : G.nx - 1;
    const uint32_t y0 = cy > 0 ? cy - 1 : 0;
    const uint32_t y1 = cy + 1 < G.ny ? cy + 1 : G.ny - 1;
    uint32_t base[3] = {s, s, s};
    bool direct = force_wide != 0;
#pragma unroll
    for (int l = 0; l < 3; ++l) {
      const int z = (int)cz + l - 1;
      if (z < 0 || z >= (int)G.nz) continue;
      const uint32_t zrow = G.base + (uint32_t)z * G.nxy;
      const uint32_t first = cstart[zrow + y0 * G.nx + x0];
      const uint32_t span = cstart[zrow + y1 * G.nx + x1 + 1] - first;
      if (span > 0u) base[l] = first;
      if (span > kCompactSpan) direct = true;
    }
    // the format is per wavefront (the lanes' quads interleave)
    wide = __ballot(direct) != 0ull;
    int cl[3] = {0, 0, 0};
    uint32_t slot = threadIdx.x;  // c * blockDim.x + threadIdx.x
    for (int dz = -1; dz <= 1; ++dz) {
      const int z = (int)cz + dz;
      if (z >= 0 && z < (int)G.nz) {
        const uint32_t lb = dz < 0 ? base[0] : (dz == 0 ? base[1] : base[2]);
        // the layer's three row ranges in one round trip (a row outside the
        // grid is read at the particle's own row and left empty)
        uint32_t r0[3], r1[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const int y = (int)cy + k - 1;
          const bool in = y >= 0 && y < (int)G.ny;
          const uint32_t row = G.base + (uint32_t)z * G.nxy + (in ? (uint32_t)y : cy) * G.nx;
          r0[k] = cstart[row + x0];
          r1[k] = cstart[row + x1 + 1];
          if (!in) r1[k] = r0[k];
        }
        for (int k = 0; k < 3; ++k) {
          const uint32_t j0 = k == 0 ? r0[0] : (k == 1 ? r0[1] : r0[2]);
          const uint32_t j1 = k == 0 ? r1[0] : (k == 1 ? r1[1] : r1[2]);
          // candidates 32 at a time: test all (8 loads in flight per group),
          // then append the hits of the chunk in j order
          for (uint32_t cb = j0; cb < j1; cb += 32) {
            const uint32_t len = j1 - cb;
            uint32_t lo = 0u, band = 0u;  // hits, and candidates within the guard band
            test32(pxy, pzz, XY + cb, Z + cb, len, lo, band);
            uint32_t keep = len >= 32u ? ~0u : (1u << len) - 1u;
            if (s - cb < 32u) keep &= ~(1u << (s - cb));  // not the particle itself
            if (nan) keep = 0u;
            band &= keep;
            lo &= keep & ~band;
            while (band) {
              const int t = __builtin_ctz(band);
              band &= band - 1u;
              const float4 q = pos[cb + t];
              if (inside_exact(p.x, p.y, p.z, q.x, q.y, q.z, P.h2d)) lo |= 1u << t;
            }
            // append the chunk's hits in j order; the cap and the end of the
            // LDS buffer are tested per hit only when this chunk can reach
            // them (`slot` = the LDS index of entry c, kept as a running sum)
            const int nh = __builtin_popcount(lo);
            if (wide && c + nh <= kMaxNb) {
              while (lo) {
                const uint32_t j = cb + (uint32_t)__builtin_ctz(lo);
                lo &= lo - 1u;
                out[(size_t)(c >> 2) * kQuadStride + (c & 3)] = j;
                ++c;
              }
            } else if (!wide && c + nh <= kLdsHits) {
              while (lo) {
                const uint32_t j = cb + (uint32_t)__builtin_ctz(lo);
                lo &= lo - 1u;
                sbuf[slot] = (uint16_t)(j - lb);
                slot += blockDim.x;
              }
              c += nh;
            } else {
              while (lo) {
                const uint32_t j = cb + (uint32_t)__builtin_ctz(lo);
                lo &= lo - 1u;
                if (c < kMaxNb) {
                  if (wide)
                    out[(size_t)(c >> 2) * kQuadStride + (c & 3)] = j;
                  else if (c < kLdsHits)
                    sbuf[slot] = (uint16_t)(j - lb);
                  else
                    store_entry16(out, c, j - lb);
                  slot += blockDim.x;
                  ++c;
                } else {
                  ++dropped;
                }
              }
            }
          }
        }
      }
      cl[dz + 1] = c;
    }
    head[s] = make_uint4(base[0], base[1], base[2],
                         (uint32_t)c | ((uint32_t)cl[0] << 8) | ((uint32_t)cl[1] << 16) |
                             (wide ? kHeadWide : 0u));
    // the rest of a directly stored last quad is padding: offset 0 (readers
    // decode whole quads, and a stale offset could index past the particles)
    if (!wide && c > kLdsHits)
      for (int e = c; (e & 7) != 0; ++e) store_entry16(out, e, 0u);
  }
  // coalesced write-out of compact quads: every lane of the wave walks the
  // wave's longest list one quad (8 entries) at a time, up to the end of the
  // LDS buffer (later quads were stored directly)
  int cmax = wide ? 0 : c;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) cmax = max(cmax, __shfl_xor(cmax, o, 64));
  for (int k = 0; k < cmax && k < kLdsHits; k += 8) {
    if (k < c) {
      uint32_t w[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const uint32_t lo = (k + 2 * t < c) ? sbuf[(k + 2 * t) * blockDim.x + threadIdx.x] : 0u;
        const uint32_t hi =
            (k + 2 * t + 1 < c) ? sbuf[(k + 2 * t + 1) * blockDim.x + threadIdx.x] : 0u;
        w[t] = lo | (hi << 16);
      }
      *reinterpret_cast<uint4 *>(out + (size_t)(k >> 3) * kQuadStride) =
          make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
  add_counter64_wave(stats, STAT_DROPPED, dropped);
  block_sum_to(pair_partial, (uint32_t)c);
}

// The same lists with several wavefronts per 64-particle group, each walking
// ROWS of a particle's nine (dz, dy) rows (one row, or a dz layer's three): the
// waves count their hits side by side, take their places in the list from the
// counts of the waves before them, and write the group's quads out of one LDS
// buffer.  For the sizes at which k_build_lists leaves the chip idle and its
// time is one wave's walk through nine rows in turn, about 20 us whatever the
// size; with more particles the particle's set-up made several times over costs
// more than the shorter walk gives.  Measured (us, events included), k_build_lists
// / three waves a group / nine: 4k particles 23.0 / 13.5 / 9.2, 33k 23.9 / 14.9 /
// 11.6, 47k 24.8 / 16.1 / 16.9, 133k 30.9 / 26.1 / 36.7, 185k 32.4 / 32.2 / 47.6,
// 262k 38.3 / 39.9 / 63.9, 8.4M (no events) 871 / 902 / 1833.
constexpr uint32_t kOneRowBuildMax = 40960, kRowBuildMax = 196608;

template <bool BATCH, int ROWS>
__global__ __launch_bounds__(9 / ROWS * kWave, 7) void k_build_rows(
    uint32_t n, const float4 *__restrict__ pos, const uint32_t *__restrict__ XY,
    const uint16_t *__restrict__ Z, const uint32_t *__restrict__ key_s,
    const uint32_t *__restrict__ cstart, DevParams P,
    uint32_t *__restrict__ list, uint4 *__restrict__ head, uint32_t *__restrict__ stats,
    uint32_t *__restrict__ pair_partial, int force_wide, BatchDev B) {
  constexpr int WAVES = 9 / ROWS;
  __shared__ uint16_t hits[kMaxNb][kWave];  // offsets from the layer's first candidate
  __shared__ uint32_t count[WAVES][kWave], layer[3][kWave];
  const uint32_t lane = threadIdx.x & 63u;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t group = xcd_block(blockIdx.x, gridDim.x);
  const uint32_t s = group * kWave + lane;
  const int l = wave * ROWS / 3;                      // dz layer of this wave
  const int dz = l - 1, dy0 = wave * ROWS - 3 * l - 1;  // its first row
  uint32_t j0[ROWS], j1[ROWS], base = s;
#pragma unroll
  for (int k = 0; k < ROWS; ++k) j0[k] = j1[k] = 0u;
  float4 p = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  s16x2 pxy = {0, 0}, pzz = {0, 0};
  bool direct = force_wide != 0, nan = false;
  if (s < n) {
    p = pos[s];
    pxy = __builtin_bit_cast(s16x2, XY[s]);
    pzz = s16x2{(short)Z[s], (short)Z[s]};
    nan = !(p.x == p.x && p.y == p.y && p.z == p.z);
    const Geo G = geo_of<BATCH>(s, P, B);
    const uint32_t key = key_s[s] - G.base;
    const uint32_t cz = key / G.nxy;
    const uint32_t rem = key - cz * G.nxy;
    const uint32_t cy = rem / G.nx;
    const uint32_t cx = rem - cy * G.nx;
    const uint32_t x0 = cx > 0 ? cx - 1 : 0;
    const uint32_t x1 = cx + 1 < G.nx ? cx + 1 : G.nx - 1;
    const int z = (int)cz + dz;
    if (z >= 0 && z < (int)G.nz) {
      const uint32_t zrow = G.base + (uint32_t)z * G.nxy;
      const uint32_t y0 = cy > 0 ? cy - 1 : 0;
      const uint32_t y1 = cy + 1 < G.ny ? cy + 1 : G.ny - 1;
      const uint32_t first = cstart[zrow + y0 * G.nx + x0];
      const uint32_t span = cstart[zrow + y1 * G.nx + x1 + 1] - first;
#pragma unroll
      for (int k = 0; k < ROWS; ++k) {
        const int y = (int)cy + dy0 + k;
        const bool in = y >= 0 && y < (int)G.ny;
        const uint32_t r = zrow + (in ? (uint32_t)y : cy) * G.nx;
        j0[k] = cstart[r + x0];
        j1[k] = cstart[r + x1 + 1];
        if (!in) j1[k] = j0[k];
      }
      if (span > 0u) base = first;
      if (span > kCompactSpan) direct = true;
    }
  }
  // hits of the up to 32 candidates [cb, end) as a mask
  auto hits_of = [&](uint32_t cb, uint32_t end) {
    const uint32_t len = end - cb;
    uint32_t lo = 0u, band = 0u;  // as in k_build_lists
    test32(pxy, pzz, XY + cb, Z + cb, len, lo, band);
    uint32_t keep = len >= 32u ? ~0u : (1u << len) - 1u;
    if (s - cb < 32u) keep &= ~(1u << (s - cb));  // not the particle itself
    if (nan) keep = 0u;
    band &= keep;
    lo &= keep & ~band;
    while (band) {
      const int t = __builtin_ctz(band);
      band &= band - 1u;
      const float4 q = pos[cb + t];
      if (inside_exact(p.x, p.y, p.z, q.x, q.y, q.z, P.h2d)) lo |= 1u << t;
    }
    return lo;
  };
  // a row's first mask is kept, later ones (rows of more than 32, in compressed
  // fluid) are made again when the hits are stored
  uint32_t m0[ROWS], mine = 0u;
#pragma unroll
  for (int k = 0; k < ROWS; ++k) {
    m0[k] = 0u;
    for (uint32_t cb = j0[k]; cb < j1[k]; cb += 32u) {
      const uint32_t m = hits_of(cb, j1[k]);
      mine += (uint32_t)__builtin_popcount(m);
      if (cb == j0[k]) m0[k] = m;
    }
  }
  count[wave][lane] = mine;
  if (wave * ROWS == 3 * l) layer[l][lane] = base;
  const bool wide = __syncthreads_or(direct ? 1 : 0) != 0;
  uint32_t at = 0u, all = 0u, c1 = 0u, c2 = 0u;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    if (w == wave) at = all;
    if (w == 3 / ROWS) c1 = all;
    if (w == 6 / ROWS) c2 = all;
    all += count[w][lane];
  }
  uint32_t *out = list + (size_t)group * kListStride + lane * 4u;
#pragma unroll
  for (int k = 0; k < ROWS; ++k) {
    for (uint32_t cb = j0[k]; cb < j1[k] && at < (uint32_t)kMaxNb; cb += 32u) {
      uint32_t m = cb == j0[k] ? m0[k] : hits_of(cb, j1[k]);
      while (m && at < (uint32_t)kMaxNb) {
        const uint32_t j = cb + (uint32_t)__builtin_ctz(m);
        m &= m - 1u;
        if (wide)
          out[(size_t)(at >> 2) * kQuadStride + (at & 3u)] = j;
        else
          hits[at][lane] = (uint16_t)(j - base);
        ++at;
      }
    }
  }
  __syncthreads();
  const uint32_t c = min(all, (uint32_t)kMaxNb);
  for (uint32_t q = wave; !wide && 8u * q < (uint32_t)kMaxNb; q += WAVES) {
    const uint32_t k = 8u * q;
    if (k < c) {
      uint32_t w[4];
#pragma unroll
      for (uint32_t t = 0; t < 4; ++t) {
        const uint32_t lo = k + 2 * t < c ? hits[k + 2 * t][lane] : 0u;
        const uint32_t hi = k + 2 * t + 1 < c ? hits[k + 2 * t + 1][lane] : 0u;
        w[t] = lo | (hi << 16);
      }
      *reinterpret_cast<uint4 *>(out + (size_t)q * kQuadStride) =
          make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
  if (wave == WAVES - 1) {
    c1 = min(c1, (uint32_t)kMaxNb);
    c2 = min(c2, (uint32_t)kMaxNb);
    if (s < n)
      head[s] = make_uint4(layer[0][lane], layer[1][lane], layer[2][lane],
                           c | (c1 << 8) | (c2 << 16) | (wide ? kHeadWide : 0u));
    add_counter64_wave(stats, STAT_DROPPED, all - c);
    uint32_t t = c;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) t += __shfl_xor(t, o, 64);
    if (lane == 0) pair_partial[blockIdx.x] = t;
  }
}

// ---------------------------------------------------------------------------
// Jacobi constraint loop
// ---------------------------------------------------------------------------
// The error maximum of a density pass: a wave's maximum of a non-negative float,
// then one atomic on its bit pattern (monotonic for non-negative floats) on the
// iteration's word for the wave's number, which nothing waits for.  Without the
// error the density pass takes 39.8 us at 1M particles and 6.0 at 32k.  With one
// word, read and if need be raised by each block at its end, it took 45.2 and 7.9
// (a barrier and a memory round trip a block); an atomic per
// wave costs 40.8 and 6.9.
// Every lane of the wave must call it.
__device__ __forceinline__ void raise_error(uint32_t *stats, int it, float v, bool active) {
  float m = active ? v : 0.0f;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  if ((threadIdx.x & 63) == 0 && m > 0.0f)
    atomicMax(&stats[err_word((uint32_t)it, wave & (kErrSlots - 1u))], __float_as_uint(m));
}

// The maximum an iteration's waves left (bits), in every lane of the wave.
__device__ __forceinline__ uint32_t max_error(const uint32_t *stats, int it) {
  uint32_t m = stats[err_word((uint32_t)it, threadIdx.x & (kErrSlots - 1u))];
#pragma unroll
  for (int o = kErrSlots / 2; o >= 1; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o, 64));
  return m;
}

__device__ __forceinline__ bool converged(const uint32_t *stats) {
  return stats[STAT_CONVERGED] != 0u;
}

// One neighbour's density term: the integer (k3 (h^2 - r^2))^3, truncated
// (W(r) = norm (h^2 - r^2)^3, 0 for r >= h).  u and u^3 are computed in
// double (half the FP32 rate on this target, a few VALU slots more per
// neighbour): in FP32 their roundings (about 4e-7 of a term, independent
// between terms) moved C = rho/rho0 - 1 by up to 2e-7, which near rest,
// where C itself is 1e-3..1e-2, is lambda's largest error.  Sums of at most
// 60 terms of at most 2^26 fit 32 bits; the sum is exact and independent of
// the order of the terms.
__device__ __forceinline__ uint32_t density_term(float r2, const DevParams &P) {
  const double u = fmax(fma(-(double)r2, P.dens_k3, P.dens_c1), 0.0);
  return (uint32_t)((u * u) * u);
}

// C = rho/rho0 - 1 from the fixed-point density sum S of cnt terms.  Each
// truncation drops half a unit on average, restored by cnt/2.  S is split
// into 20 high and 12 low bits, each exact in FP32, and C = a S + c0 is
// evaluated with a and c0 as float pairs: near rest C ~ 1e-3 is the
// difference of two terms ~0.8, and this keeps its error at the FP32
// rounding of the terms instead of that of rho ~ 1e3.
__device__ __forceinline__ float density_constraint(uint32_t S, int cnt, const DevParams &P) {
  S += (uint32_t)cnt >> 1;
  const float shi = (float)(S & 0xFFFFF000u), slo = (float)(S & 0xFFFu);
  return fmaf(P.dens_a_hi, shi, P.dens_c0_hi) +
         (P.dens_c0_lo + fmaf(P.dens_a_lo, shi, P.dens_a_hi * slo));
}

// ComputeDensities (particles.c:461-514) and ComputeLambda (particles.c:588-666)
// in one gather: rho_i needs only r^2, lambda_i needs C_i (own) and the
// spiky gradients.  Writes rho and pos.w = lambda.
// MODE 0: both, 1: density only, 2: lambda only (C from c_io).  With c_io,
// MODE 0/1 also store C there; with with_lambda, (x*, lambda) goes to that
// buffer and pos.w keeps rho (density_to_w).
template <int MODE, int NB>
__global__ GATHER_BOUNDS(NB) void k_density_lambda(
    uint32_t n, uint32_t nblocks, float4 *pos, const uint32_t *__restrict__ list,
    const uint4 *__restrict__ head, DevParams P, float *__restrict__ rho_out, float *c_io,
    uint32_t *stats, int err_slot, int check_converged, int density_to_w,
    float4 *__restrict__ with_lambda) {
  if (check_converged && converged(stats)) return;
  const uint32_t s = gather_index<NB>(nblocks);
  const bool active = s < n, lead = gather_lead<NB>();
  float err = 0.0f;
  if (active) {
    const float4 p = pos[s];
    int cnt;
    uint32_t S = 0u;
    const Records16 G(pos, n);
    const auto load = [&](uint32_t j) { return G[j]; };
    // sum of g d (three), and of g^2 r^2
    float sg[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const auto term = [&](const float4 &q) {
      const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
      const float r2 = sq3(dx, dy, dz);
      if (MODE != 2) S += density_term(r2, P);
      const float r2c = fmaxf(r2, P.rmin2);
      const float ir = fast_rsq(r2c);
      const float hr = fmaf(-r2c, ir, P.h);  // h - r, r floored at 1e-4 h
      const float hp = fmaxf(hr, 0.0f);  // a listed pair can be past h after an update
      const float g = hp * hp * ir;  // DelW(r)/r / norm
      return Terms<4>{{g, g, g, g * g}, {dx, dy, dz, r2}};
    };
    if constexpr (MODE == 1) {
      float none[1];
      sum_neighbors<float4, NB, kRaw, 1, 1>(list, head, s, &cnt, none, load,
                                            [&](const float4 &q) {
        S += density_term(sq3(p.x - q.x, p.y - q.y, p.z - q.z), P);
        return Terms<1>{{0.0f}, {0.0f}};
      });
    } else {
      sum_neighbors<float4, NB, kRaw, 4, 1>(list, head, s, &cnt, sg, load, term);
    }
    if constexpr (NB == kQuad) S = quad_sum(S);
    float C;
    if (MODE != 2) {
      C = density_constraint(S, cnt, P);
      const float rho = fmaf(C, P.rest_density, P.rest_density);
      if (lead) rho_out[s] = rho;
      if (c_io && lead) c_io[s] = C;
      // the reported error is that of the stored density, as every later
      // reader of rho (per-scene errors, the warm fallback) computes it
      err = fmaxf((rho - P.rest_density) * P.inv_rest_density, 0.0f);
      if (density_to_w && lead) pos[s].w = rho;
    } else {
      C = c_io[s];
    }
    if (MODE != 1) {
      const float Ci = fmaxf(C, 0.0f);
      const float sum_c = P.lam_k2 * (sg[3] + sq3(sg[0], sg[1], sg[2]));
      const float lam = -Ci / (sum_c + P.lambda_eps);
      if (!lead) {
      } else if (with_lambda) {
        with_lambda[s] = make_float4(p.x, p.y, p.z, lam);
      } else {
        pos[s].w = lam;
      }
    }
  }
  // every lane gets here: the only early return above is uniform
  if (MODE != 2 && err_slot >= 0) raise_error(stats, err_slot, err, active);
}

// Trilinear sample with normalised coordinates, texel centres at (i+0.5)/dim
// and clamp addressing, as tex3D with linear filtering (obstacle_cuda.cu:
// 174-180) defines it, with exact FP32 weights.
__device__ __forceinline__ float sdf_sample(const SdfDev &o, float u, float v, float w) {
  const float cu = u * (float)o.dim[0] - 0.5f;
  const float cv = v * (float)o.dim[1] - 0.5f;
  const float cw = w * (float)o.dim[2] - 0.5f;
  const float fu = floorf(cu), fv = floorf(cv), fw = floorf(cw);
  const float au = cu - fu, av = cv - fv, aw = cw - fw;
  const int iu = (int)fu, iv = (int)fv, iw = (int)fw;
  const int u0 = min(max(iu, 0), o.dim[0] - 1), u1 = min(max(iu + 1, 0), o.dim[0] - 1);
  const int v0 = min(max(iv, 0), o.dim[1] - 1), v1 = min(max(iv + 1, 0), o.dim[1] - 1);
  const int w0 = min(max(iw, 0), o.dim[2] - 1), w1 = min(max(iw + 1, 0), o.dim[2] - 1);
  const size_t sy = (size_t)o.dim[0], sz = (size_t)o.dim[0] * (size_t)o.dim[1];
  const float *d = o.data;
  const float c000 = d[u0 + v0 * sy + w0 * sz], c100 = d[u1 + v0 * sy + w0 * sz];
  const float c010 = d[u0 + v1 * sy + w0 * sz], c110 = d[u1 + v1 * sy + w0 * sz];
  const float c001 = d[u0 + v0 * sy + w1 * sz], c101 = d[u1 + v0 * sy + w1 * sz];
  const float c011 = d[u0 + v1 * sy + w1 * sz], c111 = d[u1 + v1 * sy + w1 * sz];
  const float c00 = c000 + au * (c100 - c000), c10 = c010 + au * (c110 - c010);
  const float c01 = c001 + au * (c101 - c001), c11 = c011 + au * (c111 - c011);
  const float c0 = c00 + av * (c10 - c00), c1 = c01 + av * (c11 - c01);
  return c0 + aw * (c1 - c0);
}

// The push of CalculateParticleCollisions_kernel (obstacle_cuda.cu:81-113)
// at normalised grid coordinates (u, v, w): false outside the obstacle,
// otherwise the world-space push along the SDF gradient.
__device__ __forceinline__ bool sdf_push(const SdfDev &o, float u, float v, float w,
                                         float &px, float &py, float &pz) {
  const float d = sdf_sample(o, u, v, w);
  if (!(d < 0.0f)) return false;
  const float gx = sdf_sample(o, u + o.inv_dim[0], v, w) - sdf_sample(o, u - o.inv_dim[0], v, w);
  const float gy = sdf_sample(o, u, v + o.inv_dim[1], w) - sdf_sample(o, u, v - o.inv_dim[1], w);
  const float gz = sdf_sample(o, u, v, w + o.inv_dim[2]) - sdf_sample(o, u, v, w - o.inv_dim[2]);
  const float dd = gx * gx + gy * gy + gz * gz;
  if (!(dd > 0.0f)) return false;  // the reference would normalise a zero vector to NaN
  const float inv = 1.0f / sqrtf(dd);
  const float dist = fabsf(d) * o.m2w;
  px = dist * (gx * inv);
  py = dist * (gy * inv);
  pz = dist * (gz * inv);
  return true;
}

// CalculateParticleCollisions_kernel (obstacle_cuda.cu:56-116).
__device__ __forceinline__ void collide(float &x, float &y, float &z, const SdfDev &o) {
  if (!o.data) return;
  if (!(x > o.wmin[0] && x < o.wmax[0] && y > o.wmin[1] && y < o.wmax[1] && z > o.wmin[2] &&
        z < o.wmax[2]))
    return;
  const float u = (x - o.wmin[0]) / o.len[0];
  const float v = (y - o.wmin[1]) / o.len[1];
  const float w = (z - o.wmin[2]) / o.len[2];
  float px, py, pz;
  if (!sdf_push(o, u, v, w, px, py, pz)) return;
  y += py;
  x += px;
  z += pz;
}

// UpdateDPs (particles.c:668-746): returns sum_j (lambda_i + lambda_j) DelW(r)/r d.
template <int NB>
__device__ __forceinline__ float3 dp_sum(const float4 &p, const float4 *pos, uint32_t n,
                                         const uint32_t *list, const uint4 *head, uint32_t s,
                                         const DevParams &P) {
  int cnt;
  float a[3];
  const Records16 G(pos, n);
  sum_neighbors<float4, NB, kRaw, 3, 1>(
      list, head, s, &cnt, a, [&](uint32_t j) { return G[j]; }, [&](const float4 &q) {
        const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
        const float r2c = fmaxf(sq3(dx, dy, dz), P.rmin2);
        const float ir = fast_rsq(r2c);
        const float hr = fmaf(-r2c, ir, P.h);
        const float hp = fmaxf(hr, 0.0f);
        const float g = hp * hp * ir;
        const float f = (p.w + q.w) * g;
        return Terms<3>{{f, f, f}, {dx, dy, dz}};
      });
  return make_float3(a[0], a[1], a[2]);
}

// Staged UpdateDPs: dp = stiffness * m * DelW_norm / rho0 * sum.
// With xnext, also the position update of k_position_stars from the same dp
// (x* + dp, clamp, collision, rho into w), into another buffer.
template <bool BATCH, int NB>
__global__ GATHER_BOUNDS(NB) void k_dp(uint32_t n, uint32_t nblocks,
                                               const float4 *__restrict__ pos,
                                               const uint32_t *__restrict__ list,
                                               const uint4 *__restrict__ head, DevParams P,
                                               float scale, float4 *__restrict__ dp,
                                               float4 *__restrict__ xnext,
                                               const float *__restrict__ rho, SdfDev o,
                                               BatchDev B) {
  const uint32_t s = gather_index<NB>(nblocks);
  if (s >= n) return;
  const float4 p = pos[s];
  const float3 a = dp_sum<NB>(p, pos, n, list, head, s, P);
  const float4 d = make_float4(scale * a.x, scale * a.y, scale * a.z, 0.0f);
  const bool lead = gather_lead<NB>();
  if (lead) dp[s] = d;
  if (xnext) {
    float x = p.x + d.x, y = p.y + d.y, z = p.z + d.z;
    apply_boundary(x, y, z, geo_of<BATCH>(s, P, B), P);
    collide(x, y, z, sdf_of<BATCH>(s, o, B));
    if (lead) xnext[s] = make_float4(x, y, z, rho[s]);
  }
}

// Staged UpdatePositionStars (particles.c:529-564): x* += dp, clamp, collide.
// Also stores rho in w for the velocity passes.
template <bool BATCH>
__global__ __launch_bounds__(kBlock) void k_position_stars(uint32_t n, float4 *__restrict__ pos,
                                                           const float4 *__restrict__ dp,
                                                           const float *__restrict__ rho,
                                                           DevParams P, SdfDev o, BatchDev B) {
  const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= n) return;
  const float4 p = pos[s], d = dp[s];
  float x = p.x + d.x, y = p.y + d.y, z = p.z + d.z;
  apply_boundary(x, y, z, geo_of<BATCH>(s, P, B), P);
  collide(x, y, z, sdf_of<BATCH>(s, o, B));
  pos[s] = make_float4(x, y, z, rho[s]);
}

// UpdateVelocities (particles.c:787-838).
__device__ __forceinline__ float4 velocity_of(const float4 &p, const float4 &xo,
                                              const DevParams &P) {
  float vx = (p.x - xo.x) / P.dt, vy = (p.y - xo.y) / P.dt, vz = (p.z - xo.z) / P.dt;
  vx = fminf(fmaxf(vx, -P.v_max), P.v_max);
  vy = fminf(fmaxf(vy, -P.v_max), P.v_max);
  vz = fminf(fmaxf(vz, -P.v_max), P.v_max);
  return make_float4(vx, vy, vz, 0.0f);
}

// Where a substep's last position update writes its results when nothing follows
// it: the velocity in sorted order, and position and velocity by id.
struct FinishDev {
  const float4 *xold = nullptr;  // null: not the last pass
  float4 *vel = nullptr;
  const uint32_t *id_s = nullptr;
  float4 *x_can = nullptr, *v_can = nullptr;
};

// Fused UpdateDPs + UpdatePositionStars: reads pin (x*, lambda), writes pout
// (x*', rho).  COLLIDE false leaves the obstacle to k_collide_sorted (a launch
// choice; the trilinear gradient needs no more registers than the gathers).  In
// tolerance mode, once the density pass of this iteration is
// within tolerance, the particles are copied unchanged instead.  With lam_acc,
// adds stiff * lambda_i to the particle's accumulated multiplier.  With fin, also
// UpdateVelocities and UpdatePositions of the particle (particles.c:787-838,566-586):
// a substep without velocity terms has two launches and four passes over memory
// less (a graph-replayed frame of 33k particles 694 -> 669 us).
template <bool COLLIDE, bool BATCH, int NB>
__global__ GATHER_BOUNDS(NB) void k_dp_update(
    uint32_t n, uint32_t nblocks, const float4 *__restrict__ pin, float4 *__restrict__ pout,
    const float *__restrict__ rho, const uint32_t *__restrict__ list,
    const uint4 *__restrict__ head, DevParams P, float scale, SdfDev o, uint32_t *stats,
    int err_slot, int fallback_slot, float tol, float *__restrict__ lam_acc, float stiff,
    BatchDev B, FinishDev fin) {
  bool done = false;
  if (tol > 0.0f) {
    // a substep that fell back goes on from the error before its warm start
    const int slot = stats[STAT_FALLBACK] ? fallback_slot : err_slot;
    done = converged(stats) || __uint_as_float(max_error(stats, slot)) <= tol;
  }
  const uint32_t s = gather_index<NB>(nblocks);
  if (s >= n) return;
  const bool lead = gather_lead<NB>();
  const float4 p = pin[s];
  float x = p.x, y = p.y, z = p.z;
  if (done) {
    if (s == 0) stats[STAT_CONVERGED] = 1u;
  } else {
    if (s == 0 && lead) stats[STAT_ITERS] += 1u;
    const float3 a = dp_sum<NB>(p, pin, n, list, head, s, P);
    x = fmaf(scale, a.x, p.x), y = fmaf(scale, a.y, p.y), z = fmaf(scale, a.z, p.z);
    apply_boundary(x, y, z, geo_of<BATCH>(s, P, B), P);
    if (COLLIDE) collide(x, y, z, sdf_of<BATCH>(s, o, B));
    if (lam_acc && lead) lam_acc[s] = fmaf(stiff, p.w, lam_acc[s]);
  }
  if (!lead) return;
  const float4 q = make_float4(x, y, z, rho[s]);
  pout[s] = q;
  if (!fin.xold) return;
  const float4 v = velocity_of(q, fin.xold[s], P);
  const uint32_t id = fin.id_s[s];
  fin.vel[s] = v;
  fin.x_can[id] = make_float4(x, y, z, 0.0f);
  fin.v_can[id] = v;
}

// ---------------------------------------------------------------------------
// Learned warm start
// ---------------------------------------------------------------------------
// SDF distance (in h, clamped to [-4, 4]) and unit gradient at a point, with
// the sampling of the collision pass (obstacle_cuda.cu:33-53,88).
__device__ __forceinline__ void sdf_features(float x, float y, float z, const SdfDev &o,
                                             const DevParams &P, float *f) {
  f[0] = 4.0f;
  f[1] = f[2] = f[3] = 0.0f;
  if (!o.data) return;
  if (!(x > o.wmin[0] && x < o.wmax[0] && y > o.wmin[1] && y < o.wmax[1] && z > o.wmin[2] &&
        z < o.wmax[2]))
    return;
  const float u = (x - o.wmin[0]) / o.len[0];
  const float v = (y - o.wmin[1]) / o.len[1];
  const float w = (z - o.wmin[2]) / o.len[2];
  const float d = sdf_sample(o, u, v, w);
  f[0] = fminf(fmaxf(d * o.m2w * P.inv_h, -4.0f), 4.0f);
  const float gx = sdf_sample(o, u + o.inv_dim[0], v, w) - sdf_sample(o, u - o.inv_dim[0], v, w);
  const float gy = sdf_sample(o, u, v + o.inv_dim[1], w) - sdf_sample(o, u, v - o.inv_dim[1], w);
  const float gz = sdf_sample(o, u, v, w + o.inv_dim[2]) - sdf_sample(o, u, v, w - o.inv_dim[2]);
  const float dd = gx * gx + gy * gy + gz * gz;
  if (!(dd > 0.0f)) return;
  const float inv = 1.0f / sqrtf(dd);
  f[1] = gx * inv;
  f[2] = gy * inv;
  f[3] = gz * inv;
}

// First pass of a warm-started or logged solve.  ComputeDensities and
// ComputeLambda as in k_density_lambda, plus the network features, in one
// gather of (x*, x) per neighbour.  LOG: writes the feature rows and the
// plain lambda.  Otherwise runs the network on MFMA (BF16, FP32 accumulate),
// whose output R estimates what the later iterations of a converged solve add
// to the multiplier, and writes lambda_0 - scale * max(R, 0) / (|grad C|^2 + eps):
// the plain first step plus the predicted remainder.
// Either way the particle's accumulated multiplier restarts at zero.  Every
// lane of a wave reaches the network (no early return).
template <bool LOG, bool BATCH, int NB = 8>
__global__ __launch_bounds__(kBlock) void k_warm_lambda(
    uint32_t n, uint32_t nblocks, float4 *pos, const float4 *__restrict__ xold,
    const uint32_t *__restrict__ list, const uint4 *__restrict__ head, DevParams P,
    float *__restrict__ rho_io, uint32_t *stats, const uint32_t *__restrict__ id_s,
    const float *__restrict__ lam_prev, SdfDev o, const MlpPacked *__restrict__ net,
    float *__restrict__ lam_acc, float *__restrict__ feat, float2 *__restrict__ plain,
    BatchDev B) {
  const uint32_t s = particle_index(nblocks);
  const bool active = s < n;
  float f[kMlpPad];
#pragma unroll
  for (int i = 0; i < kMlpPad; ++i) f[i] = 0.0f;
  float err = 0.0f, lam0 = 0.0f, denom = 1.0f, rho = 0.0f;
  if (active) {
    const float4 p = pos[s];
    const float4 po = xold[s];
    const float ux = p.x - po.x, uy = p.y - po.y, uz = p.z - po.z;  // dt * v_i
    int cnt;
    uint32_t S = 0u;
    float sgx = 0.0f, sgy = 0.0f, sgz = 0.0f, sc = 0.0f;
    float mx = 0.0f, my = 0.0f, mz = 0.0f, dv = 0.0f;
    const Records16 Gp(pos, n), Go(xold, n);
    auto load = [&](uint32_t j) { return Pair4{Gp[j], Go[j]}; };
    for_neighbors<Pair4, NB, kNone>(list, head, s, &cnt, load, [&](const Pair4 &qq) {
      const float4 &q = qq.a, &qo = qq.b;
      const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
      const float r2 = sq3(dx, dy, dz);
      S += density_term(r2, P);  // as k_density_lambda
      const float u = fmaxf(P.h2 - r2, 0.0f);
      const float w3 = u * u * u;
      mx = fmaf(-w3, dx, mx);
      my = fmaf(-w3, dy, my);
      mz = fmaf(-w3, dz, mz);
      const float r2c = fmaxf(r2, P.rmin2);
      const float ir = fast_rsq(r2c);
      const float hr = fmaf(-r2c, ir, P.h);
      const float hp = fmaxf(hr, 0.0f);
    const float g = hp * hp * ir;
      sgx = fmaf(g, dx, sgx);
      sgy = fmaf(g, dy, sgy);
      sgz = fmaf(g, dz, sgz);
      sc = fmaf(g * g, r2, sc);
      const float ex = (q.x - qo.x) - ux, ey = (q.y - qo.y) - uy, ez = (q.z - qo.z) - uz;
      dv = fmaf(g, fmaf(ez, dz, fmaf(ey, dy, ex * dx)), dv);
    });
    const float cr = density_constraint(S, cnt, P);
    rho = fmaf(cr, P.rest_density, P.rest_density);
    rho_io[s] = rho;
    err = fmaxf((rho - P.rest_density) * P.inv_rest_density, 0.0f);  // as k_density_lambda
    const float gc2 = P.lam_k2 * (sc + sq3(sgx, sgy, sgz));
    denom = gc2 + P.lambda_eps;
    lam0 = -fmaxf(cr, 0.0f) / denom;  // as k_density_lambda
    f[0] = (float)cnt * (1.0f / 32.0f);
    f[1] = cr;
    f[2] = -lam_prev[id_s[s]] * denom;
    f[3] = gc2 / denom;
    f[4] = P.div_k * dv;
    sdf_features(p.x, p.y, p.z, sdf_of<BATCH>(s, o, B), P, f + 5);
    const float mk = P.mWn / (rho * P.h);
    f[9] = mk * mx;
    f[10] = mk * my;
    f[11] = mk * mz;
  }
  raise_error(stats, 0, err, active);  // every lane gets here
  float lam = lam0;
  if (LOG) {
    if (active) {
      float4 *row = reinterpret_cast<float4 *>(feat + (size_t)s * kMlpPad);
      row[0] = make_float4(f[0], f[1], f[2], f[3]);
      row[1] = make_float4(f[4], f[5], f[6], f[7]);
      row[2] = make_float4(f[8], f[9], f[10], f[11]);
      row[3] = make_float4(denom, lam0, 0.0f, 0.0f);
    }
  } else {
    const float y = mlp_wave<false>(f, net);
    const float ymax = net->norm[kNormYMax], step = net->norm[kNormStep];
    const float ce = ymax > 0.0f ? fminf(fmaxf(y, 0.0f), ymax) : fmaxf(y, 0.0f);
    lam = lam0 - (step > 0.0f ? step : 1.0f) * ce / denom;
    if (active) plain[s] = make_float2(lam0, rho);  // for the plain fallback
  }
  if (active) {
    pos[s].w = lam;
    lam_acc[s] = 0.0f;
  }
}

// Warm start from the previous substep's multiplier (no network), after a
// plain density + lambda pass (rho, pos.w = lambda_0): keeps (lambda_0, rho)
// for the plain fallback and starts the solve from `scale` times the
// particle's accumulated multiplier of the previous substep (id order).
__global__ __launch_bounds__(kBlock) void k_warm_prev(uint32_t n, float4 *__restrict__ pos,
                                                      const float *__restrict__ rho,
                                                      const uint32_t *__restrict__ id_s,
                                                      const float *__restrict__ lam_prev,
                                                      float scale, float2 *__restrict__ plain,
                                                      float *__restrict__ lam_acc) {
  const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= n) return;
  plain[s] = make_float2(pos[s].w, rho[s]);
  pos[s].w = scale * lam_prev[id_s[s]];
  lam_acc[s] = 0.0f;
}

// Plain fallback of a warm start, after the density pass of iteration 1: if
// the predicted step left the maximum density error above the error before it,
// the particles return to their positions before the step with the plain
// first-iteration lambda and density, and iteration 1 proceeds from there.  The
// errors themselves stay as they are (blocks that start late decide by them too);
// STAT_FALLBACK tells their readers that iteration 1 has the pre-step error.
__global__ __launch_bounds__(kBlock) void k_warm_fallback(uint32_t n, uint32_t *stats,
                                                          const float4 *__restrict__ pre,
                                                          float4 *__restrict__ pos,
                                                          const float2 *__restrict__ plain,
                                                          float *__restrict__ rho,
                                                          float *__restrict__ lam_acc) {
  if (stats[STAT_CONVERGED]) return;
  // non-negative floats compare as their bit patterns
  if (max_error(stats, 1) <= max_error(stats, 0)) return;
  const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
  if (s < n) {
    const float4 p = pre[s];
    const float2 q = plain[s];
    pos[s] = make_float4(p.x, p.y, p.z, q.x);
    rho[s] = q.y;
    lam_acc[s] = 0.0f;
  }
  if (s == 0) stats[STAT_FALLBACK] = 1u;
}

// The same for a batch of scenes, scene by scene: a scene whose maximum error
// after the step (e1) exceeds the one before it (e0) is reverted.  A second
// kernel sets the iteration-1 error slot to the maximum over scenes of the
// error each scene continues from, and counts the reverted scenes.
__global__ __launch_bounds__(kBlock) void k_warm_fallback_scenes(
    uint32_t n, const uint32_t *stats, const uint16_t *__restrict__ scene_of,
    const uint32_t *__restrict__ e0, const uint32_t *__restrict__ e1,
    const float4 *__restrict__ pre, float4 *__restrict__ pos,
    const float2 *__restrict__ plain, float *__restrict__ rho, float *__restrict__ lam_acc) {
  if (stats[STAT_CONVERGED]) return;
  const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= n) return;
  const uint32_t k = scene_of[s];
  if (e1[k] <= e0[k]) return;  // non-negative floats compare as their bit patterns
  const float4 p = pre[s];
  const float2 q = plain[s];
  pos[s] = make_float4(p.x, p.y, p.z, q.x);
  rho[s] = q.y;
  lam_acc[s] = 0.0f;
}

__global__ __launch_bounds__(kBlock) void k_warm_fallback_stats(uint32_t nscenes,
                                                                uint32_t *stats,
                                                                const uint32_t *__restrict__ e0,
                                                                const uint32_t *__restrict__ e1) {
  if (stats[STAT_CONVERGED]) return;
  uint32_t m = 0u, reverted = 0u;
  for (uint32_t k = threadIdx.x; k < nscenes; k += blockDim.x) {
    const bool back = e1[k] > e0[k];
    m = max(m, back ? e0[k] : e1[k]);
    reverted += back ? 1u : 0u;
  }
  __shared__ uint32_t sm[kBlock], sr[kBlock];
  sm[threadIdx.x] = m;
  sr[threadIdx.x] = reverted;
  __syncthreads();
  for (uint32_t o = blockDim.x / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) {
      sm[threadIdx.x] = max(sm[threadIdx.x], sm[threadIdx.x + o]);
      sr[threadIdx.x] += sr[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x < kErrSlots) stats[err_word(1u, threadIdx.x)] = threadIdx.x == 0 ? sm[0] : 0u;
  if (threadIdx.x == 0) stats[STAT_FALLBACK] = sr[0];
}

// Keeps each particle's accumulated multiplier in particle-id order.
__global__ __launch_bounds__(kBlock) void k_scatter_lambda(uint32_t n,
                                                           const uint32_t *__restrict__ id_s,
                                                           const float *__restrict__ lam_acc,
                                                           float *__restrict__ lam_prev) {
  const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
  if (s < n) lam_prev[id_s[s]] = lam_acc[s];
}

// Dataset rows of a logged substep: every `every`-th sorted particle's
// feature row and its target R = -(Lambda - lambda_0) * (|grad C|^2 + eps), the
// part of the accumulated multiplier after the first iteration.
__global__ __launch_bounds__(kBlock) void k_warm_samples(uint32_t count, uint32_t every,
                                                         const float *__restrict__ feat,
                                                         const float *__restrict__ lam_acc,
                                                         float *__restrict__ x,
                                                         float *__restrict__ t) {
  const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= count) return;
  const size_t s = (size_t)k * every;
  const float4 *src = reinterpret_cast<const float4 *>(feat + s * kMlpPad);
  float4 *dst = reinterpret_cast<float4 *>(x + (size_t)k * kMlpPad);
  const float4 r3 = src[3];
  dst[0] = src[0];
  dst[1] = src[1];
  dst[2] = src[2];
  dst[3] = r3;
  t[k] = -(lam_acc[s] - r3.y) * r3.x;
}

// ---------------------------------------------------------------------------
// Velocity stages
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_velocity(uint32_t n, const float4 *__restrict__ pos,
                                                     const float4 *__restrict__ xold,
                                                     float4 *__restrict__ vel, DevParams P) {
  const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= n) return;
  vel[s] = velocity_of(pos[s], xold[s], P);
}

// ComputeSurfaceTension colour pass (particles.c:94-140), optionally fused
// with UpdateVelocities (own particle only).  DelWPoly(r)/r = norm (h^2-r^2)^2
// with r floored at 1e-4 h.
template <bool WITH_VELOCITY, int NB>
__global__ GATHER_BOUNDS(NB) void k_color(uint32_t n, uint32_t nblocks,
                                                  const float4 *__restrict__ pos,
                                                  const float4 *__restrict__ xold,
                                                  const uint32_t *__restrict__ list,
                                                  const uint4 *__restrict__ head, DevParams P,
                                                  float4 *__restrict__ vel,
                                                  float4 *__restrict__ color) {
  const uint32_t s = gather_index<NB>(nblocks);
  if (s >= n) return;
  const bool lead = gather_lead<NB>();
  const float4 p = pos[s];
  if (WITH_VELOCITY && lead) vel[s] = velocity_of(p, xold[s], P);
  int cnt;
  float a[3];
  const Records16 G(pos, n);
  sum_neighbors<float4, NB, NB >= 16 ? kIndices : kRaw, 3, 1>(
      list, head, s, &cnt, a, [&](uint32_t j) { return G[j]; }, [&](const float4 &q) {
        const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
        const float r2c = fmaxf(sq3(dx, dy, dz), P.rmin2);
        const float u = P.h2 - r2c;
        const float up = fmaxf(u, 0.0f);
        const float g = up * up * fast_rcp(q.w);
        return Terms<3>{{g, g, g}, {dx, dy, dz}};
      });
  if (lead)
    color[s] = make_float4(P.color_k * a[0], P.color_k * a[1], P.color_k * a[2], 0.0f);
}

// ComputeSurfaceTension force pass (particles.c:142-204): cohesion (Akinci
// spline C, particles.c:54-65) + curvature, v += dt F / rho_i in place.  The
// spline is computed without a branch per neighbour (the branch split the
// loop body and held 104 VGPRs at 8 gathers in flight, 89 without it); at 16
// gathers it runs 3 waves per SIMD without spilling.
template <int NB>
__global__ __launch_bounds__(kBlock, (NB) <= 16 ? 3 : 1) void k_surface(uint32_t n, uint32_t nblocks,
                                                    const float4 *__restrict__ pos,
                                                    const float4 *__restrict__ color,
                                                    const uint32_t *__restrict__ list,
                                                    const uint4 *__restrict__ head, DevParams P,
                                                    float4 *__restrict__ vel) {
  const uint32_t s = gather_index<NB>(nblocks);
  if (s >= n) return;
  const float4 p = pos[s];
  const float4 ci = color[s];
  int cnt;
  const float hh = 0.5f * P.h;
  float f[3];
  const Records16 Gp(pos, n), Gc(color, n);
  auto load = [&](uint32_t j) { return Pair4{Gp[j], Gc[j]}; };
  sum_neighbors<Pair4, NB, kNone, 3, 1>(list, head, s, &cnt, f, load, [&](const Pair4 &qc) {
    const float4 &q = qc.a, &cq = qc.b;
    const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
    const float r2c = fmaxf(sq3(dx, dy, dz), P.rmin2);
    const float ir = fast_rsq(r2c);
    const float r = r2c * ir;
    // (h - r) r, and 0 for r > h without a branch: max(h - r, 0) is h - r
    // exactly for r <= h, and for r > h the spline is 0 either way
    const float t = fmaxf(P.h - r, 0.0f) * r;
    const float t3 = t * t * t;
    const float spline = r <= hh ? fmaf(2.0f, t3, -P.h6_64) : t3;
    const float coh = P.coh_k * spline * ir;
    const float K = 2.0f * P.rest_density * fast_rcp(p.w + q.w);
    return Terms<3>{{K, K, K},
                    {fmaf(coh, dx, P.curv_k * (ci.x - cq.x)),
                     fmaf(coh, dy, P.curv_k * (ci.y - cq.y)),
                     fmaf(coh, dz, P.curv_k * (ci.z - cq.z))}};
  });
  if (!gather_lead<NB>()) return;
  const float k = P.dt / p.w;
  float4 v = vel[s];
  v.x = fmaf(k, f[0], v.x);
  v.y = fmaf(k, f[1], v.y);
  v.z = fmaf(k, f[2], v.z);
  vel[s] = v;
}

// ApplyViscosity (particles.c:383-459), reading v_old and writing v_new.  The
// distance keeps the reference's typo r^2 = dx^2 + dy^2 dz^2 (particles.c:439).
template <int NB>
__global__ __launch_bounds__(kBlock, (NB) <= 16 ? 3 : 1) void k_xsph(uint32_t n, uint32_t nblocks,
                                                 const float4 *__restrict__ pos,
                                                 const float4 *__restrict__ vin,
                                                 const uint32_t *__restrict__ list,
                                                 const uint4 *__restrict__ head, DevParams P,
                                                 float4 *__restrict__ vout) {
  const uint32_t s = gather_index<NB>(nblocks);
  if (s >= n) return;
  const float4 p = pos[s];
  const float4 vi = vin[s];
  int cnt;
  float a[3];
  const Records16 Gp(pos, n), Gv(vin, n);
  auto load = [&](uint32_t j) { return Pair4{Gp[j], Gv[j]}; };
  sum_neighbors<Pair4, NB, NB >= 16 ? kIndices : kNone, 3, 1>(list, head, s, &cnt, a, load, [&](const Pair4 &qv) {
    const float4 &q = qv.a, &vq = qv.b;
    const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
    const float u = P.h2 - fmaf(dy * dy * dz, dz, dx * dx);
    const float up = fmaxf(u, 0.0f);
    const float w = up * up * up * fast_rcp(q.w);
    return Terms<3>{{vq.x - vi.x, vq.y - vi.y, vq.z - vi.z}, {w, w, w}};
  });
  const float k = P.xsph_c * P.mWn;
  if (gather_lead<NB>())
    vout[s] = make_float4(fmaf(k, a[0], vi.x), fmaf(k, a[1], vi.y), fmaf(k, a[2], vi.z), 0.0f);
}

// ComputeVorticity (particles.c:207-283); aux = (omega, |omega|), and
// pw = (x*, |omega|) so that the confinement gather is one float4 per neighbour.
template <int NB>
__global__ __launch_bounds__(kBlock) void k_vorticity(uint32_t n, uint32_t nblocks,
                                                      const float4 *__restrict__ pos,
                                                      const float4 *__restrict__ vel,
                                                      const uint32_t *__restrict__ list,
                                                      const uint4 *__restrict__ head, DevParams P,
                                                      float4 *__restrict__ omega,
                                                      float4 *__restrict__ pw) {
  const uint32_t s = gather_index<NB>(nblocks);
  if (s >= n) return;
  const float4 p = pos[s];
  const float4 vi = vel[s];
  int cnt;
  float o[3];
  const Records16 Gp(pos, n), Gv(vel, n);
  auto load = [&](uint32_t j) { return Pair4{Gp[j], Gv[j]}; };
  sum_neighbors<Pair4, NB, kNone, 3, 2>(list, head, s, &cnt, o, load, [&](const Pair4 &qv) {
    const float4 &q = qv.a, &vq = qv.b;
    const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
    const float r2c = fmaxf(sq3(dx, dy, dz), P.rmin2);
    const float ir = fast_rsq(r2c);
    const float hr = fmaf(-r2c, ir, P.h);
    const float hp = fmaxf(hr, 0.0f);
    float g = hp * hp * ir;
    if (P.vort_model == 1) g *= fast_rcp(q.w);
    const float wx = g * dx, wy = g * dy, wz = g * dz;
    const float vx = vq.x - vi.x, vy = vq.y - vi.y, vz = vq.z - vi.z;
    return Terms<3, 2>{{-vz, vy, -vx, vz, -vy, vx}, {wy, wz, wz, wx, wx, wy}};
  });
  if (!gather_lead<NB>()) return;
  const float k = P.vort_model == 1 ? P.DelW_norm * P.mass : P.DelW_norm;
  const float ox = o[0] * k, oy = o[1] * k, oz = o[2] * k;
  const float wn = sqrtf(sq3(ox, oy, oz));
  omega[s] = make_float4(ox, oy, oz, wn);
  pw[s] = make_float4(p.x, p.y, p.z, wn);
}

// ApplyVorticityConfinement (particles.c:285-381): eta = sum |omega_j| gradW,
// N = eta / max(|eta|, 1e-4 h), v += dt eps (N x omega_i) / m.  When COMMIT
// is set the result is also UpdatePositions (particles.c:566-586): x* and v
// are scattered back to particle-id order.
template <bool COMMIT, int NB>
__global__ GATHER_BOUNDS(NB) void k_confine(
    uint32_t n, uint32_t nblocks, const float4 *__restrict__ pw,
    const float4 *__restrict__ omega, const uint32_t *__restrict__ list,
    const uint4 *__restrict__ head, DevParams P, const float4 *__restrict__ vin,
    float4 *__restrict__ vout, const uint32_t *__restrict__ id_s, float4 *__restrict__ x_can,
    float4 *__restrict__ v_can) {
  const uint32_t s = gather_index<NB>(nblocks);
  if (s >= n) return;
  const float4 p = pw[s];
  int cnt;
  float e[3];
  // only x_j and |omega_j| of the neighbour are needed
  const Records16 G(pw, n);
  sum_neighbors<float4, NB, NB >= 16 ? kIndices : kRaw, 3, 1>(
      list, head, s, &cnt, e, [&](uint32_t j) { return G[j]; }, [&](const float4 &q) {
        const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
        const float r2c = fmaxf(sq3(dx, dy, dz), P.rmin2);
        const float ir = fast_rsq(r2c);
        const float hr = fmaf(-r2c, ir, P.h);
        const float hp = fmaxf(hr, 0.0f);
        const float g = q.w * hp * hp * ir;
        return Terms<3>{{g, g, g}, {dx, dy, dz}};
      });
  if (!gather_lead<NB>()) return;
  const float ex = e[0] * P.DelW_norm, ey = e[1] * P.DelW_norm, ez = e[2] * P.DelW_norm;
  const float em = fmaxf(sqrtf(sq3(ex, ey, ez)), P.rmin);
  const float Nx = ex / em, Ny = ey / em, Nz = ez / em;
  const float4 wi = omega[s];
  float4 v = vin[s];
  v.x += P.conf_k * (Ny * wi.z - Nz * wi.y);
  v.y += P.conf_k * (Nz * wi.x - Nx * wi.z);
  v.z += P.conf_k * (Nx * wi.y - Ny * wi.x);
  v.w = 0.0f;
  if (COMMIT) {
    const uint32_t id = id_s[s];
    x_can[id] = make_float4(p.x, p.y, p.z, 0.0f);
    v_can[id] = v;
  } else {
    vout[s] = v;
  }
}

// UpdatePositions (particles.c:566-586) with the scatter to id order.
__global__ __launch_bounds__(kBlock) void k_commit(uint32_t n, const float4 *__restrict__ pos,
                                                   const float4 *__restrict__ vel,
                                                   const uint32_t *__restrict__ id_s,
                                                   float4 *__restrict__ x_can,
                                                   float4 *__restrict__ v_can) {
  const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= n) return;
  const uint32_t id = id_s[s];
  const float4 p = pos[s];
  const float4 v = vel[s];
  x_can[id] = make_float4(p.x, p.y, p.z, 0.0f);
  v_can[id] = make_float4(v.x, v.y, v.z, 0.0f);
}

// The statistics for the host: the flags and, a wave per iteration, its maximum.
__global__ __launch_bounds__(kBlock) void k_collect_stats(const uint32_t *__restrict__ stats,
                                                          uint32_t iterations,
                                                          uint32_t *__restrict__ out) {
  const uint32_t it = (blockIdx.x * kBlock + threadIdx.x) >> 6, lane = threadIdx.x & 63u;
  if (it == 0) out[lane] = stats[lane];
  if (it >= iterations) return;
  const uint32_t m = max_error(stats, (int)it);
  if (lane == 0) out[STAT_ERR0 + it] = m;
}

// The error words of iterations first..last, for density stages past those that the
// last search cleared.
__global__ __launch_bounds__(kBlock) void k_clear_errors(uint32_t *stats, uint32_t first,
                                                         uint32_t last) {
  const uint32_t e = blockIdx.x * kBlock + threadIdx.x;
  if (e < (last + 1u - first) * kErrSlots) stats[err_word(first, e)] = 0u;
}

// clear_substep_stats for a context without particles.
__global__ __launch_bounds__(kBlock) void k_substep_init(uint32_t *stats) {
  clear_substep_stats(stats, kMaxIters);
}

// Standalone CalculateParticleCollisions on SoA float arrays.
__global__ __launch_bounds__(kBlock) void k_collide_soa(uint32_t n, float *__restrict__ x,
                                                        float *__restrict__ y,
                                                        float *__restrict__ z, SdfDev o) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  float a = x[i], b = y[i], c = z[i];
  collide(a, b, c, o);
  x[i] = a;
  y[i] = b;
  z[i] = c;
}

// CalculateParticleCollisions_kernel on the reference's own FP64 arrays
// (obstacle_cuda.cu:56-116): the bounds test and the normalised coordinates
// in double against the double world box, the SDF arithmetic in FP32, and
// the FP32 push added to the double coordinate.
__global__ __launch_bounds__(kBlock) void k_collide_soa_f64(uint32_t n, double *__restrict__ x,
                                                            double *__restrict__ y,
                                                            double *__restrict__ z, SdfDev o,
                                                            SdfBox64 b) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const double xw = x[i], yw = y[i], zw = z[i];
  if (!(xw > b.lo[0] && xw < b.hi[0] && yw > b.lo[1] && yw < b.hi[1] && zw > b.lo[2] &&
        zw < b.hi[2]))
    return;
  const float u = (float)((xw - b.lo[0]) / (double)o.len[0]);
  const float v = (float)((yw - b.lo[1]) / (double)o.len[1]);
  const float w = (float)((zw - b.lo[2]) / (double)o.len[2]);
  float px, py, pz;
  if (!sdf_push(o, u, v, w, px, py, pz)) return;
  y[i] = yw + (double)py;
  x[i] = xw + (double)px;
  z[i] = zw + (double)pz;
}

// CalculateParticleCollisions over the sorted positions (after a k_dp_update
// without the fused push).  Only particles inside the obstacle's box are
// written.
template <bool BATCH>
__global__ __launch_bounds__(kBlock) void k_collide_sorted(uint32_t n, float4 *__restrict__ pos,
                                                           SdfDev o0, BatchDev B) {
  const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= n) return;
  const SdfDev &o = sdf_of<BATCH>(s, o0, B);
  if (!o.data) return;
  const float4 p = pos[s];
  if (!(p.x > o.wmin[0] && p.x < o.wmax[0] && p.y > o.wmin[1] && p.y < o.wmax[1] &&
        p.z > o.wmin[2] && p.z < o.wmax[2]))
    return;
  float x = p.x, y = p.y, z = p.z;
  collide(x, y, z, o);
  if (x != p.x || y != p.y || z != p.z) pos[s] = make_float4(x, y, z, p.w);
}

// Max density error per scene of a batch, from the last density pass (rho in
// sorted order; a scene's particles are one index range there).  One block
// per chunk of at most kSceneChunk particles of one scene (the chunk table is
// built with the batch): the block reduces its chunk and issues one atomic,
// at most a few dozen per scene.  With one atomic per wave, as first written,
// the ~440 waves of a 28k-particle scene serialised on its word (0.96 ms for
// 512 scenes, 14.3M particles, against ~0.01 ms of traffic).
__global__ __launch_bounds__(kBlock) void k_scene_errors(const uint4 *__restrict__ chunks,
                                                         const float *__restrict__ rho,
                                                         DevParams P, uint32_t *err_bits) {
  __shared__ float wmax[kBlock / kWave];
  const uint4 ch = chunks[blockIdx.x];  // scene, first, end
  float m = 0.0f;
  for (uint32_t i = ch.y + threadIdx.x; i < ch.z; i += kBlock)
    m = fmaxf(m, (rho[i] - P.rest_density) * P.inv_rest_density);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    float b = wmax[0];
    for (int w = 1; w < kBlock / kWave; ++w) b = fmaxf(b, wmax[w]);
    if (b > 0.0f) atomicMax(&err_bits[ch.x], __float_as_uint(b));
  }
}

__global__ __launch_bounds__(kBlock) void k_fill_words(uint32_t n, uint32_t *p, uint32_t v) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = v;
}

// FP64 kinetic energy: one partial sum per block into out[blockIdx.x] (the
// caller adds them in block order, so the result does not depend on the order
// in which blocks finish, as it did with one atomic per block).
__global__ __launch_bounds__(kBlock) void k_kinetic_energy(uint32_t n,
                                                           const float4 *__restrict__ v,
                                                           double half_m, double *out) {
  __shared__ double part[kBlock / 64];
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  double e = 0.0;
  if (i < n) {
    const float4 u = v[i];
    e = half_m * ((double)u.x * u.x + (double)u.y * u.y + (double)u.z * u.z);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) e += __shfl_xor(e, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = e;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < kBlock / 64; ++w) t += part[w];
    out[blockIdx.x] = t;  // summed in block order on the host
  }
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
// Gathers in flight per wave of a gather kernel where neither the autotuner nor
// the caller chose: four lanes a particle up to kQuadMax; 8 where the chip holds all
// or most waves at once anyway, which lets more of them in per SIMD (70 VGPRs); 16
// beyond.  Measured (us, 64 threads a block, events included), 16 / 8: density 439k
// particles 25.6 / 23.0, 2.1M 87.4 / 85.8, 3.4M 145.9 / 154.9; delta p 439k 22.4 /
// 21.1, 1M 42.6 / 41.3, 1.6M 58.5 / 58.8; XSPH 133k 14.7 / 13.8, 439k 33.8 / 33.3,
// 1M 69.9 / 72.0; surface 681k 48.8 / 50.6, 1M 70.1 / 76.8.
static inline int tuned_depth(const sph_ctx *c, int kernel) {
  const int d = c->tune.depth[kernel];
  if (d) return d;
  if (c->n <= kQuadMax) return kQuad;
  int most = 1 << 19;
  if (kernel == K_DENSITY_LAMBDA || kernel == K_DENSITY || kernel == K_LAMBDA) most = 1 << 21;
  if (kernel == K_DP || kernel == K_DP_UPDATE) most = 1 << 20;
  return c->n <= most ? 8 : 16;
}

template <typename F>
static inline void with_depth(int depth, F &&f) {
  if (depth == 32)
    f(std::integral_constant<int, 32>{});
  else if (depth == 8)
    f(std::integral_constant<int, 8>{});
  else if (depth == kQuad)
    f(std::integral_constant<int, kQuad>{});
  else
    f(std::integral_constant<int, 16>{});
}

// Threads per block of a gather kernel where neither the autotuner nor the
// caller chose.  A block of one wave frees its place as soon as that wave ends
// and, of few particles, spreads the waves over the CUs (a wave's gathers keep a
// vector L1 busy): surface 10.8 -> 8.8 us at 4k particles, 79.2 -> 70.1 at 1M
// (256 / 64 threads, events included), XSPH 10.2 -> 7.9 and 75.3 -> 69.9, delta p
// 8.5 -> 7.7 and 46.1 -> 42.5, density 9.3 -> 8.4 and 50.4 -> 46.9.  At 8.4M the
// neighbouring waves of a larger block share more lines: colour 363 / 370,
// confinement 394 / 400, delta p 327 (128) / 329, but surface 616 / 597 and density
// 352 / 343.
static inline uint32_t tuned_block(const sph_ctx *c, int kernel) {
  const uint32_t b = c->tune.block[kernel];
  if (b) return b;
  switch (kernel) {
    case K_BUILD_LISTS: return kBlock;
    case K_COLOR: case K_XSPH: case K_VORTICITY: case K_CONFINE:
      return c->n <= (1 << 21) ? 64 : kBlock;
    case K_DP: case K_DP_UPDATE: return c->n <= (1 << 21) ? 64 : 128;
    default: return 64;  // density, surface, warm start
  }
}

// Depth, threads per block and blocks of a gather kernel's launch; the threads as
// chosen for block_of.
struct Gather {
  int depth;
  uint32_t threads, blocks;
};
static inline Gather gather_launch(const sph_ctx *c, int kernel, int block_of) {
  const int depth = tuned_depth(c, kernel);
  if (depth == kQuad) return {depth, kWave, blocks_for(c->n, kWave / 4)};
  const uint32_t t = tuned_block(c, block_of);
  return {depth, t, blocks_for(c->n, t)};
}

#define LAUNCH_TIMED(ctx, kid, grid, ...)                               \
  do {                                                                  \
    hipEvent_t ev_ = nullptr;                                           \
    prof_begin(ctx, kid, &ev_);                                         \
    __VA_ARGS__;                                                        \
    prof_end(ctx, kid, ev_);                                            \
  } while (0)

int launch_gravity(sph_ctx *c) {
  const uint32_t n = c->n;
  if (!n) return SPH_OK;
  LAUNCH_TIMED(c, K_GRAVITY, 0,
               k_gravity<<<blocks_for(n), kBlock, 0, c->stream>>>(n, c->v_can, c->dev));
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

int launch_predict(sph_ctx *c) {
  const uint32_t n = c->n;
  if (!n) return SPH_OK;
  const BatchDev B = c->batch();
  if (c->nscenes)
    LAUNCH_TIMED(c, K_PREDICT, 0,
                 k_predict<true><<<blocks_for(n), kBlock, 0, c->stream>>>(
                     n, c->x_can, c->v_can, c->xs_can, c->dev, B));
  else
    LAUNCH_TIMED(c, K_PREDICT, 0,
                 k_predict<false><<<blocks_for(n), kBlock, 0, c->stream>>>(
                     n, c->x_can, c->v_can, c->xs_can, c->dev, B));
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

// Hash (fused with gravity+predict when `fused`), sort, cell tables, reorder,
// lists: FindAllNeighbors (neighbors.c:68-75) in sorted space.
int launch_neighbor_search(sph_ctx *c, bool fused) {
  const uint32_t n = c->n;
  hipStream_t s = c->stream;
  const BatchDev B = c->batch();
  // the stage calls may run any number of density passes
  const uint32_t last = (uint32_t)(fused ? c->P.solve_iterations : kMaxIters);
  c->err_cleared = (int)last;
  if (n) {
    if (fused && c->nscenes) {
      LAUNCH_TIMED(c, K_PREDICT_HASH, 0,
                   k_predict_hash<true><<<blocks_for(n), kBlock, 0, s>>>(
                       n, c->x_can, c->v_can, c->xs_can, c->keys, c->cell_rank, c->cell_count,
                       c->dev, c->stats, last, B));
    } else if (fused) {
      LAUNCH_TIMED(c, K_PREDICT_HASH, 0,
                   k_predict_hash<false><<<blocks_for(n), kBlock, 0, s>>>(
                       n, c->x_can, c->v_can, c->xs_can, c->keys, c->cell_rank, c->cell_count,
                       c->dev, c->stats, last, B));
    } else if (c->nscenes) {
      LAUNCH_TIMED(c, K_HASH, 0,
                   k_hash<true><<<blocks_for(n), kBlock, 0, s>>>(
                       n, c->xs_can, c->keys, c->cell_rank, c->cell_count, c->dev, c->stats, last,
                       B));
    } else {
      LAUNCH_TIMED(c, K_HASH, 0,
                   k_hash<false><<<blocks_for(n), kBlock, 0, s>>>(
                       n, c->xs_can, c->keys, c->cell_rank, c->cell_count, c->dev, c->stats, last,
                       B));
    }
  } else {
    k_substep_init<<<1, kBlock, 0, s>>>(c->stats);
  }
  SPH_HIP(hipGetLastError());
  // cell_start[c] = #keys < c (lower bound), cell_start[cells] = n
  const int rc = scan(c->cell_count, c->cell_start, c->cells, false, true, &c->scan, s, c);
  if (rc) return rc;
  c->pos = c->pos_a;
  if (n) {
    LAUNCH_TIMED(c, K_PLACE, 0,
                 k_place<<<blocks_for(n), kBlock, 0, s>>>(n, c->keys, c->cell_rank, c->cell_start,
                                                          c->slots, c->cell_count));
    LAUNCH_TIMED(c, K_REORDER, 0,
                 k_reorder<<<blocks_for(n), kBlock, 0, s>>>(
                     n, c->slots, c->cell_start, c->xs_can, c->x_can, c->key_s, c->id_s, c->pos,
                     c->xold, c->fixed_xy, c->fixed_z, c->dev.fixed_scale));
    SPH_HIP(hipGetLastError());
  }
  if (n) {
    const int wide = c->tune.wide_lists ? 1 : 0;
    if (n <= kRowBuildMax) {
      const uint32_t groups = blocks_for(n, kWave);
#define BUILD_ROWS(BAT, ROWS)                                                                  \
  LAUNCH_TIMED(c, K_BUILD_LISTS, 0,                                                            \
               (k_build_rows<BAT, ROWS><<<groups, 9 / ROWS * kWave, 0, s>>>(                   \
                   n, c->pos, c->fixed_xy, c->fixed_z, c->key_s, c->cell_start, c->dev, c->list,  \
                   c->list_head, c->stats, c->pair_partial, wide, B)))
      if (n <= kOneRowBuildMax) {
        if (c->nscenes) BUILD_ROWS(true, 1); else BUILD_ROWS(false, 1);
      } else {
        if (c->nscenes) BUILD_ROWS(true, 3); else BUILD_ROWS(false, 3);
      }
#undef BUILD_ROWS
      c->pair_blocks = groups;
    } else {
      const uint32_t bs = tuned_block(c, K_BUILD_LISTS);
      const uint32_t nb = blocks_for(n, bs);
      if (c->nscenes)
        LAUNCH_TIMED(c, K_BUILD_LISTS, 0,
                     k_build_lists<true><<<nb, bs, kLdsHits * bs * sizeof(uint16_t), s>>>(
                         n, nb, c->pos, c->fixed_xy, c->fixed_z, c->key_s, c->cell_start, c->dev,
                         c->list, c->list_head, c->stats, c->pair_partial, wide, B));
      else
        LAUNCH_TIMED(c, K_BUILD_LISTS, 0,
                     k_build_lists<false><<<nb, bs, kLdsHits * bs * sizeof(uint16_t), s>>>(
                         n, nb, c->pos, c->fixed_xy, c->fixed_z, c->key_s, c->cell_start, c->dev,
                         c->list, c->list_head, c->stats, c->pair_partial, wide, B));
      c->pair_blocks = nb;
    }
    SPH_HIP(hipGetLastError());
  }
  c->vel = c->vel_a;
  c->sorted_valid = true;
  c->lists_valid = true;
  return SPH_OK;
}

static float stiffness_scale(const sph_ctx *c, int substep) {
  // particles.c:693-694, 742-744: stiffness * m * DelW_norm / rho0
  const double st = 1.0 - pow(1.0 - c->P.stiffness_k, 1.0 / (double)substep);
  return (float)(st * c->P.rest_mass * (-45.0 / (M_PI * pow(c->P.smoothing_radius, 6.0))) /
                 c->P.rest_density);
}

int launch_density(sph_ctx *c, int mode, int err_slot) {
  const uint32_t n = c->n;
  if (!n) return SPH_OK;
  const int kernel = mode == 2 ? K_LAMBDA : mode == 3 ? K_DENSITY : K_DENSITY_LAMBDA;
  const Gather g = gather_launch(c, kernel, K_DENSITY_LAMBDA);
  const uint32_t bs = g.threads, nb = g.blocks;
  hipStream_t s = c->stream;
  if (mode == 0)
    with_depth(g.depth, [&](auto D_) {
      constexpr int NBv = decltype(D_)::value;
      LAUNCH_TIMED(c, K_DENSITY_LAMBDA, 0,
                   k_density_lambda<0, NBv><<<nb, bs, 0, s>>>(
                       n, nb, c->pos, c->list, c->list_head, c->dev, c->rho, nullptr, c->stats,
                       err_slot, c->P.density_tolerance > 0, 0, nullptr));
    });
  else if (mode == 4)  // density and lambda in one gather: rho into w, (x*, lambda) aside
    with_depth(g.depth, [&](auto D_) {
      constexpr int NBv = decltype(D_)::value;
      LAUNCH_TIMED(c, K_DENSITY_LAMBDA, 0,
                   k_density_lambda<0, NBv><<<nb, bs, 0, s>>>(
                       n, nb, c->pos, c->list, c->list_head, c->dev, c->rho, c->cstage, c->stats,
                       err_slot, 0, 1, c->pos == c->pos_a ? c->pos_b : c->pos_a));
    });
  else if (mode == 3)  // final density of a capped tolerance loop: rho also into w
    with_depth(g.depth, [&](auto D_) {
      constexpr int NBv = decltype(D_)::value;
      LAUNCH_TIMED(c, K_DENSITY, 0,
                   k_density_lambda<1, NBv><<<nb, bs, 0, s>>>(
                       n, nb, c->pos, c->list, c->list_head, c->dev, c->rho, c->cstage, c->stats,
                       err_slot, 1, 1, nullptr));
    });
  else
    with_depth(g.depth, [&](auto D_) {
      constexpr int NBv = decltype(D_)::value;
      LAUNCH_TIMED(c, K_LAMBDA, 0,
                   k_density_lambda<2, NBv><<<nb, bs, 0, s>>>(
                       n, nb, c->pos, c->list, c->list_head, c->dev, c->rho, c->cstage, c->stats,
                       -1, 0, 0, nullptr));
    });
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

int launch_dp(sph_ctx *c, int substep, float4 *xnext) {
  const uint32_t n = c->n;
  if (!n) return SPH_OK;
  const Gather g = gather_launch(c, K_DP, K_DP);
  const uint32_t bs = g.threads, nb = g.blocks;
  const float scale = stiffness_scale(c, substep);
  const BatchDev B = c->batch();
  with_depth(g.depth, [&](auto D_) {
    constexpr int NBv = decltype(D_)::value;
    if (c->nscenes)
      LAUNCH_TIMED(c, K_DP, 0,
                   (k_dp<true, NBv><<<nb, bs, 0, c->stream>>>(n, nb, c->pos, c->list,
                                                             c->list_head, c->dev, scale,
                                                             c->dpbuf, xnext, c->rho, c->sdf, B)));
    else
      LAUNCH_TIMED(c, K_DP, 0,
                   (k_dp<false, NBv><<<nb, bs, 0, c->stream>>>(n, nb, c->pos, c->list,
                                                              c->list_head, c->dev, scale,
                                                              c->dpbuf, xnext, c->rho, c->sdf,
                                                              B)));
  });
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

int launch_position_stars(sph_ctx *c) {
  const uint32_t n = c->n;
  if (!n) return SPH_OK;
  if (c->nscenes)
    LAUNCH_TIMED(c, K_POS_STARS, 0,
                 k_position_stars<true><<<blocks_for(n), kBlock, 0, c->stream>>>(
                     n, c->pos, c->dpbuf, c->rho, c->dev, c->sdf, c->batch()));
  else
    LAUNCH_TIMED(c, K_POS_STARS, 0,
                 k_position_stars<false><<<blocks_for(n), kBlock, 0, c->stream>>>(
                     n, c->pos, c->dpbuf, c->rho, c->dev, c->sdf, c->batch()));
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

static float stiffness_unitless(const sph_ctx *c, int substep) {
  return (float)(1.0 - pow(1.0 - c->P.stiffness_k, 1.0 / (double)substep));
}

bool finishes_in_update(const sph_ctx *c) {
  const bool obstacle = c->nscenes ? c->batch_sdf != nullptr : c->sdf.data != nullptr;
  return !c->P.surface_tension && !c->P.viscosity && !c->P.vorticity &&
         !(obstacle && c->tune.split_collide);
}

int launch_dp_update(sph_ctx *c, int substep, int err_slot, bool accumulate, bool finish) {
  const uint32_t n = c->n;
  if (finish) c->vel = c->vel_a;
  if (!n) return SPH_OK;
  const Gather g = gather_launch(c, K_DP_UPDATE, K_DP_UPDATE);
  const uint32_t bs = g.threads, nb = g.blocks;
  float4 *out = (c->pos == c->pos_a) ? c->pos_b : c->pos_a;
  float *acc = accumulate ? c->lam_acc : nullptr;
  const float scale = stiffness_scale(c, substep), stiff = stiffness_unitless(c, substep);
  const float tol = (float)c->P.density_tolerance;
  const int fallback_slot = err_slot == 1 && !c->nscenes ? 0 : err_slot;
  const BatchDev B = c->batch();
  const bool obstacle = c->nscenes ? c->batch_sdf != nullptr : c->sdf.data != nullptr;
  const bool split = obstacle && c->tune.split_collide;
  FinishDev fin;
  if (finish) fin = {c->xold, c->vel, c->id_s, c->x_can, c->v_can};
#define DP_UPDATE(COL, BAT)                                                                 \
  with_depth(g.depth, [&](auto D_) {                                                        \
    constexpr int NBv = decltype(D_)::value;                                                \
    LAUNCH_TIMED(c, K_DP_UPDATE, 0,                                                         \
                 (k_dp_update<COL, BAT, NBv><<<nb, bs, 0, c->stream>>>(                      \
                     n, nb, c->pos, out, c->rho, c->list, c->list_head, c->dev, scale, c->sdf, \
                     c->stats, err_slot, fallback_slot, tol, acc, stiff, B, fin)));         \
  })
  if (c->nscenes) {
    if (split) DP_UPDATE(false, true); else DP_UPDATE(true, true);
  } else {
    if (split) DP_UPDATE(false, false); else DP_UPDATE(true, false);
  }
#undef DP_UPDATE
  SPH_HIP(hipGetLastError());
  if (split) {
    if (c->nscenes)
      LAUNCH_TIMED(c, K_COLLIDE, 0,
                   k_collide_sorted<true><<<blocks_for(n), kBlock, 0, c->stream>>>(
                       n, out, c->sdf, B));
    else
      LAUNCH_TIMED(c, K_COLLIDE, 0,
                   k_collide_sorted<false><<<blocks_for(n), kBlock, 0, c->stream>>>(
                       n, out, c->sdf, B));
    SPH_HIP(hipGetLastError());
  }
  c->pos = out;
  return SPH_OK;
}

int launch_warm_lambda(sph_ctx *c, bool log) {
  const uint32_t n = c->n;
  if (!n) return SPH_OK;
  const uint32_t bs = tuned_block(c, K_WARM_LAMBDA);
  const uint32_t nb = blocks_for(n, bs);
  const BatchDev B = c->batch();
  float2 *plain = reinterpret_cast<float2 *>(c->dpbuf);
#define WARM(LOG, BAT)                                                                      \
  LAUNCH_TIMED(c, K_WARM_LAMBDA, 0,                                                         \
               (k_warm_lambda<LOG, BAT><<<nb, bs, 0, c->stream>>>(                       \
                   n, nb, c->pos, c->xold, c->list, c->list_head, c->dev, c->rho, c->stats,   \
                   c->id_s, c->lam_prev, c->sdf, LOG ? nullptr : c->warm_net, c->lam_acc,   \
                   LOG ? c->feat : nullptr, LOG ? nullptr : plain, B)))
  if (c->nscenes) {
    if (log) WARM(true, true); else WARM(false, true);
  } else {
    if (log) WARM(true, false); else WARM(false, false);
  }
#undef WARM
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

int launch_warm_prev(sph_ctx *c) {
  const uint32_t n = c->n;
  if (!n) return SPH_OK;
  int rc = launch_density(c, 0, 0);
  if (rc) return rc;
  LAUNCH_TIMED(c, K_AUX, 0,
               k_warm_prev<<<blocks_for(n), kBlock, 0, c->stream>>>(
                   n, c->pos, c->rho, c->id_s, c->lam_prev, c->warm_prev_scale,
                   reinterpret_cast<float2 *>(c->dpbuf), c->lam_acc));
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

int launch_warm_fallback(sph_ctx *c, const float4 *pre_warm) {
  const uint32_t n = c->n;
  if (!n) return SPH_OK;
  if (c->nscenes) {
    // per scene; scene_err0 / scene_err hold the errors before and after the step
    LAUNCH_TIMED(c, K_AUX, 0,
                 k_warm_fallback_scenes<<<blocks_for(n), kBlock, 0, c->stream>>>(
                     n, c->stats, c->scene_of, c->scene_err0, c->scene_err, pre_warm, c->pos,
                     reinterpret_cast<const float2 *>(c->dpbuf), c->rho, c->lam_acc));
    SPH_HIP(hipGetLastError());
    k_warm_fallback_stats<<<1, kBlock, 0, c->stream>>>((uint32_t)c->nscenes, c->stats,
                                                       c->scene_err0, c->scene_err);
    SPH_HIP(hipGetLastError());
    return SPH_OK;
  }
  LAUNCH_TIMED(c, K_AUX, 0,
               k_warm_fallback<<<blocks_for(n), kBlock, 0, c->stream>>>(
                   n, c->stats, pre_warm, c->pos, reinterpret_cast<const float2 *>(c->dpbuf),
                   c->rho, c->lam_acc));
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

int launch_scene_errors(sph_ctx *c, uint32_t *dst) {
  const uint32_t ns = (uint32_t)c->nscenes;
  if (!ns) return SPH_OK;
  if (!dst) dst = c->scene_err;
  k_fill_words<<<blocks_for(ns), kBlock, 0, c->stream>>>(ns, dst, 0u);
  SPH_HIP(hipGetLastError());
  if (c->n && c->nchunks) {
    k_scene_errors<<<c->nchunks, kBlock, 0, c->stream>>>(c->scene_chunks, c->rho, c->dev, dst);
    SPH_HIP(hipGetLastError());
  }
  return SPH_OK;
}

int launch_scatter_lambda(sph_ctx *c) {
  const uint32_t n = c->n;
  if (!n) return SPH_OK;
  LAUNCH_TIMED(c, K_AUX, 0,
               k_scatter_lambda<<<blocks_for(n), kBlock, 0, c->stream>>>(n, c->id_s,
                                                                         c->lam_acc,
                                                                         c->lam_prev));
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

int launch_warm_samples(sph_ctx *c, float *x, float *t, uint32_t count, int every) {
  if (!count) return SPH_OK;
  k_warm_samples<<<blocks_for(count), kBlock, 0, c->stream>>>(count, (uint32_t)every, c->feat,
                                                              c->lam_acc, x, t);
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}


int launch_velocity(sph_ctx *c) {
  const uint32_t n = c->n;
  c->vel = c->vel_a;
  if (!n) return SPH_OK;
  LAUNCH_TIMED(c, K_VELOCITY, 0,
               k_velocity<<<blocks_for(n), kBlock, 0, c->stream>>>(n, c->pos, c->xold, c->vel,
                                                                   c->dev));
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

int launch_color(sph_ctx *c, bool with_velocity) {
  const uint32_t n = c->n;
  if (with_velocity) c->vel = c->vel_a;
  if (!n) return SPH_OK;
  const Gather g = gather_launch(c, K_COLOR, K_COLOR);
  const uint32_t bs = g.threads, nb = g.blocks;
  if (with_velocity)
    with_depth(g.depth, [&](auto D_) {
      constexpr int NBv = decltype(D_)::value;
      LAUNCH_TIMED(c, K_COLOR, 0,
                   k_color<true, NBv><<<nb, bs, 0, c->stream>>>(n, nb, c->pos, c->xold, c->list,
                                                               c->list_head, c->dev, c->vel,
                                                               c->aux));
    });
  else
    with_depth(g.depth, [&](auto D_) {
      constexpr int NBv = decltype(D_)::value;
      LAUNCH_TIMED(c, K_COLOR, 0,
                   k_color<false, NBv><<<nb, bs, 0, c->stream>>>(n, nb, c->pos, c->xold, c->list,
                                                                c->list_head, c->dev, c->vel,
                                                                c->aux));
    });
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

int launch_surface(sph_ctx *c) {
  const uint32_t n = c->n;
  if (!n) return SPH_OK;
  const Gather g = gather_launch(c, K_SURFACE, K_SURFACE);
  const uint32_t bs = g.threads, nb = g.blocks;
  with_depth(g.depth, [&](auto D_) {
    constexpr int NBv = decltype(D_)::value;
    LAUNCH_TIMED(c, K_SURFACE, 0,
                 k_surface<NBv><<<nb, bs, 0, c->stream>>>(n, nb, c->pos, c->aux, c->list,
                                                         c->list_head, c->dev, c->vel));
  });
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

int launch_xsph(sph_ctx *c) {
  const uint32_t n = c->n;
  float4 *out = (c->vel == c->vel_a) ? c->vel_b : c->vel_a;
  if (n) {
    const Gather g = gather_launch(c, K_XSPH, K_XSPH);
    const uint32_t bs = g.threads, nb = g.blocks;
    with_depth(g.depth, [&](auto D_) {
      constexpr int NBv = decltype(D_)::value;
      LAUNCH_TIMED(c, K_XSPH, 0,
                   k_xsph<NBv><<<nb, bs, 0, c->stream>>>(n, nb, c->pos, c->vel, c->list,
                                                        c->list_head, c->dev, out));
    });
    SPH_HIP(hipGetLastError());
  }
  c->vel = out;
  return SPH_OK;
}

int launch_vorticity(sph_ctx *c) {
  const uint32_t n = c->n;
  if (!n) return SPH_OK;
  const Gather g = gather_launch(c, K_VORTICITY, K_VORTICITY);
  const uint32_t bs = g.threads, nb = g.blocks;
  with_depth(g.depth, [&](auto D_) {
    constexpr int NBv = decltype(D_)::value;
    LAUNCH_TIMED(c, K_VORTICITY, 0,
                 k_vorticity<NBv><<<nb, bs, 0, c->stream>>>(n, nb, c->pos, c->vel, c->list,
                                                           c->list_head, c->dev, c->aux,
                                                           c->pw));
  });
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

int launch_confine(sph_ctx *c, bool commit) {
  const uint32_t n = c->n;
  float4 *out = (c->vel == c->vel_a) ? c->vel_b : c->vel_a;
  if (n) {
    const Gather g = gather_launch(c, K_CONFINE, K_CONFINE);
    const uint32_t bs = g.threads, nb = g.blocks;
    if (commit)
      with_depth(g.depth, [&](auto D_) {
        constexpr int NBv = decltype(D_)::value;
        LAUNCH_TIMED(c, K_CONFINE, 0,
                       k_confine<true, NBv><<<nb, bs, 0, c->stream>>>(
                           n, nb, c->pw, c->aux, c->list, c->list_head, c->dev, c->vel, out,
                           c->id_s, c->x_can, c->v_can));
      });
    else
      with_depth(g.depth, [&](auto D_) {
        constexpr int NBv = decltype(D_)::value;
        LAUNCH_TIMED(c, K_CONFINE, 0,
                       k_confine<false, NBv><<<nb, bs, 0, c->stream>>>(
                           n, nb, c->pw, c->aux, c->list, c->list_head, c->dev, c->vel, out,
                           c->id_s, c->x_can, c->v_can));
      });
    SPH_HIP(hipGetLastError());
  }
  if (!commit) c->vel = out;
  return SPH_OK;
}

int launch_commit(sph_ctx *c) {
  const uint32_t n = c->n;
  if (!n) return SPH_OK;
  LAUNCH_TIMED(c, K_COMMIT, 0,
               k_commit<<<blocks_for(n), kBlock, 0, c->stream>>>(n, c->pos, c->vel, c->id_s,
                                                                 c->x_can, c->v_can));
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

int launch_clear_errors(sph_ctx *c, int last) {
  if (last <= c->err_cleared) return SPH_OK;
  const uint32_t first = (uint32_t)(c->err_cleared + 1);
  k_clear_errors<<<blocks_for((last + 1u - first) * kErrSlots), kBlock, 0, c->stream>>>(
      c->stats, first, (uint32_t)last);
  SPH_HIP(hipGetLastError());
  c->err_cleared = last;
  return SPH_OK;
}

int launch_collect_stats(sph_ctx *c, uint32_t *out) {
  static_assert(STAT_ERR0 == kWave, "a wave copies the flags");
  constexpr uint32_t its = kMaxIters + 1;
  k_collect_stats<<<blocks_for(its, kBlock / kWave), kBlock, 0, c->stream>>>(c->stats, its,
                                                                            out);
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

int launch_collide_soa(float *x, float *y, float *z, uint32_t n, const SdfDev &o,
                       hipStream_t s) {
  if (!n) return SPH_OK;
  k_collide_soa<<<blocks_for(n), kBlock, 0, s>>>(n, x, y, z, o);
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

int launch_collide_soa_f64(double *x, double *y, double *z, uint32_t n, const SdfDev &o,
                           const SdfBox64 &b, hipStream_t s) {
  if (!n) return SPH_OK;
  k_collide_soa_f64<<<blocks_for(n), kBlock, 0, s>>>(n, x, y, z, o, b);
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

int launch_kinetic_energy(sph_ctx *c, double *out_dev) {
  if (c->n)
    k_kinetic_energy<<<blocks_for(c->n), kBlock, 0, c->stream>>>(
        c->n, c->v_can, 0.5 * c->P.rest_mass, out_dev);
  SPH_HIP(hipGetLastError());
  return SPH_OK;
}

}  // namespace sph
