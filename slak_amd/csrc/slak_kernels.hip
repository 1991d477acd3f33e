// HIP kernels of the Catmull-Clark level pipeline for gfx950 (MI355X).
//
// First level (the caller's mesh):
//   gather        check the input and bring corners into position order
//                 (sortKeyValuePairsSegmentedInPlace, LAKCatmullClarkKernels.cuh:147-180);
//                 valence per vertex (spmv_right with ones, LAKCatmullClarkImpl.cu:347-356)
//                 and the corners of M^T's rows into fixed slots per vertex
//   symbolic      row sizing of the mapped SpGEMM -> edges owned per vertex;
//                 corner and edge counts summed per tile of vertices
//   number        offsets from those sums (scan_exclusive, cub_wrappers.cuh:30-43),
//                 M^T's rows sorted, with their in-neighbours (csr2cscEx2,
//                 LAKCatmullClarkImpl.cu:381-423); mapped SpGEMM rows -> E numbering:
//                 edge id and twin of every corner's half-edge, boundary flags
//   first_small   all of it in one block for a small mesh
// Every level:
//   face points   left mapped SpMV fp = M^T P / order (spmv.cuh:64-81)
//   refine        per corner: edge points (calculateInternal/ExternalEdgepoints),
//                 refined quads (refineTopology[Homogeneous],
//                 LAKCatmullClarkKernels.cuh:320-431) and, for a level that
//                 feeds another, the refined mesh's twins, edge ids and the
//                 face- and edge-point rows of its M^T, all in closed form
//   vertex        per vertex: the two right SpMVs of the vertex update
//                 (LAKCatmullClarkImpl.cu:200-235) and boundary rule
//                 (LAKCatmullClarkKernels.cuh:464-511); the vertex rows of the
//                 refined M^T
// Last levels of a chain:
//   final         from the mesh M two levels back (quads, or the caller's
//                 polygons): the output quads, edge, face and vertex points of
//                 the level (or its positions only, for the level before it);
//                 several meshes per launch through a table
//   final_deep    the output level of a closed LAK mesh from three levels back
//   LAK form      several meshes: the output level's ptr / vals in a launch
//                 of their own (createQuadColPtr / createQuadVals)
// All kernels are pull-based and atomic-free except the integer valence
// count and row slots, whose result does not depend on atomic order,
// so every output is bitwise deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdlib>
#include <mutex>
#include <type_traits>
#include <vector>

#include "slak_device.hpp"
#include "slak_internal.hpp"

namespace slak {

namespace {

constexpr int kBlock = kBlockItems;

// Workgroups are dispatched round-robin over the 8 XCDs, each with its own L2.
// With the remap, consecutive tiles (which gather from neighbouring parts of
// the mesh) land on the same XCD: XCD x runs the x-th eighth of the grid in
// order. Selected once per process by the bit mask SLAK_XCD_REMAP: bit 0 for
// the level kernels that hand on a structure, bit 1 for k_final (its gathers
// then stay in one L2: 136 -> 113 us on the 4-level chain of the 256x128
// torus), bit 2 for the other level kernels, bit 3 for every other kernel.
// For the level kernels it pays together with vertex items in class runs
// (alone it measured 10-25 % slower). Default 3.
__device__ int g_xcd_remap;
constexpr int kRemapLevel = 1, kRemapFinal = 2, kRemapPositions = 4, kRemapOther = 8;

template <int BIT = kRemapOther>
__device__ __forceinline__ int64_t block_index() {
  const int b = blockIdx.x;
  if (!(g_xcd_remap & BIT)) return b;
  const int nb = gridDim.x;
  const int per = nb >> 3, rem = nb & 7, x = b & 7, i = b >> 3;
  return (int64_t)((x < rem ? x * (per + 1) : rem * (per + 1) + (x - rem) * per) + i);
}

inline unsigned grid_for(int64_t n, int block = kBlock) {
  int64_t g = (n + block - 1) / block;
  return (unsigned)(g < 1 ? 1 : g);
}

// ---------------------------------------------------------------------------
// fills

__global__ void k_fill_i32(int32_t* __restrict__ p, int64_t n, int32_t value) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = value;
}

// A plan's start in one launch: its tables from pinned host memory (read
// across the bus by the kernel itself) and its zeroed state.
__global__ void __launch_bounds__(kBlock) k_setup(const int4* __restrict__ src, int4* __restrict__ dst, int64_t n,
                                                  int4* __restrict__ zero, int64_t nzero) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (int64_t i = i0; i < n; i += stride) dst[i] = src[i];
  for (int64_t i = i0; i < nzero; i += stride) zero[i] = make_int4(0, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// HBM reference: a float4 stream copy (bandwidth probe and counter
// calibration), one float4 per lane over a grid that covers the buffer (on
// MI355X this reaches about 6.3 TB/s read + write; a grid-stride loop over a
// fixed grid stays near 4.5)

__global__ void __launch_bounds__(kBlock) k_copy_probe(const float4* __restrict__ a, float4* __restrict__ b,
                                                        int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
}

// Order-sensitive 64-bit digest of a byte buffer: the sum (mod 2^64) over its
// 32-bit words w_i (the last one zero-padded) of mix64(w_i + (i + 1) * G), a
// splitmix64 finaliser. A sum is independent of the reduction order, so the
// digest is deterministic; each block adds its partial to *out (zeroed first).
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

constexpr int kDigestBlocks = 2048;

__global__ void __launch_bounds__(kBlock) k_digest(const uint8_t* __restrict__ p, int64_t bytes,
                                                   unsigned long long* __restrict__ out) {
  const int64_t nw = (bytes + 3) / 4, full = bytes / 4;
  const uint32_t* __restrict__ w = reinterpret_cast<const uint32_t*>(p);
  uint64_t acc = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nw; i += (int64_t)gridDim.x * blockDim.x) {
    uint32_t x;
    if (i < full) {
      x = w[i];
    } else {  // the zero-padded last word
      x = 0;
      for (int64_t b = 4 * i; b < bytes; ++b) x |= (uint32_t)p[b] << (8 * (b - 4 * i));
    }
    acc += mix64((uint64_t)x + (uint64_t)(i + 1) * 0x9E3779B97F4A7C15ull);
  }
  __shared__ uint64_t part[kBlock / 64];
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t s = 0;
    for (int k = 0; k < kBlock / 64; ++k) s += part[k];
    atomicAdd(out, (unsigned long long)s);
  }
}

// ---------------------------------------------------------------------------
// first level: validate each caller mesh and gather it into the union in
// position order (sortKeyValuePairsSegmentedInPlace, LAKCatmullClarkKernels.cuh:147-180)

constexpr int kHistBins = kRowHistBins;  // row lengths 0..15, 16 = longer
static_assert(kHistBins <= kHistStride, "a histogram copy holds every bin");

// Adds 1 to bin `bin` of an LDS histogram for every calling lane, with one
// LDS atomic per distinct bin of the wave: same-address LDS atomics from the
// lanes of a wave serialize (on a quad mesh every lane has the same bin).
__device__ __forceinline__ void hist_add_wave(int32_t* lds, int bin) {
  unsigned long long todo = __ballot(1);
  while (todo) {
    const int leader = __ffsll(todo) - 1;
    const int b = __shfl(bin, leader);
    const unsigned long long same = __ballot(bin == b) & todo;
    if ((int)(threadIdx.x & 63) == leader) atomicAdd(&lds[b], __popcll(same));
    todo &= ~same;
  }
}

// Block-local histogram in LDS, added to copy blockIdx % kHistCopies of a
// zeroed global histogram block (one atomic per nonzero bin).
struct BlockHist {
  int32_t* lds;
  __device__ __forceinline__ void init() {
    for (int i = threadIdx.x; i < kHistBins; i += blockDim.x) lds[i] = 0;
    __syncthreads();
  }
  __device__ __forceinline__ void flush(int32_t* global) {
    __syncthreads();
    int32_t* copy = global + (blockIdx.x % kHistCopies) * kHistStride;
    for (int i = threadIdx.x; i < kHistBins; i += blockDim.x)
      if (lds[i]) atomicAdd(&copy[i], lds[i]);
  }
};

// What the gather hands on of one face to the row building: the corners of
// the union (first corner c0) and their union vertices, in storage order for
// the corners kept in registers (v[i] < 0: none, or an invalid corner).
constexpr int kGatherRegs = 8;

template <int REGS>
struct FaceCorners {
  int32_t v[REGS];
  int32_t c[REGS];
};

// M^T rows under construction (first level): cnt[v] corners of vertex v so
// far, the first kRowSlots of them in slots[kRowSlots v ..], the others in a
// linked list (head[v], then next[corner]) of cnt[v] - kRowSlots entries.
struct RowBuild {
  int32_t* cnt;
  int32_t* slots;
  int32_t* head;
  int32_t* next;
};

__device__ __forceinline__ void put_row(const RowBuild& rb, int32_t v, int32_t slot, int32_t c) {
  if (slot < kRowSlots)
    rb.slots[(int64_t)kRowSlots * v + slot] = c;
  else
    rb.next[c] = atomicExch(&rb.head[v], c);
}

template <bool QUAD, bool ONE>
__device__ __forceinline__ void gather_face(const SegTable& seg, int32_t f, int32_t nf_total, int use_vals,
                                            int32_t* __restrict__ ids_pos, int32_t* __restrict__ fptr,
                                            int32_t* __restrict__ cface, int* __restrict__ flags,
                                            const RowBuild& rb, FaceCorners<QUAD ? 4 : kGatherRegs>& out);

// min / max over the block (mm: kBlock / 64 LDS entries)
__device__ __forceinline__ int2 block_minmax(int lo, int hi, int2* mm) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    lo = min(lo, __shfl_xor(lo, d));
    hi = max(hi, __shfl_xor(hi, d));
  }
  if ((threadIdx.x & 63) == 0) mm[threadIdx.x >> 6] = make_int2(lo, hi);
  __syncthreads();
  int2 r = mm[0];
#pragma unroll
  for (int w = 1; w < kBlock / 64; ++w) r = make_int2(min(r.x, mm[w].x), max(r.y, mm[w].y));
  return r;
}

// The corners of a block's 256 faces usually reference a narrow range of
// vertex ids (grids, refined meshes, each mesh of a batch): the block then
// counts into LDS over [vmin, vmax] and reserves each touched vertex's row
// slots with one device atomic. A block whose range is wider than
// kCountWindow vertices takes one per corner (device-scope atomics are what
// the row building costs).
constexpr int kCountWindow = 2048;

// Gather, valence count and row placement in one pass over the caller's
// faces: the corners of a face are in registers when they are placed, and a
// row needs no offset while its corners go to fixed slots, so no scan stands
// between the count and the placement.
template <bool QUAD, bool ONE>
__global__ void __launch_bounds__(kBlock) k_gather(SegTable seg, int32_t nf_total, int use_vals, int32_t* __restrict__ ids_pos,
                         int32_t* __restrict__ fptr, int32_t* __restrict__ cface, int* __restrict__ flags,
                         RowBuild rb, int window) {
  constexpr int REGS = QUAD ? 4 : kGatherRegs;
  __shared__ int32_t win[kCountWindow];
  __shared__ int2 mm[kBlock / 64];
  const int32_t f = (int32_t)(block_index() * blockDim.x + threadIdx.x);
  FaceCorners<REGS> fc;
#pragma unroll
  for (int i = 0; i < REGS; ++i) fc.v[i] = -1;
  if (f < nf_total) gather_face<QUAD, ONE>(seg, f, nf_total, use_vals, ids_pos, fptr, cface, flags, rb, fc);
  int lo = INT_MAX, hi = INT_MIN;
#pragma unroll
  for (int i = 0; i < REGS; ++i)
    if (fc.v[i] >= 0) {
      lo = min(lo, fc.v[i]);
      hi = max(hi, fc.v[i]);
    }
  const int2 w = block_minmax(lo, hi, mm);
  const int64_t n = (int64_t)w.y - w.x + 1;  // <= 0 when no corner is placed
  if (window && n <= kCountWindow) {          // block-uniform
    for (int i = threadIdx.x; i < n; i += kBlock) win[i] = 0;
    __syncthreads();
    int32_t rank[REGS];
#pragma unroll
    for (int i = 0; i < REGS; ++i)
      if (fc.v[i] >= 0) rank[i] = atomicAdd(&win[fc.v[i] - w.x], 1);
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += kBlock) {
      const int32_t k = win[i];
      if (k) win[i] = atomicAdd(&rb.cnt[w.x + i], k);  // the first slot of the block's corners
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < REGS; ++i)
      if (fc.v[i] >= 0) put_row(rb, fc.v[i], win[fc.v[i] - w.x] + rank[i], fc.c[i]);
  } else {
#pragma unroll
    for (int i = 0; i < REGS; ++i)
      if (fc.v[i] >= 0) put_row(rb, fc.v[i], atomicAdd(&rb.cnt[fc.v[i]], 1), fc.c[i]);
  }
}

// first level: validate caller face f and gather it into the union in
// position order. out: the face's
// valid corners for the row building; the corners of a longer face beyond
// the registers are placed here, one device atomic each.
template <bool QUAD, bool ONE>
__device__ __forceinline__ void gather_face(const SegTable& seg, int32_t f, int32_t nf_total, int use_vals,
                                            int32_t* __restrict__ ids_pos, int32_t* __restrict__ fptr,
                                            int32_t* __restrict__ cface, int* __restrict__ flags,
                                            const RowBuild& rb, FaceCorners<QUAD ? 4 : kGatherRegs>& out) {
  const SegDesc* S = face_seg<ONE>(seg, f);
  int* const mflags = seg.mflags + (ONE ? 0 : S - seg.d);
  const int32_t lf = (int32_t)(f - S->fb);
  const int32_t* sp = to_global(S->src_ptr);
  const int32_t* sid = to_global(S->src_ids);
  const int32_t* sval = use_vals ? to_global(S->src_vals) : nullptr;
  const int64_t snnz = S->nnz;
  int64_t s = sp ? sp[lf] : (int64_t)S->src_stride * lf;
  int64_t e = sp ? sp[lf + 1] : (int64_t)S->src_stride * (lf + 1);
  int bad = 0;
  if (lf == 0 && s != 0) bad |= kFlagBadPtr;
  if (lf == S->nf - 1 && e != snnz) bad |= kFlagBadPtr;
  if (s < 0 || e < s || e > snnz) {
    bad |= kFlagBadPtr;
    atomicOr(mflags, bad);
    atomicOr(flags, bad);
    return;
  }
  const int32_t order = (int32_t)(e - s);
  if (order < 3) bad |= kFlagBadOrder;
  if (S->require_quad && (order != 4 || s != 4ll * lf)) bad |= kFlagBadQuad;
  const int64_t cb = S->cb;
  const int32_t vb = (int32_t)S->vb;
  if (order == 4 && ((reinterpret_cast<uintptr_t>(sid + s) | (sval ? reinterpret_cast<uintptr_t>(sval + s) : 0)) & 15) == 0) {
    // a quad with 16-byte aligned corners: one load of its ids (and vals),
    // one store when the union position is aligned too; anything unusual
    // takes the per-corner path below
    const int4 q = *reinterpret_cast<const int4*>(sid + s);
    const int4 p = sval ? *reinterpret_cast<const int4*>(sval + s) : make_int4(1, 2, 3, 4);
    const uint32_t in_range = (uint32_t)q.x < (uint32_t)S->nv && (uint32_t)q.y < (uint32_t)S->nv &&
                              (uint32_t)q.z < (uint32_t)S->nv && (uint32_t)q.w < (uint32_t)S->nv;
    const bool pos_ok = (uint32_t)(p.x - 1) < 4u && (uint32_t)(p.y - 1) < 4u && (uint32_t)(p.z - 1) < 4u &&
                        (uint32_t)(p.w - 1) < 4u;
    if (in_range && pos_ok && ((1u << (p.x - 1)) | (1u << (p.y - 1)) | (1u << (p.z - 1)) | (1u << (p.w - 1))) == 15u) {
      // the corner at position k (1-based) is the one whose vals entry is k
      auto at = [&](int k) __attribute__((always_inline)) {
        return vb + (p.x == k ? q.x : p.y == k ? q.y : p.z == k ? q.z : q.w);
      };
      const int4 o = make_int4(at(1), at(2), at(3), at(4));
      int32_t* dst = ids_pos + cb + s;
      if ((reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
        *reinterpret_cast<int4*>(dst) = o;
      } else {
        dst[0] = o.x;
        dst[1] = o.y;
        dst[2] = o.z;
        dst[3] = o.w;
      }
      if (cface) {
        int32_t* cf = cface + cb + s;
        if ((reinterpret_cast<uintptr_t>(cf) & 15) == 0) {
          *reinterpret_cast<int4*>(cf) = make_int4(f, f, f, f);
        } else {
          cf[0] = f;
          cf[1] = f;
          cf[2] = f;
          cf[3] = f;
        }
      }
      if (fptr) {
        fptr[f] = (int32_t)(cb + s);
        if (f == nf_total - 1) fptr[nf_total] = (int32_t)(cb + e);
      }
      if (bad) {
        atomicOr(mflags, bad);
        atomicOr(flags, bad);
      }
      const int32_t c0 = (int32_t)(cb + s);
      out.v[0] = o.x;
      out.v[1] = o.y;
      out.v[2] = o.z;
      out.v[3] = o.w;
#pragma unroll
      for (int i = 0; i < 4; ++i) out.c[i] = c0 + i;
      return;
    }
  }
  // any other face: its first REGS corners are loaded before the
  // first store (a load issued after a store would wait for it), the rest
  // one by one
  constexpr int REGS = QUAD ? 4 : kGatherRegs;
  const int32_t snv = S->nv;
  uint32_t mask = 0;
  // returns whether the corner can be placed in its vertex's row
  auto corner = [&](int64_t c, int32_t id, int32_t pos) __attribute__((always_inline)) -> bool {
    const bool known = id >= 0 && id < snv;
    if (!known) {
      bad |= kFlagBadId;
      id = 0;
    }
    if (pos < 1 || pos > order) {
      bad |= kFlagBadVals;
      return false;
    }
    if (order <= 32) {
      uint32_t bit = 1u << (pos - 1);
      if (mask & bit) bad |= kFlagBadVals;
      mask |= bit;
    } else {
      for (int64_t c2 = s; c2 < c; ++c2)
        if ((sval ? sval[c2] : (int32_t)(c2 - s + 1)) == pos) bad |= kFlagBadVals;
    }
    ids_pos[cb + s + pos - 1] = vb + id;
    if (cface) cface[cb + c] = f;
    return known;
  };
  int32_t rid[REGS], rpos[REGS];
#pragma unroll
  for (int i = 0; i < REGS; ++i)
    if (i < order) {
      rid[i] = sid[s + i];
      rpos[i] = sval ? sval[s + i] : i + 1;
    }
#pragma unroll
  for (int i = 0; i < REGS; ++i)
    if (i < order && corner(s + i, rid[i], rpos[i])) {
      out.v[i] = vb + rid[i];
      out.c[i] = (int32_t)(cb + s + rpos[i] - 1);
    }
  for (int64_t c = s + REGS; c < e; ++c) {
    const int32_t id = sid[c], pos = sval ? sval[c] : (int32_t)(c - s + 1);
    if (corner(c, id, pos))
      put_row(rb, vb + id, atomicAdd(&rb.cnt[vb + id], 1), (int32_t)(cb + s + pos - 1));
  }
  if (fptr) {
    fptr[f] = (int32_t)(cb + s);
    if (f == nf_total - 1) fptr[nf_total] = (int32_t)(cb + e);
  }
  if (bad) {
    atomicOr(mflags, bad);
    atomicOr(flags, bad);
  }
}

__global__ void k_gather_verts(SegTable seg, int32_t nv_total, float4* __restrict__ P) {
  int32_t v = (int32_t)(block_index() * blockDim.x + threadIdx.x);
  if (v >= nv_total) return;
  const SegDesc* S = vertex_seg<false>(seg, v);
  P[v] = to_global(S->src_verts)[v - S->vb];
}

// ---------------------------------------------------------------------------
// face points into each segment's destination

template <bool QUAD, bool ONE>
__device__ __forceinline__ void faces_item(const int32_t* __restrict__ ids, const int32_t* __restrict__ fptr,
                                           const float4* __restrict__ P, int32_t nf, const SegTable& seg, int32_t f) {
  if (f >= nf) return;
  const SegDesc* S = face_seg<ONE>(seg, f);
  float4* const dst = to_global(S->dst_verts) + S->nv + (f - S->fb);
  if (QUAD) {
    int4 c = reinterpret_cast<const int4*>(ids)[f];
    *dst = f4div(f4add(f4add(f4add(P[c.x], P[c.y]), P[c.z]), P[c.w]), 4.0f);
  } else {
    int32_t s = fptr[f], e = fptr[f + 1];
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int32_t c = s; c < e; ++c) acc = f4add(acc, P[ids[c]]);
    *dst = f4div(acc, (float)(e - s));
  }
}

template <bool QUAD, bool ONE>
__global__ void k_faces(const int32_t* __restrict__ ids, const int32_t* __restrict__ fptr, const float4* __restrict__ P,
                        int32_t nf, SegTable seg, const int* stop) {
  if (stopped(stop)) return;
  faces_item<QUAD, ONE>(ids, fptr, P, nf, seg, (int32_t)(block_index() * blockDim.x + threadIdx.x));
}

// 64-bit lane exchange by DPP (row_shr / row_bcast); lanes without a source,
// and rows outside ROWMASK, read 0.
template <int CTRL, int ROWMASK>
__device__ __forceinline__ int64_t dpp64(int64_t x) {
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)x, CTRL, ROWMASK, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(x >> 32), CTRL, ROWMASK, 0xF, false);
  return (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}
// Inclusive scan over the 64 lanes of a wave: shifts by 1, 2, 4, 8 inside
// each row of 16 lanes, then lane 15 of rows 0 / 2 into rows 1 / 3 and lane
// 31 into rows 2 and 3.
__device__ __forceinline__ int64_t wave_scan64(int64_t x) {
  x += dpp64<0x111, 0xF>(x);
  x += dpp64<0x112, 0xF>(x);
  x += dpp64<0x114, 0xF>(x);
  x += dpp64<0x118, 0xF>(x);
  x += dpp64<0x142, 0xA>(x);
  x += dpp64<0x143, 0xC>(x);
  return x;
}

// ---------------------------------------------------------------------------
// mapped SpGEMM, symbolic and numeric

__device__ void sort_row_in_place(int32_t* a, int n) {
  for (int i = 1; i < n; ++i) {
    int32_t x = a[i];
    int j = i;
    while (j > 0 && a[j - 1] > x) {
      a[j] = a[j - 1];
      --j;
    }
    a[j] = x;
  }
}

// The unsorted corners of vertex v's row of n: its slots, or (more than
// kRowSlots) the run of the tids pool that slot 0 points to once k_symbolic
// has gathered the row there.
__device__ __forceinline__ int32_t* row_corners(const LevelView& L, int32_t v, int n) {
  int32_t* const slots = L.slots + (int64_t)kRowSlots * v;
  return n <= kRowSlots ? slots : L.tids + slots[0];
}

// Row lengths and owned-edge counts are summed per tile of kBlock vertices
// (packed: corners << 31 | edges; a level's totals stay below 2^31) and per
// kTilesPerGroup tiles, so that any later block adds up the offsets of its
// rows from the sums before it, one group sum for 16384 vertices and at most 64
// tile sums, 256 at a time: no scan launches, and no block waits for another.
// The sums grow with the square of the vertices, but int32 corners end a quad
// mesh at 134 M vertices, where they are 32 loads a thread: one level of quad
// tori of 5, 20, 40 and 80 M vertices takes 0.81, 2.97, 5.93 and 12.1 ms a call
// (with scan launches 0.97, 3.64, 7.35, 14.7), the last 2 % above linear. (A decoupled look-back in the sizing pass measured slower: its
// ticket, one atomic per block on one address, takes about 20 ns a block --
// 89 against 31 us on 4096 blocks.)
__device__ __forceinline__ uint64_t pack_row(int32_t n, int32_t owned) {
  return ((uint64_t)(uint32_t)n << 31) | (uint32_t)owned;
}
constexpr uint64_t kOwnedMask = (1ull << 31) - 1;

// sum over the block; lds: kBlock / 64 entries, free again after a barrier
__device__ __forceinline__ uint64_t block_sum(uint64_t x, uint64_t* lds) {
  for (int d = 32; d > 0; d >>= 1) x += __shfl_xor(x, d, 64);
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = x;
  __syncthreads();
  uint64_t t = 0;
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) t += lds[w];
  return t;
}

// exclusive scan over the block; total: the block's sum
__device__ __forceinline__ uint64_t block_scan_packed(uint64_t x, uint64_t* lds, uint64_t& total) {
  const uint64_t inc = (uint64_t)wave_scan64((int64_t)x);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 63) lds[wave] = inc;
  __syncthreads();
  uint64_t off = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) {
    off += w < wave ? lds[w] : 0;
    total += lds[w];
  }
  return off + inc - x;
}

// this thread's share of the packed sum of all tiles before `tile`
__device__ __forceinline__ uint64_t tiles_before(const LevelView& L, int tile, int tid, int nthreads) {
  const int group = tile / kTilesPerGroup;
  uint64_t acc = 0;
  for (int i = tid; i < group; i += nthreads) acc += L.group_sum[i];
  for (int i = group * kTilesPerGroup + tid; i < tile; i += nthreads) acc += L.tile_sum[i];
  return acc;
}

// Runs fn(row) on vertex v's row of n <= cap corners in registers, from its
// slots. Sorting and pairing a row of capacity C costs about C^2 selects, so
// each wave takes the smallest of three capacities that holds all of its rows.
template <bool QUAD, class Fn>
__device__ __forceinline__ void with_row(const LevelView& L, const int32_t* slots, int n, Fn&& fn) {
  auto run = [&](auto row) __attribute__((always_inline)) {
    row.load_slots(L, slots, n);
    fn(row);
  };
  if (__any(n > 6))
    run(RegRow<8, QUAD>{});
  else if (__any(n > 4))
    run(RegRow<6, QUAD>{});
  else
    run(RegRow<4, QUAD>{});
}

// Mapped-SpGEMM row sizing, one lane per vertex: the row's corners from their
// slots, validated, the edges the vertex owns counted; a row longer than its
// slots is gathered into a run of the pool, and rows beyond the register
// capacity are sorted in place.
template <bool QUAD, int SCHEME>
__global__ void __launch_bounds__(kBlock) k_symbolic(LevelView L) {
  __shared__ int32_t h[kHistBins];
  __shared__ uint64_t wave_sum[kBlock / 64];
  if (*L.flags & kFlagsInput) return;  // set by the gather alone: the same for every block
  BlockHist bh{h};
  bh.init();
  const int tile = (int)block_index();
  const int32_t v = tile * kBlock + (int32_t)threadIdx.x;
  int32_t n = 0, owned = 0, bcount = 0;
  int bad = 0;
  if (v < L.nv) {
    n = L.cnt[v];
    hist_add_wave(h, n < kHistBins - 1 ? n : kHistBins - 1);
    int32_t* row = L.slots + (int64_t)kRowSlots * v;
    if (n <= L.row_cap) {
      with_row<QUAD>(L, row, n, [&](auto& r) __attribute__((always_inline)) {
        row_symbolic<SCHEME>(r, v, owned, bcount, bad);
      });
    } else {
      if (n > kRowSlots) {  // the whole row to a run of the pool
        int32_t* const run = L.tids + atomicAdd(L.pool, n);
        for (int i = 0; i < kRowSlots; ++i) run[i] = row[i];
        int32_t c = L.head[v];
        for (int i = n - 1; i >= kRowSlots; --i) {  // (the list is last in, first out: nearly ascending this way)
          run[i] = c;
          c = L.next[c];
        }
        row[0] = (int32_t)(run - L.tids);
        row = run;
      }
      sort_row_in_place(row, n);
      const MemRow<QUAD> r(L, row, n);
      row_symbolic<SCHEME>(r, v, owned, bcount, bad);
    }
    (void)bcount;
    L.ecnt[v] = owned;
    if (bad) {
      atomicOr(L.flags, bad);
      atomicOr(L.seg.mflags + seg_of(L.seg.vbase, L.seg.n, v), bad);
    }
  }
  const uint64_t sum = block_sum(pack_row(n, owned), wave_sum);
  if (threadIdx.x == 0) {
    L.tile_sum[tile] = sum;
    atomicAdd(reinterpret_cast<unsigned long long*>(L.group_sum) + tile / kTilesPerGroup, (unsigned long long)sum);
  }
  bh.flush(L.hist_rows);
}

// bounds[k] = owned edges before mesh k, k = 0 .. n (several meshes), one
// wave each
__global__ void __launch_bounds__(kBlock) k_seg_bounds(LevelView L) {
  if (*L.flags & kFlagsInput) return;
  const int32_t k = (int32_t)((blockIdx.x * kBlock + threadIdx.x) >> 6);
  if (k > L.seg.n) return;  // wave-uniform
  const int lane = threadIdx.x & 63;
  const int32_t b = (int32_t)L.seg.vbase[k];
  const int tile = b / kBlock;
  uint64_t acc = tiles_before(L, tile, lane, 64) & kOwnedMask;
  for (int32_t v = tile * kBlock + lane; v < b; v += 64) acc += (uint64_t)L.ecnt[v];
  for (int d = 32; d > 0; d >>= 1) acc += __shfl_xor(acc, d, 64);
  if (lane) return;
  L.bounds[k] = (int32_t)acc;
  if (L.planned) {
    const SegDesc& S = L.seg.d[k < L.seg.n ? k : L.seg.n - 1];
    if ((int64_t)acc != S.eb + (k < L.seg.n ? 0 : S.ne)) atomicOr(L.flags, kFlagChanged);
  }
}

// What the host waits for, written straight to its memory by one block (a
// copy and an event after the analysis cost 5 us more a call): the flags, the
// row-length histogram, the owned edges before each mesh; then the done word.
__device__ void report(const LevelView& L, uint64_t* lds) {
  int32_t* const out = L.report;
  const int tid = threadIdx.x;
  if (tid == 0) out[1] = *L.flags;
  if (tid < kRowHistBins) {
    int32_t x = 0;
    for (int c = 0; c < kHistCopies; ++c) x += L.hist_rows[c * kHistStride + tid];
    out[2 + tid] = x;
  }
  int32_t* const bounds = out + 2 + kRowHistBins;
  if (L.seg.n > 1) {
    for (int k = tid; k <= L.seg.n; k += kBlock) bounds[k] = L.bounds[k];
  } else {
    uint64_t acc = 0;
    for (int i = tid; i < L.ngroups; i += kBlock) acc += L.group_sum[i];
    const uint64_t sum = block_sum(acc, lds);
    if (tid == 0) {
      bounds[0] = 0;
      bounds[1] = (int32_t)(sum & kOwnedMask);
    }
  }
  __threadfence_system();
  __syncthreads();
  if (tid == 0) __hip_atomic_store(out, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void __launch_bounds__(kBlock) k_report(LevelView L) {
  __shared__ uint64_t lds[kBlock / 64];
  report(L, lds);
}

// First level, blocks [0, nbn): the rows of R = L.rows_per_block vertices (a
// part of a sizing tile), one lane per row. The block forms its rows' offsets
// from the tile sums, writes them and the sorted rows with their
// in-neighbours (through its LDS tile when they fit: L.tile_entries entries
// of dynamic LDS), and numbers the edges its vertices own. The other blocks
// form the face points, which are independent.
extern __shared__ __align__(16) unsigned char row_tile_lds[];

template <bool QUAD, int SCHEME, bool ONE>
__global__ void __launch_bounds__(kBlock) k_number_faces(LevelView L, int32_t nbn) {
  __shared__ uint64_t wave_sum[2][kBlock / 64];
  __shared__ uint64_t row_at[kBlock + 1];
  // an invalid mesh: its ids, rows and counts were not (all) written; a
  // single mesh's numbering is launched before the host has read the flags
  const bool reports = ONE && L.report;
  if (reports && blockIdx.x == 0) {
    report(L, wave_sum[0]);
    return;
  }
  if (*L.flags & kFlagsInput) return;
  const int64_t b = block_index() - (reports ? 1 : 0);
  if (b >= nbn) {
    faces_item<QUAD, ONE>(L.ids, L.fptr, L.P, L.nf, L.seg, (int32_t)((b - nbn) * blockDim.x + threadIdx.x));
    return;
  }
  int2* const tile_out = reinterpret_cast<int2*>(row_tile_lds);  // (corner, in-neighbour)
  const int R = L.rows_per_block;
  const int32_t v0 = (int32_t)b * R;
  const int tile = v0 / kBlock, r0 = v0 - tile * kBlock;  // the block's rows [r0, r0 + R) of the tile
  {
    const int32_t tv = tile * kBlock + (int32_t)threadIdx.x;
    const uint64_t own = tv < L.nv ? pack_row(L.cnt[tv], L.ecnt[tv]) : 0;
    const uint64_t before = block_sum(tiles_before(L, tile, threadIdx.x, kBlock), wave_sum[0]);
    uint64_t total;
    const uint64_t ex = block_scan_packed(own, wave_sum[1], total);
    row_at[threadIdx.x] = before + ex;
    if (threadIdx.x == 0) row_at[kBlock] = before + total;
  }
  __syncthreads();
  const int32_t s0 = (int32_t)(row_at[r0] >> 31);
  const int32_t len = (int32_t)(row_at[r0 + R] >> 31) - s0;  // 0 rows beyond the last vertex
  const bool staged = len <= L.tile_entries;                 // block-uniform
  const int32_t v = v0 + (int32_t)threadIdx.x;
  if ((int)threadIdx.x < R && v < L.nv) {
    const uint64_t at = row_at[r0 + threadIdx.x];
    const int32_t s = (int32_t)(at >> 31), e0 = (int32_t)(at & kOwnedMask);
    const int n = (int)((int32_t)(row_at[r0 + threadIdx.x + 1] >> 31) - s);
    L.tptr[v] = s;
    L.eptr[v] = e0;
    if (v == L.nv - 1) {
      const int32_t edges = (int32_t)(row_at[r0 + threadIdx.x + 1] & kOwnedMask);
      L.tptr[L.nv] = s + n;
      L.eptr[L.nv] = edges;
      if (ONE && L.planned && edges != L.seg.one.ne) atomicOr(L.flags, kFlagChanged);
    }
    // the sorted row to the LDS tile, or straight to its place
    // (by a branch around each store: a pointer that may address LDS or
    // global memory makes every access through it a FLAT instruction)
    auto put = [&](int i, int32_t t, int32_t u) __attribute__((always_inline)) {
      if (staged)
        tile_out[s - s0 + i] = make_int2(t, u);
      else
        L.trow[s + i] = make_int2(t, u);
      if (SCHEME == kSLAK) L.mpos[t] = s + i;
    };
    if (n <= L.row_cap) {
      with_row<QUAD>(L, L.slots + (int64_t)kRowSlots * v, n, [&](auto& r) __attribute__((always_inline)) {
        constexpr int C = std::decay_t<decltype(r)>::kCap;
#pragma unroll
        for (int i = 0; i < C; ++i)
          if (i < n) put(i, r.T(i), r.U(i));
        row_number<SCHEME, ONE>(r, L, v, e0);
      });
    } else {
      // the sizing pass sorted every row longer than its own capacity; this
      // one must be sorted whatever that capacity was (idempotent)
      int32_t* const row = row_corners(L, v, n);
      sort_row_in_place(row, n);
      MemRow<QUAD> r(L, row, n);
      for (int i = 0; i < n; ++i) put(i, r.T(i), r.U(i));
      row_number<SCHEME, ONE>(r, L, v, e0);
    }
  }
  __syncthreads();
  if (staged)
    for (int i = threadIdx.x; i < len; i += kBlock) L.trow[s0 + i] = tile_out[i];
}

// The whole first level of a small mesh (at most kSmallItems faces and
// vertices, four times as many corners) in one block: gather, row sizing,
// report, numbering and face points, one item per thread, phases apart by
// barriers; counters and offsets stay in LDS. A call on such a mesh is bound
// by its chain of dependent launches, and this is one of them in place of
// four (zeroed state, gather, sizing, numbering). Whole calls: cube, 3 levels
// 59.8 -> 51.3 us; torus of 512 quads, 3 levels 62.5 -> 55.5; of 1024 quads
// 62.7 -> 60.8; 968 triangles, 2 levels 68.4 -> 64.0; open grid of 930 quads
// 70.5 -> 61.6. The line is the largest block: beyond it one compute unit
// would do in turn what the launches spread. Same rows, numbers and points as
// theirs: both run the same row and face code.
constexpr int kSmallItems = 1024;

template <bool QUAD, int SCHEME>
__global__ void __launch_bounds__(kSmallItems) k_first_small(LevelView L, int use_vals, int faces) {
  constexpr int REGS = QUAD ? 4 : kGatherRegs;
  __shared__ int32_t cnt[kSmallItems], head[kSmallItems];  // blockDim.x used: one per thread
  __shared__ uint64_t wave_sum[kSmallItems / 64];
  __shared__ int32_t pool;
  __shared__ int32_t flags;
  const int tid = threadIdx.x;
  cnt[tid] = 0;
  if (tid == 0) {
    pool = 0;
    flags = 0;
    L.seg.mflags[0] = 0;
  }
  __syncthreads();
  const RowBuild rb{cnt, L.slots, head, L.next};
  FaceCorners<REGS> fc;
#pragma unroll
  for (int i = 0; i < REGS; ++i) fc.v[i] = -1;
  if (tid < L.nf)
    gather_face<QUAD, true>(L.seg, tid, L.nf, use_vals, const_cast<int32_t*>(L.ids), const_cast<int32_t*>(L.fptr),
                            const_cast<int32_t*>(L.cface), &flags, rb, fc);
#pragma unroll
  for (int i = 0; i < REGS; ++i)
    if (fc.v[i] >= 0) put_row(rb, fc.v[i], atomicAdd(&cnt[fc.v[i]], 1), fc.c[i]);
  __syncthreads();
  const bool valid = !(flags & kFlagsInput);  // the sizing sets no input flag: the same for every thread
  const int32_t v = tid;
  const bool active = valid && v < L.nv;
  const int n = active ? cnt[v] : 0;
  int32_t* row = L.slots + (int64_t)kRowSlots * v;
  int32_t owned = 0, bcount = 0;
  int bad = 0;
  if (active) {
    if (n <= L.row_cap) {
      with_row<QUAD>(L, row, n, [&](auto& r) __attribute__((always_inline)) {
        row_symbolic<SCHEME>(r, v, owned, bcount, bad);
      });
    } else {
      if (n > kRowSlots) {  // the whole row to a run of the pool
        int32_t* const run = L.tids + atomicAdd(&pool, n);
        for (int i = 0; i < kRowSlots; ++i) run[i] = row[i];
        int32_t c = head[v];
        for (int i = n - 1; i >= kRowSlots; --i) {  // (the list is last in, first out: nearly ascending this way)
          run[i] = c;
          c = L.next[c];
        }
        row[0] = (int32_t)(run - L.tids);
        row = run;
      }
      sort_row_in_place(row, n);
      const MemRow<QUAD> r(L, row, n);
      row_symbolic<SCHEME>(r, v, owned, bcount, bad);
    }
    (void)bcount;
    if (bad) {
      atomicOr(&flags, bad);
      atomicOr(L.seg.mflags, bad);
    }
  }
  const uint64_t own = pack_row(n, owned);
  const uint64_t inc = (uint64_t)wave_scan64((int64_t)own);
  if ((tid & 63) == 63) wave_sum[tid >> 6] = inc;
  __syncthreads();  // (also: L.next is read before the numbering overwrites it)
  uint64_t at = inc - own, total = 0;
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
    at += w < (tid >> 6) ? wave_sum[w] : 0;
    total += wave_sum[w];
  }
  static_assert(2 + kRowHistBins + 2 <= 64);
  if (tid < 2 + kRowHistBins + 2) {  // one wave; the host goes on from here
    int32_t x = 0;                   // (no histogram: it tunes launches that a small mesh does not have)
    if (tid == 0) *L.flags = flags;
    if (tid == 1) x = flags;
    if (tid == 2 + kRowHistBins + 1) x = (int32_t)(total & kOwnedMask);
    if (tid > 0) L.report[tid] = x;
    __threadfence_system();
    if (tid == 0) __hip_atomic_store(L.report, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);  // (after the wave's stores)
  }
  if (!valid) return;
  if (active) {
    const int32_t s = (int32_t)(at >> 31), e0 = (int32_t)(at & kOwnedMask);
    L.tptr[v] = s;
    L.eptr[v] = e0;
    if (v == L.nv - 1) {
      L.tptr[L.nv] = s + n;
      L.eptr[L.nv] = e0 + owned;
    }
    auto put = [&](int i, int32_t t, int32_t u) __attribute__((always_inline)) {
      L.trow[s + i] = make_int2(t, u);
      if (SCHEME == kSLAK) L.mpos[t] = s + i;
    };
    if (n <= L.row_cap) {
      with_row<QUAD>(L, row, n, [&](auto& r) __attribute__((always_inline)) {
        constexpr int C = std::decay_t<decltype(r)>::kCap;
#pragma unroll
        for (int i = 0; i < C; ++i)
          if (i < n) put(i, r.T(i), r.U(i));
        row_number<SCHEME, true>(r, L, v, e0);
      });
    } else {
      MemRow<QUAD> r(L, row, n);  // sorted above
      for (int i = 0; i < n; ++i) put(i, r.T(i), r.U(i));
      row_number<SCHEME, true>(r, L, v, e0);
    }
  }
  if (faces) faces_item<QUAD, true>(L.ids, L.fptr, L.P, L.nf, L.seg, tid);
}

template <bool QUAD>
__global__ void __launch_bounds__(kBlock) k_spgemm_fde(LevelView L) {
  int32_t v = (int32_t)(block_index() * blockDim.x + threadIdx.x);
  if (v >= L.nv) return;
  int32_t s = L.tptr[v];
  int n = L.tptr[v + 1] - s;
  if (n <= kRowSlots) {
    RegRow<kRowSlots, QUAD> r;
    r.load_slots(L, L.slots + (int64_t)kRowSlots * v, n);
    row_fde(r, L, v);
  } else {
    MemRow<QUAD> r(L, row_corners(L, v, n), n);  // sorted by k_symbolic
    row_fde(r, L, v);
  }
}

__device__ __forceinline__ int32_t clampi(int32_t x, int32_t hi) { return min(max(x, 0), hi); }

// Streamed outputs of the final level are written once and not read back by
// this pipeline: non-temporal stores keep them from displacing the gathered
// positions in the caches.
typedef int v4i_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void store_nt(int32_t* p, int a, int b, int c, int d) {
  v4i_t x = {a, b, c, d};
  __builtin_nontemporal_store(x, reinterpret_cast<v4i_t*>(p));
}
__device__ __forceinline__ void store_nt(int32_t* p, int a) { __builtin_nontemporal_store(a, p); }
typedef float v4f_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void store_nt(float4* p, float4 q) {
  __builtin_nontemporal_store(__builtin_bit_cast(v4f_t, q), reinterpret_cast<v4f_t*>(p));
}

// DPP quad permutations (the four lanes of a quad hold the corners of one
// quad face): every lane of the quad reads lane K / lane i+1 / lane i-1.
template <int K>
__device__ __forceinline__ float4 quad_lane(float4 x) {
  constexpr int ctrl = K * 0x55;
  return make_float4(__int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x.x), ctrl, 0xF, 0xF, false)),
                     __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x.y), ctrl, 0xF, 0xF, false)),
                     __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x.z), ctrl, 0xF, 0xF, false)),
                     __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x.w), ctrl, 0xF, 0xF, false)));
}
__device__ __forceinline__ float4 quad_next(float4 x) {
  constexpr int ctrl = 0x39;  // [1, 2, 3, 0]
  return make_float4(__int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x.x), ctrl, 0xF, 0xF, false)),
                     __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x.y), ctrl, 0xF, 0xF, false)),
                     __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x.z), ctrl, 0xF, 0xF, false)),
                     __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x.w), ctrl, 0xF, 0xF, false)));
}
__device__ __forceinline__ float4 quad_prev(float4 x) {
  constexpr int ctrl = 0x93;  // [3, 0, 1, 2]
  return make_float4(__int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x.x), ctrl, 0xF, 0xF, false)),
                     __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x.y), ctrl, 0xF, 0xF, false)),
                     __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x.z), ctrl, 0xF, 0xF, false)),
                     __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x.w), ctrl, 0xF, 0xF, false)));
}
template <int K>
__device__ __forceinline__ int32_t quad_lane_i(int32_t x) {
  return __builtin_amdgcn_mov_dpp(x, K * 0x55, 0xF, 0xF, false);
}
__device__ __forceinline__ int32_t quad_next_i(int32_t x) { return __builtin_amdgcn_mov_dpp(x, 0x39, 0xF, 0xF, false); }
__device__ __forceinline__ int32_t quad_prev_i(int32_t x) { return __builtin_amdgcn_mov_dpp(x, 0x93, 0xF, 0xF, false); }

// entry k of the next level's M^T rows: (corner, in-neighbour), or the corner
// alone when those rows are read by the last level's kernel only
__device__ __forceinline__ void put_next_row(const RefineView& R, int64_t k, int2 x) {
  if (R.next_rows_x)
    reinterpret_cast<int32_t*>(R.ntrow)[k] = x.x;
  else
    R.ntrow[k] = x;
}

// Per-segment constants of a refine thread, all read from the segment table
// up front: a table read issued after a store would wait for that store.
struct SegK {
  int32_t vb, fb, cb, snv, snf, snnz, emax, off;
  int64_t eb;
  float4* dst_verts;
  int32_t* dst_ids;
  int32_t* dst_ptr;
  int32_t* dst_vals;
  int32_t ncb, nvb, neb;  // next level's union bases (ncb < 0: the mesh finishes here)
  int64_t own;  // base in the next level's edge owners, < 0: not wanted
  bool next, dst_final;
};

template <bool ONE>
__device__ __forceinline__ SegK seg_consts(const SegTable& seg, int32_t t) {
  SegK K;
  const SegDesc* __restrict__ S = corner_seg<ONE>(seg, t);
  K.vb = (int32_t)S->vb;
  K.fb = (int32_t)S->fb;
  K.cb = (int32_t)S->cb;
  K.snv = S->nv;
  K.snf = S->nf;
  K.snnz = (int32_t)S->nnz;
  K.emax = S->ne > 0 ? (int32_t)S->ne - 1 : 0;
  K.off = (int32_t)S->id_offset;
  K.eb = S->eb;
  K.dst_verts = to_global(S->dst_verts);
  K.dst_ids = to_global(S->dst_ids);
  K.dst_ptr = to_global(S->dst_ptr);
  K.dst_vals = to_global(S->dst_vals);
  K.ncb = (int32_t)S->next_cb;
  K.nvb = (int32_t)S->next_vb;
  K.neb = (int32_t)S->next_eb;
  K.next = S->next_cb >= 0;
  K.dst_final = S->dst_final != 0;
  K.own = S->next_own;
  return K;
}

// Everything one corner's stores need, loaded beforehand.
struct CornerIn {
  int32_t t, f, tn, tp;   // corner, face, successor / predecessor corner
  int32_t v, w, u;        // its vertex, out- and in-neighbour
  int32_t e1, e0, s1, s0; // out / in edge ids and twin corners
  int32_t g1, g0, n1, ns0;  // twin faces, successors of the twins
  int32_t bl1, bl0;       // boundary edges before e1 / e0
  int32_t mp_t, mp_s0;    // M^T positions of t and s0 (SLAK, next level)
  bool own;               // this half-edge writes edge e1
  float4 plo, phi, fa, fz;  // edge point inputs (own only)
};

// First round of a corner's loads: ids and (edge, twin) pairs already in
// hand; derives twins' faces and decides ownership.
template <bool QUAD>
__device__ __forceinline__ void corner_topology(const RefineView& R, const SegK& K, CornerIn& c, int2 c1, int2 c0) {
  c.e1 = clampi(c1.x, K.emax);
  c.e0 = clampi(c0.x, K.emax);
  c.s1 = c1.y;
  c.s0 = c0.y;
  c.g1 = c.f;
  c.g0 = c.f;
  c.n1 = 0;
  c.ns0 = 0;
  if (c.s1 >= 0) {
    int32_t x;
    corner_nbrs<QUAD>(R.fptr, R.cface, c.s1, c.g1, c.n1, x);
  }
  if (c.s0 >= 0) {
    int32_t x;
    corner_nbrs<QUAD>(R.fptr, R.cface, c.s0, c.g0, c.ns0, x);
  }
  c.own = c.s1 < 0 || c.t < c.s1;
}

// Second round: boundary ranks and SLAK positions.
template <int SCHEME>
__device__ __forceinline__ void corner_ranks(const RefineView& R, const SegK& K, CornerIn& c) {
  c.bl1 = 0;
  c.bl0 = 0;
  if (R.blk) {
    const int32_t bb = R.blk[K.eb];
    c.bl1 = R.blk[K.eb + c.e1] - bb;
    c.bl0 = R.blk[K.eb + c.e0] - bb;
  }
  c.mp_t = 0;
  c.mp_s0 = 0;
  if (SCHEME == kSLAK && K.next) {
    c.mp_t = R.mpos[c.t];
    if (c.s0 >= 0) c.mp_s0 = R.mpos[c.s0];
  }
}

// Every store of one corner t: refined quad, LAK form, edge point (owner)
// and, for a level that feeds another, the refined mesh's structure.
template <bool QUAD, int SCHEME>
__device__ __forceinline__ void corner_store(const RefineView& R, const SegK& K, const CornerIn& c) {
  const int32_t lt = c.t - K.cb, lf = c.f - K.fb;
  const int32_t epb = K.snv + K.snf + K.off, fpid = K.snv + lf + K.off;
  const bool final_level = K.dst_final;  // the caller's output: not read again here
  if (final_level) {
    store_nt(K.dst_ids + 4 * lt, c.v - K.vb + K.off, epb + c.e1, fpid, epb + c.e0);
    if (K.dst_ptr) {
      // LAK form of refined face lt (createQuadColPtr / createQuadVals,
      // LAKCatmullClarkKernels.cuh:396-431): ptr = 4 lt, vals 1..4
      store_nt(K.dst_ptr + lt, 4 * lt);
      if (lt == K.snnz - 1) store_nt(K.dst_ptr + K.snnz, 4 * K.snnz);
      if (K.dst_vals) store_nt(K.dst_vals + 4 * (int64_t)lt, 1, 2, 3, 4);
    }
  } else if (K.dst_ids) {  // null: the next level is computed without them (k_final)
    reinterpret_cast<int4*>(K.dst_ids)[lt] = make_int4(c.v - K.vb + K.off, epb + c.e1, fpid, epb + c.e0);
  }
  if (c.own) {
    float4 q;
    if (c.s1 >= 0)
      q = f4mul(f4add(f4add(f4add(c.plo, c.phi), c.fa), c.fz), 0.25f);
    else
      q = f4mul(f4add(c.plo, c.phi), 0.5f);
    float4* const dv = K.dst_verts + (K.snv + K.snf + c.e1);
    if (final_level) store_nt(dv, q);
    else *dv = q;
  }
  if (!K.next) return;

  // ---- the refined mesh's structure
  const int32_t cb = K.cb, snnz = K.snnz, snv = K.snv, snf = K.snf;
  const int32_t ncb = K.ncb, nvb = K.nvb;
  const int32_t c4 = ncb + 4 * lt;
  const int32_t tw0 = c.s1 >= 0 ? ncb + 4 * (c.n1 - cb) + 3 : -1;
  const int32_t tw1 = ncb + 4 * (c.tn - cb) + 2;
  const int32_t tw2 = ncb + 4 * (c.tp - cb) + 1;
  const int32_t tw3 = c.s0 >= 0 ? ncb + 4 * (c.s0 - cb) : -1;
  // edge point rows (the clamp only matters for inconsistent edge ids: it
  // keeps a row inside the mesh's refined M^T)
  const int32_t row1 = min(ncb + 2 * snnz + 4 * c.e1 - 2 * c.bl1, ncb + 4 * snnz - (c.s1 < 0 ? 2 : 4));
  const int32_t row0 = min(ncb + 2 * snnz + 4 * c.e0 - 2 * c.bl0, ncb + 4 * snnz - (c.s0 < 0 ? 2 : 4));
  int32_t ex, ey, ez, ew;
  if (SCHEME == kLAK) {
    const int32_t base1 = 4 * c.e1 - c.bl1, base0 = 4 * c.e0 - c.bl0;
    ex = base1 + (c.v > c.w ? 1 : 0);
    ey = base1 + 2 + ((c.s1 >= 0 && c.f > c.g1) ? 1 : 0);
    ez = base0 + 2 + ((c.s0 >= 0 && c.f > c.g0) ? 1 : 0);
    ew = base0 + (c.v > c.u ? 1 : 0);
  } else {
    ex = c.mp_t - cb;
    ey = snnz + (c.tn - cb);
    ez = snnz + lt;
    ew = c.s0 < 0 ? 2 * snnz + c.bl0 : c.mp_s0 - cb;
    // M^T positions of the refined corners
    const int32_t a1 = c4 + 1, a3 = c4 + 3;
    int32_t r1 = (ncb + 4 * (c.tn - cb) + 3 < a1) ? 1 : 0;
    if (c.s1 >= 0) r1 += (ncb + 4 * (c.s1 - cb) + 1 < a1 ? 1 : 0) + (ncb + 4 * (c.n1 - cb) + 3 < a1 ? 1 : 0);
    int32_t r3 = (ncb + 4 * (c.tp - cb) + 1 < a3) ? 1 : 0;
    if (c.s0 >= 0) r3 += (ncb + 4 * (c.s0 - cb) + 1 < a3 ? 1 : 0) + (ncb + 4 * (c.ns0 - cb) + 3 < a3 ? 1 : 0);
    reinterpret_cast<int4*>(R.nmpos)[c4 >> 2] =
        make_int4(ncb + (c.mp_t - cb), row1 + r1, ncb + snnz + lt, row0 + r3);
  }
  int4* __restrict__ o = reinterpret_cast<int4*>(R.nci + c4);
  o[0] = make_int4(ex, tw0, ey, tw1);
  o[1] = make_int4(ez, tw2, ew, tw3);
  // face point row: corner 2 of each refined quad of f, in corner order;
  // in-neighbour ep(e1)
  const int32_t nep = nvb + snv + snf;
  put_next_row(R, ncb + snnz + lt, make_int2(c4 + 2, nep + c.e1));
  bool first;
  if (QUAD) first = (c.t & 3) == 0;
  else first = c.t == R.fptr[c.f];
  if (first) R.ntptr[nvb + snv + lf] = ncb + snnz + lt;
  int32_t* __restrict__ nbnd = R.nbnd;
  const int32_t neb = K.neb;
  if (SCHEME == kSLAK && nbnd) nbnd[neb + snnz + lt] = 0;  // face point edges are interior
  if (c.own) {
    R.ntptr[nep + c.e1] = row1;
    if (SCHEME == kLAK && K.own >= 0 && c.s1 >= 0) {
      // the half-edges of the refined edges 4 e1 + 0 .. 3 (closed mesh): to
      // the lower and the higher end, to the lower and the higher face
      const int32_t s4 = ncb + 4 * (c.s1 - cb), n4 = ncb + 4 * (c.n1 - cb), tn4 = ncb + 4 * (c.tn - cb);
      auto pair = [](int32_t x, int32_t y) __attribute__((always_inline)) { return make_int2(min(x, y), max(x, y)); };
      const int2 ev = pair(c4, n4 + 3), ew = pair(s4, tn4 + 3), ef = pair(c4 + 1, tn4 + 2), eg = pair(s4 + 1, n4 + 2);
      const bool vw = c.v > c.w, fg = c.f > c.g1;
      int4* __restrict__ o4 = reinterpret_cast<int4*>(R.nown + (K.own + 4 * (int64_t)c.e1));
      const int2 l0 = vw ? ew : ev, l1 = vw ? ev : ew, l2 = fg ? eg : ef, l3 = fg ? ef : eg;
      o4[0] = make_int4(l0.x, l0.y, l1.x, l1.y);
      o4[1] = make_int4(l2.x, l2.y, l3.x, l3.y);
    }
    int2 a0 = make_int2(c4 + 1, nvb + (c.v - K.vb));
    int2 a1 = make_int2(ncb + 4 * (c.tn - cb) + 3, nvb + snv + lf);
    if (a1.x < a0.x) {
      int2 x = a0;
      a0 = a1;
      a1 = x;
    }
    auto q = [&](int k, int2 x) __attribute__((always_inline)) { put_next_row(R, row1 + k, x); };
    if (c.s1 < 0) {
      q(0, a0);
      q(1, a1);
    } else {
      int2 b0 = make_int2(ncb + 4 * (c.s1 - cb) + 1, nvb + (c.w - K.vb));
      int2 b1 = make_int2(ncb + 4 * (c.n1 - cb) + 3, nvb + snv + (c.g1 - K.fb));
      if (b1.x < b0.x) {
        int2 x = b0;
        b0 = b1;
        b1 = x;
      }
      // merge two sorted pairs
      const bool alo = a0.x < b0.x, ahi = a1.x > b1.x;
      const int2 m0 = alo ? a0 : b0, m3 = ahi ? a1 : b1;
      const int2 l = alo ? b0 : a0, h = ahi ? b1 : a1;
      const bool lh = l.x < h.x;
      q(0, m0);
      q(1, lh ? l : h);
      q(2, lh ? h : l);
      q(3, m3);
    }
    if (nbnd) {
      // the refined mesh has snnz + 2 ne edges
      const int32_t nlast = neb + snnz + 2 * (K.emax + 1) - 1;
      if (SCHEME == kLAK) {
        const int32_t base1 = min(neb + 4 * c.e1 - c.bl1, nlast - (c.s1 < 0 ? 2 : 3));
        // the next level's boundary ranks, not its flags: the halves of the
        // bl(e) boundary edges before e, and e's own two come first. (Against
        // flags and a scan launch per level: open grid 301 x 203, 3 levels 124 ->
        // 118 us a call, 64 x 64, 4 levels 108 -> 100, 500 x 400 unchanged.)
        const int32_t b = c.s1 < 0 ? 1 : 0, bl = 2 * c.bl1;
        nbnd[base1] = bl;
        nbnd[base1 + 1] = bl + b;
        nbnd[base1 + 2] = bl + 2 * b;
        if (c.s1 >= 0) nbnd[base1 + 3] = bl;
      } else if (c.s1 < 0) {
        nbnd[min(neb + 2 * snnz + c.bl1, nlast)] = 1;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// refine: for every corner t of face f, v -> w the corner's out-half-edge
// (edge e1, twin s1), u -> v the in-half-edge (edge e0, twin s0).
//   refined quad t = (v, ep(e1), fp(f), ep(e0))   in the mesh's local numbering
//   edge point e1  (written by the half-edge min(t, s1), or t on the boundary)
//                  = (P_lo + P_hi + fp(face of lo->hi) + fp(face of hi->lo)) / 4,
//                    (P_lo + P_hi) / 2 on the boundary
// and for a level that feeds another, in closed form:
//   twins          4t -> 4 next(s1) + 3, 4t+1 -> 4 next(t) + 2,
//                  4t+2 -> 4 prev(t) + 1, 4t+3 -> 4 s0
//   LAK edge ids   edge point e owns its edges to the two end points, then to
//                  the face points, ranked by the smaller id: base(e) = 4e - bl(e)
//   LAK bl(e)      of its edges: 2 bl(e), for a boundary edge e + 0, 1, 2
//   SLAK edge ids  vertices own one edge per corner, numbered by the corner's
//                  M^T storage position; face points one per corner
//                  (nnz + corner); boundary edge points one (2 nnz + bl(e))
//   M^T rows       face point f: its corners 4t+2; edge point e: 4t+1,
//                  4 next(t) + 3 of both half-edges, sorted (row 2 nnz + 4e - 2 bl(e))
//   M^T positions  (SLAK) 4t keeps t's, 4t+2 -> nnz + t, 4t+1 / 4t+3 -> rank
//                  in their edge point's row
// bl(e) = boundary edges with a smaller id (0 on closed levels). One thread
// per corner, so that each store instruction of a wave covers contiguous
// memory; every load is issued before the first store.

template <bool QUAD, int SCHEME, bool ONE>
__device__ __forceinline__ void refine_item(const RefineView& R, int64_t t64) {
  if (t64 >= R.nnz) return;
  CornerIn c;
  c.t = (int32_t)t64;
  corner_nbrs<QUAD>(R.fptr, R.cface, c.t, c.f, c.tn, c.tp);
  const SegK K = seg_consts<ONE>(R.seg, c.t);
  c.v = R.ids[c.t];
  const int2 c1 = R.ci[c.t];
  if (QUAD) {
    // the face's other corners are the quad's other lanes (nnz = 4 nf, and
    // blocks start on a face): w, u and the in-half-edge by DPP, not loads
    c.w = quad_next_i(c.v);
    c.u = quad_prev_i(c.v);
    corner_topology<QUAD>(R, K, c, c1, make_int2(quad_prev_i(c1.x), quad_prev_i(c1.y)));
  } else {
    c.w = R.ids[c.tn];
    c.u = R.ids[c.tp];
    corner_topology<QUAD>(R, K, c, c1, R.ci[c.tp]);
  }
  const bool vlo = c.v < c.w;
  const float4* __restrict__ fp = K.dst_verts + K.snv;  // face points, by mesh-local face
  if (c.own) {
    const float4 Pv = R.P[c.v], Pw = R.P[c.w];
    c.plo = vlo ? Pv : Pw;
    c.phi = vlo ? Pw : Pv;
    if (c.s1 >= 0) {
      c.fa = fp[(vlo ? c.f : c.g1) - K.fb];
      c.fz = fp[(vlo ? c.g1 : c.f) - K.fb];
    }
  }
  corner_ranks<SCHEME>(R, K, c);
  corner_store<QUAD, SCHEME>(R, K, c);
}

// vertex: one thread per vertex v with M^T row (t_i, u_i), i < n, sorted.
//   interior  q = ((sum_i fp(face t_i) + sum_i P[u_i]) / n + P[v] (n - 2)) / n
//   boundary  q = 3/4 P[v] + 1/8 (neighbours across boundary edges)
// and for a level that feeds another: the vertex's refined M^T row (corners
// 4 t_i, in-neighbours ep(e0(t_i))) and, for SLAK, the boundary flags of the
// edges it owns. The first kVertexRegs row entries and everything they gather
// are loaded before any store; longer rows loop.
constexpr int kVertexRegs = 4;

template <bool QUAD, int SCHEME, bool NEXT, bool BND, bool ONE>
__device__ __forceinline__ void vertex_item(const RefineView& R, int32_t v) {
  if (v >= R.nv) return;
  // the segment's constants, all read before the first store (a table read
  // issued after a store would wait for that store)
  const SegDesc* __restrict__ S = vertex_seg<ONE>(R.seg, v);
  const int32_t vb = (int32_t)S->vb, fb = (int32_t)S->fb, cb = (int32_t)S->cb;
  const int32_t snv = S->nv, snf = S->nf;
  const int32_t semax = S->ne > 0 ? (int32_t)S->ne - 1 : 0;
  float4* __restrict__ dst = to_global(S->dst_verts);
  const bool dst_final = S->dst_final != 0;
  const int32_t ncb = NEXT ? (int32_t)S->next_cb : -1, nvb = NEXT ? (int32_t)S->next_vb : 0;
  const int32_t neb = NEXT ? (int32_t)S->next_eb : 0;
  const float4* __restrict__ fpts = dst + snv;  // face points, by mesh-local face
  const float4* __restrict__ P = R.P;
  const int2* __restrict__ ci = R.ci;
  // NEXT: some mesh of the level continues (R.ntptr set); BND: the level has a
  // boundary (R.blk set)
  const bool next = NEXT && ncb >= 0;
  constexpr bool bnd_level = BND;
  constexpr bool need_prev = NEXT || BND;  // (edge, twin) of the in-half-edge
  constexpr bool need_own = BND;           // (edge, twin) of the out-half-edge
  const int32_t p0 = R.tptr[v];
  const int n = R.tptr[v + 1] - p0;
  const int2* __restrict__ row = R.trow + p0;
  const float4 Pv = P[v];
  auto face = [&](int32_t t) __attribute__((always_inline)) { return (QUAD ? (t >> 2) : R.cface[t]) - fb; };
  auto prevc = [&](int32_t t) __attribute__((always_inline)) {
    int32_t f, tn, tp;
    corner_nbrs<QUAD>(R.fptr, R.cface, t, f, tn, tp);
    return tp;
  };
  // the in-half-edges give the refined row's in-neighbours (and the boundary
  // rule): not needed when the next level's rows are corners alone
  const bool load_cp = BND || (NEXT && !R.next_rows_x);
  int2 e[kVertexRegs], cp[kVertexRegs], co[kVertexRegs];
  float4 a[kVertexRegs], b[kVertexRegs];
#pragma unroll
  for (int i = 0; i < kVertexRegs; ++i)
    if (i < n) e[i] = row[i];
#pragma unroll
  for (int i = 0; i < kVertexRegs; ++i)
    if (i < n) {
      a[i] = fpts[face(e[i].x)];
      b[i] = P[e[i].y];
      if (need_prev && load_cp) cp[i] = ci[prevc(e[i].x)];
      if (need_own) co[i] = ci[e[i].x];
    }
  bool boundary = false;
  if (bnd_level) {
#pragma unroll
    for (int i = 0; i < kVertexRegs; ++i)
      if (i < n) boundary |= co[i].y < 0 || cp[i].y < 0;
    for (int i = kVertexRegs; i < n; ++i) boundary |= ci[row[i].x].y < 0 || ci[prevc(row[i].x)].y < 0;
  }
  float4 q;
  if (!boundary) {
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < kVertexRegs; ++i)
      if (i < n) s = f4add(s, a[i]);
    for (int i = kVertexRegs; i < n; ++i) s = f4add(s, fpts[face(row[i].x)]);
#pragma unroll
    for (int i = 0; i < kVertexRegs; ++i)
      if (i < n) s = f4add(s, b[i]);
    for (int i = kVertexRegs; i < n; ++i) s = f4add(s, P[row[i].y]);
    const float nf = (float)n;
    q = f4div(f4add(f4div(s, nf), f4mul(Pv, nf - 2.0f)), nf);
  } else {
    q = f4mul(Pv, 0.75f);
    for (int i = 0; i < n; ++i) {
      const int32_t t = row[i].x;
      if (ci[t].y < 0) {
        int32_t f, tn, tp;
        corner_nbrs<QUAD>(R.fptr, R.cface, t, f, tn, tp);
        q = f4add(q, f4mul(P[R.ids[tn]], 0.125f));
      }
    }
    for (int i = 0; i < n; ++i)
      if (ci[prevc(row[i].x)].y < 0) q = f4add(q, f4mul(P[row[i].y], 0.125f));
  }
  // end of the next level's M^T: written with the last vertex, which every
  // union that feeds a level has (a union without faces has no corner items)
  if (NEXT && v == R.nv - 1) R.ntptr[R.next_nv] = R.next_nnz;
  if (!next && dst_final) {
    store_nt(dst + (v - vb), q);
    return;
  }
  dst[v - vb] = q;
  if (!next) return;

  const int32_t nep = nvb + snv + snf;
  const int32_t emax = semax;
  const int32_t pos = p0 - cb;  // mesh-local M^T storage position of the row
  R.ntptr[nvb + (v - vb)] = ncb + pos;
  const int64_t nrow = (int64_t)ncb + pos;  // first entry of the refined row
  int32_t* __restrict__ nbnd = (SCHEME == kSLAK) ? R.nbnd : nullptr;
#pragma unroll
  for (int i = 0; i < kVertexRegs; ++i)
    if (i < n) {
      put_next_row(R, nrow + i, make_int2(ncb + 4 * (e[i].x - cb), load_cp ? nep + clampi(cp[i].x, emax) : 0));
      if (nbnd) nbnd[neb + pos + i] = co[i].y < 0 ? 1 : 0;
    }
  for (int i = kVertexRegs; i < n; ++i) {
    const int32_t t = row[i].x;
    put_next_row(R, nrow + i, make_int2(ncb + 4 * (t - cb), load_cp ? nep + clampi(ci[prevc(t)].x, emax) : 0));
    if (nbnd) nbnd[neb + pos + i] = ci[t].y < 0 ? 1 : 0;
  }
}

// One launch per level: the refine items (one per corner) and the vertex
// items (one per vertex) are independent once the face points exist, and they
// write disjoint outputs. Their blocks are interleaved in proportion over the
// grid, so write-bound refine waves and gather-bound vertex waves share the
// machine (share_ratio).
template <bool QUAD, int SCHEME, bool NEXT, bool BND, bool ONE>
__global__ void __launch_bounds__(kBlock) k_level(RefineView R) {
  if (stopped(R.stop)) return;
  const int32_t b = (int32_t)(NEXT ? block_index<kRemapLevel>() : block_index<kRemapPositions>());
  const int32_t before = share_of(b, R.vratio), after = share_of(b + 1, R.vratio);
  if (after > before) {
    int32_t end;
    const int32_t v = run_block(R.runs, before, end) + (int32_t)threadIdx.x;
    vertex_item<QUAD, SCHEME, NEXT, BND, ONE>(R, v < end ? v : R.nv);
  } else {
    refine_item<QUAD, SCHEME, ONE>(R, (int64_t)(b - before) * kBlock + threadIdx.x);
  }
}

// ---------------------------------------------------------------------------
// A level in closed form from the mesh M two levels before it (one mesh,
// or several through a device table): the output level (IDS:
// quads, LAK form, positions) or the level before it (positions only). M1
// (the refinement of M, whose positions P1 are in hand; its ids and
// structure are never written) has corners 4t + k for the corners t of M:
//   quad t of M1   (v, ep(e1), fp(F), ep(e0))  in M1 vertex ids
//   M1 edge ids    corner 4t + k leaves along E1[k] = (ex, ey, ez, ew) and
//                  enters along E0[k] = (ew, ex, ey, ez), the ids the refine
//                  items give M1 (LAK: 4e - bl(e) + rank, SLAK: M^T positions)
//   output quad    of M1 corner 4t + k: (vertex, ep'(E1[k]), fp'(t), ep'(E0[k]))
// One lane per corner t of M computes the face point of M1 face t from its
// four corners (the fourth comes from the previous lane) and its four output
// quads (64 contiguous bytes, written out by the block through LDS). The
// owner of edge e1 of M (t < twin, or no twin) writes the edge points of the
// three or four M1 edges around ep(e1) (both halves of e1 and the edges to
// fp(F) and fp(G); for SLAK each lane writes its own edge to fp(F) instead),
// contiguous for LAK, and the vertex point of ep(e1), from the same nine
// positions. Lane 0 of each quad writes the vertex
// point of fp(F) from its four lanes. Vertex items remain only for the
// vertices of M. Every sum adds the same terms in the same order as the
// refine and vertex items of M1 would: the results are the same bits.
// M may be the caller's polygons (second level): the same closed forms with
// the neighbours of a corner through cface / fptr instead of lane exchange,
// and one more run of items for the vertex points of the face points. Against
// the refine and vertex items of M1, which read M1's structure (4 corners for
// each of M's) and needed it written: 4096 meshes of levels 1 to 4, second
// level 1340 (face points, items) -> 880 us and first level 1000 -> 749 (meshes
// of two levels write no structure, the others rows of corners alone); 16
// serve meshes 2950 -> 2680 us a call; no difference on calls of one small mesh.

__device__ __forceinline__ float4 f4sel(bool c, float4 a, float4 b) { return c ? a : b; }
// face point of a quad from its corners' positions in corner order (the sum
// and division k_faces uses)
__device__ __forceinline__ float4 face_point(float4 a, float4 b, float4 c, float4 d) {
  return f4div(f4add(f4add(f4add(a, b), c), d), 4.0f);
}

constexpr int kStageStride = 5;  // int4 per lane in the staging area (4 used; 5 spreads the banks)

struct Quads4 {
  int4 a, b, c, d;
};

// Lanes exchange positions through LDS (quads or rows of 16 lanes, so inside one wave):
// orders the accesses for the compiler, the hardware keeps a wave's in order.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// face, successor and predecessor of a mesh's corner t (all mesh-local)
template <bool QUAD>
__device__ __forceinline__ void final_nbrs(const FinalView& V, const FinalMesh& S, int32_t t, int32_t& f, int32_t& tn,
                                           int32_t& tp) {
  if (QUAD) {
    corner_nbrs<true>(nullptr, nullptr, t, f, tn, tp);
  } else {
    const int32_t cb = (int32_t)S.cb;
    corner_nbrs<false>(V.fptr, V.cface, cb + t, f, tn, tp);
    f -= (int32_t)S.fb;
    tn -= cb;
    tp -= cb;
  }
}

// Corner t (mesh-local) of M in mesh S: returns its 16 output ids (IDS),
// which the block stages in LDS.
// rows: this lane's quad of lanes' 4 x kStageStride float4 of LDS (QUAD, LAK).
template <bool QUAD, int SCHEME, bool BND, bool IDS, bool EARLY>
__device__ __forceinline__ Quads4 final_corner(const FinalView& V, const FinalMesh& S, int32_t t, float4* rows) {
  // QUAD: every lane of a quad runs (nnz = 4 nf, meshes and blocks hold whole
  // quads): the quad's four lanes load their own corner once; w (next corner's
  // vertex), u and the in-half-edge's (edge, twin) come from the
  // neighbouring lanes. Polygons: each lane loads its neighbours' itself (they
  // are in the lines the neighbouring lanes load).
  const int64_t cb = S.cb;
  const int32_t vb = (int32_t)S.vb;
  int32_t F, tn, tp;
  final_nbrs<QUAD>(V, S, t, F, tn, tp);
  const int32_t* __restrict__ ids = V.ids + cb;
  const int2* __restrict__ ci = V.ci + cb;
  const int32_t v = ids[t] - vb;
  const int32_t w = QUAD ? quad_next_i(v) : ids[tn] - vb;
  const int32_t u = QUAD ? quad_prev_i(v) : IDS && SCHEME == kLAK ? ids[tp] - vb : 0;
  const int2 c1 = ci[t];
  const int2 c0 = QUAD ? make_int2(quad_prev_i(c1.x), quad_prev_i(c1.y)) : ci[tp];
  const int32_t emax = S.ne > 0 ? S.ne - 1 : 0;
  const int32_t e1 = clampi(c1.x, emax), e0 = clampi(c0.x, emax);
  // twins are union corners
  const int32_t s1 = c1.y >= 0 ? (int32_t)(c1.y - cb) : -1, s0 = c0.y >= 0 ? (int32_t)(c0.y - cb) : -1;
  const bool own = s1 < 0 || t < s1;
  // faces across e1 and e0, next(s1) and prev(s1)
  int32_t g1 = F, g0 = F, n1 = 0, p1 = 0;
  if (QUAD) {
    g1 = s1 >= 0 ? (s1 >> 2) : F;
    g0 = s0 >= 0 ? (s0 >> 2) : F;
    n1 = s1 >= 0 ? ((s1 & ~3) | ((s1 + 1) & 3)) : 0;
    p1 = (s1 & ~3) | ((s1 + 3) & 3);
  } else {
    if (s1 >= 0 && (own || (IDS && SCHEME == kLAK))) final_nbrs<QUAD>(V, S, s1, g1, n1, p1);
    if (s0 >= 0 && IDS && SCHEME == kLAK) g0 = V.cface[cb + s0] - (int32_t)S.fb;
  }
  const int32_t nv = S.nv, nnz = S.nnz;
  const int32_t ep0 = nv + S.nf;     // M1 vertex of the edge point of edge 0 of M
  const int32_t nv1 = ep0 + S.ne;    // M1 vertices
  const int32_t epb2 = nv1 + nnz;    // output vertex of the edge point of M1 edge 0
  const float4* __restrict__ P1 = S.P1;
  float4* __restrict__ out = S.out_verts;
  int32_t bl1 = 0, bl0 = 0;
  if (BND) {
    const int32_t* __restrict__ blk = V.blk + S.eb;
    const int32_t bb = blk[0];
    bl1 = blk[e1] - bb;
    bl0 = blk[e0] - bb;
  }
  int32_t mp_t = 0, mp_s0 = 0, mp_s1 = 0;  // mesh-local M^T positions
  if (SCHEME == kSLAK) {
    const int32_t* __restrict__ mpos = V.mpos + cb;
    mp_t = mpos[t] - (int32_t)cb;
    if (s0 >= 0) mp_s0 = mpos[s0] - (int32_t)cb;
    if (own && s1 >= 0) mp_s1 = mpos[s1] - (int32_t)cb;
  }
  int2 cs0 = make_int2(0, 0), cn1 = make_int2(0, 0);  // (edge, twin) of prev(s1) and next(s1)
  if (own && s1 >= 0) {
    cs0 = ci[p1];
    cn1 = ci[n1];
  }
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  const float4 Pe = P1[ep0 + e1];   // ep(e1)
  const float4 Pv = P1[v];
  const float4 PF = P1[nv + F];     // fp(F)
  // across e1: fp(G) and the edge points of prev(s1) and next(s1). EARLY:
  // loaded before the first store, since a wait for a load also waits for
  // the stores issued before it (more registers: one wave fewer per SIMD)
  float4 PG = zero, Pa = zero, Pb = zero;
  if (EARLY && own && s1 >= 0) {
    PG = P1[nv + g1];
    Pa = P1[ep0 + clampi(cs0.x, emax)];
    Pb = P1[ep0 + clampi(cn1.x, emax)];
  }
  // w is the vertex of the next corner, ep(e0) the edge point of the previous
  // one; the M1 face of the next corner is needed around ep(e1)
  const bool next_face = own || SCHEME == kSLAK;
  float4 Pw = zero, Pu, fptn = zero;
  if (QUAD) {
    Pw = quad_next(Pv);
    Pu = quad_prev(Pe);
  } else {
    Pu = P1[ep0 + e0];
    if (next_face) {
      Pw = P1[w];
      fptn = face_point(Pw, P1[ep0 + clampi(ci[tn].x, emax)], PF, Pe);
    }
  }
  // face point of M1 face t = (v, ep(e1), fp(F), ep(e0)), as k_faces forms it;
  // it is an output position too
  const float4 fpt = face_point(Pv, Pe, PF, Pu);
  if (QUAD) fptn = quad_next(fpt);
  if (IDS)
    store_nt(out + (nv1 + t), fpt);  // (1 KB a wave; the partial lines of the others stay cached)
  else
    out[nv1 + t] = fpt;
  // vertex point of fp(F): row 4t'+2 for the corners t' of F in order,
  // in-neighbours ep(e1(t')); never on the boundary. Every lane of the quad
  // forms the sum from the quad's lanes in corner order (each term consumed
  // as it arrives), lane 0 stores it (polygons: final_face).
  if (QUAD) {
    float4 s = zero;
    s = f4add(s, quad_lane<0>(fpt));
    s = f4add(s, quad_lane<1>(fpt));
    s = f4add(s, quad_lane<2>(fpt));
    s = f4add(s, quad_lane<3>(fpt));
    s = f4add(s, quad_lane<0>(Pe));
    s = f4add(s, quad_lane<1>(Pe));
    s = f4add(s, quad_lane<2>(Pe));
    s = f4add(s, quad_lane<3>(Pe));
    if ((t & 3) == 0) out[nv + F] = f4div(f4add(f4div(s, 4.0f), f4mul(PF, 2.0f)), 4.0f);
  }
  // across e1: M1 faces s1 = (w, ep(e1), fp(G), ep(e0(s1))) and
  // next(s1) = (v, ep(e1(next(s1))), fp(G), ep(e1))
  float4 fps = zero, fpsn = zero;
  if (own && s1 >= 0) {
    if (!EARLY) {
      PG = P1[nv + g1];
      Pa = P1[ep0 + clampi(cs0.x, emax)];
      Pb = P1[ep0 + clampi(cn1.x, emax)];
    }
    fps = face_point(Pw, Pe, PG, Pa);
    fpsn = face_point(Pv, Pb, PG, Pe);
  }

  // M1 edge ids of the corners 4t .. 4t+3 (as the refine items number M1)
  int32_t ex, ey, ez, ew;
  if (!IDS) {
    ex = ey = ez = ew = 0;
  } else if (SCHEME == kLAK) {
    const int32_t base1 = 4 * e1 - bl1, base0 = 4 * e0 - bl0;
    ex = base1 + (v > w ? 1 : 0);
    ey = base1 + 2 + ((s1 >= 0 && F > g1) ? 1 : 0);
    ez = base0 + 2 + ((s0 >= 0 && F > g0) ? 1 : 0);
    ew = base0 + (v > u ? 1 : 0);
  } else {
    ex = mp_t;
    ey = nnz + tn;
    ez = nnz + t;
    ew = s0 < 0 ? 2 * nnz + bl0 : mp_s0;
  }
  // the four output quads of M1 face t
  Quads4 q4{};
  if (IDS) {
    const int32_t eb2 = epb2;
    const int32_t x0 = v, x1 = ep0 + e1, x2 = nv + F, x3 = ep0 + e0, fid = nv1 + t;
    // the block stages them in LDS and writes them out as 1 KB runs
    // (64-byte pieces per lane, stored directly, cost several times more)
    q4.a = make_int4(x0, eb2 + ex, fid, eb2 + ew);
    q4.b = make_int4(x1, eb2 + ey, fid, eb2 + ex);
    q4.c = make_int4(x2, eb2 + ez, fid, eb2 + ey);
    q4.d = make_int4(x3, eb2 + ew, fid, eb2 + ez);
  }
  if (SCHEME == kSLAK) {
    // the M1 edge from ep(e1) to fp(F), SLAK slot nnz + next(t): every lane
    // writes its own, so a wave stores 1 KB of consecutive slots (the owner
    // of e1 would form the same sum, in the same order, for both faces)
    const float4 q = f4mul(f4add(f4add(f4add(PF, Pe), fptn), fpt), 0.25f);
    float4* const d = out + epb2 + nnz + tn;
    if (IDS)
      store_nt(d, q);
    else
      *d = q;
  }
  constexpr bool kGroups = QUAD && SCHEME == kLAK;  // whole quads of lanes store the groups below
  if (!kGroups && !own) return q4;
  // edge points of the M1 edges around ep(e1), by lower end point then the
  // faces of the half-edges lower -> upper and upper -> lower
  const bool inner = !BND || s1 >= 0;
  const float4 q_vh = inner ? f4mul(f4add(f4add(f4add(Pv, Pe), fpt), fpsn), 0.25f) : f4mul(f4add(Pv, Pe), 0.5f);
  const float4 q_wh = inner ? f4mul(f4add(f4add(f4add(Pw, Pe), fps), fptn), 0.25f) : f4mul(f4add(Pw, Pe), 0.5f);
  const float4 q_fF = f4mul(f4add(f4add(f4add(PF, Pe), fptn), fpt), 0.25f);
  int32_t i_vh, i_wh, i_fF, i_fG;
  if (SCHEME == kLAK) {
    const int32_t base1 = 4 * e1 - bl1;
    i_vh = base1 + (v > w ? 1 : 0);
    i_wh = base1 + (w > v ? 1 : 0);
    i_fF = base1 + 2 + ((s1 >= 0 && F > g1) ? 1 : 0);
    i_fG = base1 + 2 + (g1 > F ? 1 : 0);
  } else {
    i_vh = mp_t;
    i_wh = s1 >= 0 ? mp_s1 : 2 * nnz + bl1;
    i_fF = nnz + tn;
    i_fG = nnz + n1;
  }
  // LAK: one 64-byte group, cached; SLAK: the two halves of e1 (the edges
  // to the face points are written above), non-temporal at the output level
  // (cached when the next kernel reads them)
  float4* __restrict__ eo = out + epb2;
  const float4 q_fG = f4mul(f4add(f4add(f4add(PG, Pe), fpsn), fps), 0.25f);
  if (kGroups) {
    // an owner's points are one group of 64 contiguous bytes: the four lanes
    // of the quad store them side by side, one owner after the other. (A lane
    // storing its own four takes four times as many L1 accesses, 128 of about
    // 600 per 64 corners, and the L1's are what the kernel is bound by: third
    // level of 4096 meshes, positions only, 803 -> 743 us.) Past the caches
    // where the launch's positions exceed them (kStreamBytes): 1024 x 1024
    // quads, 2 levels 401 -> 348 us a call; stored by single lanes that cost
    // 218 -> 324 on 512 x 256, 3 levels.
    const int32_t base1 = 4 * e1 - bl1;
    const int lane = threadIdx.x & 3;
    float4* const mine = rows + kStageStride * lane;
    if (own) {
      mine[i_vh - base1] = q_vh;
      mine[i_wh - base1] = q_wh;
      mine[i_fF - base1] = q_fF;
      if (inner) mine[i_fG - base1] = q_fG;
    }
    wave_lds_fence();
    const int32_t len = own ? (inner ? 4 : 3) : 0;
    auto put = [&](int k, int32_t b, int32_t n) __attribute__((always_inline)) {
      if (lane < n) {
        if (IDS && V.stream)
          store_nt(eo + (b + lane), rows[kStageStride * k + lane]);
        else
          eo[b + lane] = rows[kStageStride * k + lane];
      }
    };
    put(0, quad_lane_i<0>(base1), quad_lane_i<0>(len));
    put(1, quad_lane_i<1>(base1), quad_lane_i<1>(len));
    put(2, quad_lane_i<2>(base1), quad_lane_i<2>(len));
    put(3, quad_lane_i<3>(base1), quad_lane_i<3>(len));
    wave_lds_fence();  // read before the block's quads overwrite it
    if (!own) return q4;
  } else if (SCHEME == kLAK) {
    eo[i_vh] = q_vh;
    eo[i_wh] = q_wh;
    eo[i_fF] = q_fF;
    if (inner) eo[i_fG] = q_fG;
  } else if (!IDS) {
    eo[i_vh] = q_vh;
    eo[i_wh] = q_wh;
  } else {
    store_nt(eo + i_vh, q_vh);
    store_nt(eo + i_wh, q_wh);
  }
  // vertex point of ep(e1)
  float4 q;
  if (inner) {
    // row: corners 4t+1 (face t, in-neighbour v), 4tn+3 (tn, fp(F)),
    // 4s1+1 (s1, w), 4n1+3 (n1, fp(G)), sorted
    const int32_t ka = 4 * t + 1, kb = 4 * tn + 3, kc = 4 * s1 + 1, kd = 4 * n1 + 3;
    const int ra = (kb < ka) + (kc < ka) + (kd < ka);
    const int rb = (ka < kb) + (kc < kb) + (kd < kb);
    const int rc = (ka < kc) + (kb < kc) + (kd < kc);
    // the face points, then the in-neighbours, each in row order
    float4 sm = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < 4; ++i) sm = f4add(sm, f4sel(ra == i, fpt, f4sel(rb == i, fptn, f4sel(rc == i, fps, fpsn))));
#pragma unroll
    for (int i = 0; i < 4; ++i) sm = f4add(sm, f4sel(ra == i, Pv, f4sel(rb == i, PF, f4sel(rc == i, Pw, PG))));
    q = f4div(f4add(f4div(sm, 4.0f), f4mul(Pe, 2.0f)), 4.0f);
  } else {
    q = f4add(f4add(f4mul(Pe, 0.75f), f4mul(Pw, 0.125f)), f4mul(Pv, 0.125f));
  }
  out[ep0 + e1] = q;
  return q4;
}

// vertex point of a vertex v of M in the output: row 4t for its corners t in
// order, faces t, in-neighbours ep(e0(t)); on the boundary 3/4 P1[v] plus 1/8
// of ep(e1(t)) across every boundary out-edge and of ep(e0(t)) across every
// boundary in-edge
template <bool QUAD, int SCHEME, bool BND>
__device__ __forceinline__ void final_vertex(const FinalView& V, const FinalMesh& S, int32_t v) {
  const int32_t cb = (int32_t)S.cb;
  const int32_t ep0 = S.nv + S.nf;
  const int32_t emax = S.ne > 0 ? S.ne - 1 : 0;
  const float4* __restrict__ P1 = S.P1;
  const int2* __restrict__ ci = V.ci + cb;  // mesh-local corners from here on
  const int32_t p0 = V.tptr[S.vb + v];
  const int n = V.tptr[S.vb + v + 1] - p0;
  // the row's corners (union corners): (corner, in-neighbour) pairs, or
  // corners alone
  const int32_t* __restrict__ rx = V.trow_x ? V.trow_x + p0 : reinterpret_cast<const int32_t*>(V.trow + p0);
  const int rs = V.trow_x ? 1 : 2;
  const float4 Pv = P1[v];
  auto face = [&](int32_t t) __attribute__((always_inline)) {
    return QUAD ? t >> 2 : V.cface[cb + t] - (int32_t)S.fb;
  };
  auto prevc = [&](int32_t t) __attribute__((always_inline)) {
    int32_t f, tn, tp;
    final_nbrs<QUAD>(V, S, t, f, tn, tp);
    return tp;
  };
  // face point of M1 face t = (v, ep(e1(t)), fp(face of t), ep(e0(t)))
  auto fp_of = [&](int32_t t, int2 c1, float4 pe0) __attribute__((always_inline)) {
    return face_point(Pv, P1[ep0 + clampi(c1.x, emax)], P1[S.nv + face(t)], pe0);
  };
  int32_t tt[kVertexRegs];
  int2 cp[kVertexRegs], co[kVertexRegs];
  float4 a[kVertexRegs], b[kVertexRegs];
#pragma unroll
  for (int i = 0; i < kVertexRegs; ++i)
    if (i < n) tt[i] = rx[rs * i] - cb;
#pragma unroll
  for (int i = 0; i < kVertexRegs; ++i)
    if (i < n) {
      cp[i] = ci[prevc(tt[i])];
      co[i] = ci[tt[i]];
    }
#pragma unroll
  for (int i = 0; i < kVertexRegs; ++i)
    if (i < n) b[i] = P1[ep0 + clampi(cp[i].x, emax)];
  // ep(e1(t_i)) is ep(e0) of the face across e1(t_i), another face of the
  // row (but on the boundary): taken from b when an in-edge of the row has
  // the same edge id (the same position, so the same bits), else loaded
#pragma unroll
  for (int i = 0; i < kVertexRegs; ++i)
    if (i < n) {
      int m = -1;
#pragma unroll
      for (int j = 0; j < kVertexRegs; ++j)
        if (j < n && cp[j].x == co[i].x) m = j;
      float4 e1 = b[0];
#pragma unroll
      for (int j = 1; j < kVertexRegs; ++j) e1 = f4sel(m == j, b[j], e1);
      if (m < 0) e1 = P1[ep0 + clampi(co[i].x, emax)];
      a[i] = face_point(Pv, e1, P1[S.nv + face(tt[i])], b[i]);
    }
  bool boundary = false;
  if (BND) {
#pragma unroll
    for (int i = 0; i < kVertexRegs; ++i)
      if (i < n) boundary |= co[i].y < 0 || cp[i].y < 0;
    for (int i = kVertexRegs; i < n; ++i) {
      const int32_t t = rx[rs * i] - cb;
      boundary |= ci[t].y < 0 || ci[prevc(t)].y < 0;
    }
  }
  float4 q;
  if (!boundary) {
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < kVertexRegs; ++i)
      if (i < n) s = f4add(s, a[i]);
    for (int i = kVertexRegs; i < n; ++i) {
      const int32_t t = rx[rs * i] - cb;
      s = f4add(s, fp_of(t, ci[t], P1[ep0 + clampi(ci[prevc(t)].x, emax)]));
    }
#pragma unroll
    for (int i = 0; i < kVertexRegs; ++i)
      if (i < n) s = f4add(s, b[i]);
    for (int i = kVertexRegs; i < n; ++i) s = f4add(s, P1[ep0 + clampi(ci[prevc(rx[rs * i] - cb)].x, emax)]);
    const float nf = (float)n;
    q = f4div(f4add(f4div(s, nf), f4mul(Pv, nf - 2.0f)), nf);
  } else {
    q = f4mul(Pv, 0.75f);
    for (int i = 0; i < n; ++i) {
      const int2 c = ci[rx[rs * i] - cb];
      if (c.y < 0) q = f4add(q, f4mul(P1[ep0 + clampi(c.x, emax)], 0.125f));
    }
    for (int i = 0; i < n; ++i) {
      const int2 c = ci[prevc(rx[rs * i] - cb)];
      if (c.y < 0) q = f4add(q, f4mul(P1[ep0 + clampi(c.x, emax)], 0.125f));
    }
  }
  S.out_verts[v] = q;
}

// vertex point of the face point of a polygon f of M: row 4t + 2 for its
// corners t in order, faces t, in-neighbours ep(e1(t)); never on the boundary.
// (A lane per face: the corners of a polygon do not fill lanes of one wave as
// a quad's do.)
__device__ __forceinline__ void final_face(const FinalView& V, const FinalMesh& S, int32_t f) {
  const int32_t vb = (int32_t)S.vb, ep0 = S.nv + S.nf;
  const int32_t emax = S.ne > 0 ? S.ne - 1 : 0;
  const float4* __restrict__ P1 = S.P1;
  const int32_t t0 = V.fptr[S.fb + f], n = V.fptr[S.fb + f + 1] - t0;  // union corners
  const float4 PF = P1[S.nv + f];
  auto edge = [&](int32_t i) __attribute__((always_inline)) { return P1[ep0 + clampi(V.ci[t0 + i].x, emax)]; };
  auto vert = [&](int32_t i) __attribute__((always_inline)) { return P1[V.ids[t0 + i] - vb]; };
  float4 a[kVertexRegs], b[kVertexRegs];
  float4 last = edge(n - 1);
#pragma unroll
  for (int i = 0; i < kVertexRegs; ++i)
    if (i < n) {
      a[i] = vert(i);
      b[i] = edge(i);
    }
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int i = 0; i < kVertexRegs; ++i)
    if (i < n) {
      s = f4add(s, face_point(a[i], b[i], PF, last));
      last = b[i];
    }
  for (int i = kVertexRegs; i < n; ++i) {
    const float4 e = edge(i);
    s = f4add(s, face_point(vert(i), e, PF, last));
    last = e;
  }
#pragma unroll
  for (int i = 0; i < kVertexRegs; ++i)
    if (i < n) s = f4add(s, b[i]);
  for (int i = kVertexRegs; i < n; ++i) s = f4add(s, edge(i));
  const float nf = (float)n;
  S.out_verts[S.nv + f] = f4div(f4add(f4div(s, nf), f4mul(PF, nf - 2.0f)), nf);
}

// The output quads of a block's corners t0 .. t0 + cnt (of nnz in the mesh):
// staged in LDS and stored with consecutive lanes on consecutive 16-byte
// pieces; one mesh: their LAK form too.
template <bool MULTI>
__device__ __forceinline__ void store_quads(const FinalMesh& S, const Quads4& q4, int4* stage, int32_t t0, int32_t cnt,
                                            int32_t nnz) {
  const int32_t t = t0 + (int32_t)threadIdx.x;
  if ((int)threadIdx.x < cnt) {
    int4* __restrict__ o = stage + kStageStride * threadIdx.x;
    o[0] = q4.a;
    o[1] = q4.b;
    o[2] = q4.c;
    o[3] = q4.d;
  }
  // the barrier keeps the block's waves together: their stores leave as one
  // 16 KB run (wave-local staging measured 1 % slower on the batch)
  __syncthreads();
  const int nq = 4 * cnt;
  int32_t* __restrict__ dst = S.out_ids + 16 * (int64_t)t0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = j * kBlock + threadIdx.x;
    if (i < nq) {
      const int4 x = stage[kStageStride * (i >> 2) + (i & 3)];
      store_nt(dst + 4 * i, x.x, x.y, x.z, x.w);
    }
  }
  // LAK form of the block's 4 x 256 output quads (createQuadColPtr /
  // createQuadVals): every int4 of vals is (1, 2, 3, 4) and int4 q of ptr
  // is 16q + (0, 4, 8, 12), so consecutive lanes take consecutive pieces.
  // Several meshes: written by k_lak_form instead.
  if (MULTI) return;
  if (S.out_vals) {
    int32_t* __restrict__ vals = S.out_vals + 16 * (int64_t)t0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = j * kBlock + threadIdx.x;
      if (i < nq) store_nt(vals + 4 * i, 1, 2, 3, 4);
    }
  }
  if (S.out_ptr) {
    if ((int)threadIdx.x < cnt) store_nt(S.out_ptr + 4 * (int64_t)t, 16 * t, 16 * t + 4, 16 * t + 8, 16 * t + 12);
    if (t == nnz - 1) store_nt(S.out_ptr + 4 * (int64_t)nnz, 16 * nnz);
  }
}

// the mesh of this block (block-uniform) and its descriptor
template <bool MULTI>
__device__ __forceinline__ FinalMesh block_mesh(const FinalView& V, const FinalSeg*& seg) {
  if (!MULTI) {
    seg = &V.one;
    return V.one.m;
  }
  seg = V.segs + V.block_seg[block_index<kRemapFinal>()];
  FinalMesh S = seg->m;
  S.P1 = to_global(S.P1);
  S.out_verts = to_global(S.out_verts);
  S.out_ids = to_global(S.out_ids);
  return S;
}

// Corner and vertex blocks interleaved (FinalSeg). A corner block stages its
// 16 KB of output quads in LDS and stores them with consecutive lanes on
// consecutive 16-byte pieces.
template <bool QUAD, int SCHEME, bool BND, bool MULTI, bool IDS>
__global__ void __launch_bounds__(kBlock) k_final(FinalView V) {
  if (stopped(V.stop)) return;
  const FinalSeg* seg;
  const FinalMesh S = block_mesh<MULTI>(V, seg);
  const int32_t b = (int32_t)block_index<kRemapFinal>() - (MULTI ? seg->block0 : 0);
  const int32_t before = share_of(b, seg->vratio), after = share_of(b + 1, seg->vratio);
  if (after > before) {
    int32_t end;
    const int32_t v = run_block(seg->runs, before, end) + (int32_t)threadIdx.x;
    if (v >= end) return;
    if (QUAD || v < S.nv)
      final_vertex<QUAD, SCHEME, BND>(V, S, v);
    else
      final_face(V, S, v - S.nv);  // (polygons: a run of their own after the vertices)
    return;
  }
  const int32_t t0 = (b - before) * kBlock, cnt = min(kBlock, S.nnz - t0);
  const int32_t t = t0 + (int32_t)threadIdx.x;
  __shared__ int4 stage[IDS || (QUAD && SCHEME == kLAK) ? kStageStride * kBlock : 1];
  float4* const rows = reinterpret_cast<float4*>(stage) + (QUAD && SCHEME == kLAK ? kStageStride * (threadIdx.x & ~3) : 0);
  if (!IDS) {  // positions only
    if ((int)threadIdx.x < cnt) final_corner<QUAD, SCHEME, BND, false, MULTI>(V, S, t, rows);
    return;
  }
  Quads4 q4{};
  if ((int)threadIdx.x < cnt) q4 = final_corner<QUAD, SCHEME, BND, true, MULTI>(V, S, t, rows);
  store_quads<MULTI>(S, q4, stage, t0, cnt, S.nnz);
}

// ---------------------------------------------------------------------------
// The output level of a closed mesh from three levels back (LAK): N is the
// quad mesh three levels before the output, M = refine(N), M1 = refine(M),
// the output refine(M1). Only N's structure and M1's positions P1 are read;
// M's structure, which the refine items would have written and k_final reads,
// is a function of N's:
//   M corner 4t + k of N corner t (v -> w along e1, twin s1; u -> v along e0,
//   twin s0; face f): vertices (v, ep(e1), fp(f), ep(e0)), out-edges
//   4e1 + (v > w), 4e1 + 2 + (f > g1), 4e0 + 2 + (f > g0), 4e0 + (v > u),
//   faces across them next(s1), next(t), prev(t), s0
// so the level before the last two writes no structure at all, and what a
// wave gathers is shared: k_final is bound by the number of lines its lanes
// gather and scatter (without its vertex items and with neighbouring instead
// of real partners it ran at 4.7 TB/s instead of 3.0), so the work is laid
// out over rows of 16 lanes that hold everything around one face or one edge
// of N.
//   corner items  one lane per M corner, 16 lanes per N face: the face points
//                 of M1, the vertex points of M's face points, and of M's
//                 vertex fp(f) (its four corners are in the row)
//   edge items    16 lanes per N edge: the four M edges at X = ep(e), four M1
//                 edges around each: 16 edge points (one 256-byte run), the
//                 vertex points of the four M edge points and of X
//   vertex items  one lane per N vertex
// Every sum adds the same terms in the same order as k_final's: same bits.
// Face points leave by non-temporal stores (whole lines of a wave), edge points
// (64 bytes per quad of lanes) only when the launch's positions exceed what the
// 256 MB last-level cache holds (FinalView.stream, kStreamBytes): they would
// displace the positions still to be gathered, but below that line the cache
// takes them faster. Whole calls, cached -> non-temporal edge points: torus
// 256 x 256, 4 levels (268 MB of positions) 291 -> 271 us, 400 x 200 with a
// quarter triangles (300 MB) 433 -> 351, 4096 meshes 10497 -> 10366; but
// 256 x 192 (201 MB) 194 -> 207. Face points: 300 meshes 763 -> 742.

template <int N>
__device__ __forceinline__ int32_t row_ror_i(int32_t x) {  // lane i of a row of 16 reads lane i - N
  return __builtin_amdgcn_mov_dpp(x, 0x120 + N, 0xF, 0xF, false);
}
template <int N>
__device__ __forceinline__ float4 row_ror(float4 x) {
  return make_float4(__int_as_float(row_ror_i<N>(__float_as_int(x.x))), __int_as_float(row_ror_i<N>(__float_as_int(x.y))),
                     __int_as_float(row_ror_i<N>(__float_as_int(x.z))), __int_as_float(row_ror_i<N>(__float_as_int(x.w))));
}
// sizes of N, M and M1 of one mesh, as vertex bases of the output
struct DeepBase {
  int32_t epN;   // M vertex ep(edge 0 of N) = N vertices + N faces
  int32_t fM;    // M1 vertex fp(M face 0) = M vertices
  int32_t eM;    // M1 vertex ep(M edge 0)
  int32_t fM1;   // output vertex fp(M1 face 0) = M1 vertices
  int32_t eM1;   // output vertex ep(M1 edge 0)
  __device__ __forceinline__ explicit DeepBase(const FinalMesh& S) {
    epN = S.nv + S.nf;
    fM = epN + S.ne;
    eM = fM + S.nnz;
    fM1 = eM + 2 * S.nnz;
    eM1 = fM1 + 4 * S.nnz;
  }
};

// What the vector memory unit pays for is lines per four neighbouring lanes:
// a gather whose every lane has its own line takes four times as long as one
// whose quads of lanes read 64 contiguous bytes. So a row loads each position
// it needs once, neighbouring lanes neighbouring positions where there are
// any, and its lanes take their operands from LDS.

// Corner items: lane 4j + k of a row holds corner k of M face t_j = 4f + j. The
// row loads v_j, ep(e_j), fp(f), fp(t_j) (four lanes each) and, a quad per
// j, the four M edge points around ep(e_j). ex: the row's exchange, kRowEx
// float4. Returns the 16 output ids of M corner c.
constexpr int kRowEx = 65;  // loaded 0-31, M1 face points 32-47, out-edge points 48-63, one pad

__device__ __forceinline__ Quads4 deep_corner(const FinalView& V, const FinalMesh& S, int32_t c, float4* ex) {
  const DeepBase B(S);
  const int i = threadIdx.x & 15, k = i & 3, j = i >> 2, jp = (j + 3) & 3;
  const int32_t t = c >> 2, f = c >> 4, q0 = t & ~3;
  const int32_t tn = q0 | ((t + 1) & 3), tp = q0 | ((t + 3) & 3);
  const int32_t cb = (int32_t)S.cb, vb = (int32_t)S.vb, emax = S.ne > 0 ? S.ne - 1 : 0;
  const float4* __restrict__ P1 = S.P1;
  float4* __restrict__ out = S.out_verts;
  float* __restrict__ outf = reinterpret_cast<float*>(S.out_verts);
  const int32_t v = V.ids[cb + t] - vb;
  const int2 c1 = V.ci[cb + t];
  const int32_t vk = V.ids[cb + q0 + k] - vb;  // corner k of the face, for the row's loads
  const int32_t ek = clampi(V.ci[cb + q0 + k].x, emax);
  const int32_t e1 = clampi(c1.x, emax), s1 = c1.y - cb;
  const float4 p0 = P1[j == 0 ? vk : j == 1 ? B.epN + ek : j == 2 ? S.nv + f : B.fM + q0 + k];
  const float4 p1 = P1[B.eM + 4 * e1 + k];
  // the face's other corners are 4 lanes on in the row
  const int32_t w = row_ror_i<12>(v), u = row_ror_i<4>(v);
  const int32_t e0 = row_ror_i<4>(e1), s0 = row_ror_i<4>(s1);
  const int32_t n1 = (s1 & ~3) | ((s1 + 1) & 3);
  // vertex, out-edge and face across it of M corner c
  const int32_t x = k == 0 ? v : k == 1 ? B.epN + e1 : k == 2 ? S.nv + f : B.epN + e0;
  const int slot = k == 0   ? (v > w ? 1 : 0)
                   : k == 1 ? 2 + (f > (s1 >> 2) ? 1 : 0)
                   : k == 2 ? 2 + (f > (s0 >> 2) ? 1 : 0)
                            : (v > u ? 1 : 0);
  const int32_t E1 = 4 * (k < 2 ? e1 : e0) + slot;
  const int32_t G1 = k == 0 ? n1 : k == 1 ? tn : k == 2 ? tp : s0;
  const int32_t E0 = quad_prev_i(E1), G0 = quad_prev_i(G1), xn = quad_next_i(x), xp = quad_prev_i(x);
  ex[i] = p0;
  ex[16 + i] = p1;
  wave_lds_fence();
  const float4 Pv = ex[k == 0 ? j : k == 1 ? 4 + j : k == 2 ? 8 : 4 + jp];
  const float4 PF = ex[12 + j];
  const float4 Pe = ex[16 + 4 * (k < 2 ? j : jp) + slot];
  const float4 fpt = face_point(Pv, Pe, PF, quad_prev(Pe));
  ex[32 + i] = fpt;
  ex[48 + i] = Pe;
  wave_lds_fence();
  const float* const xf = reinterpret_cast<const float*>(ex);
  float sF = 0.f, sV = 0.f;  // component k of two vertex points
  {  // M face t's face point: the quad's M1 faces and out-edge points in corner order
    const float* const q = xf + 128 + 16 * j + k;
    sF = sF + q[0];
    sF = sF + q[4];
    sF = sF + q[8];
    sF = sF + q[12];
    sF = sF + q[64];
    sF = sF + q[68];
    sF = sF + q[72];
    sF = sF + q[76];
    sF = (sF / 4.0f + xf[4 * (12 + j) + k] * 2.0f) / 4.0f;
  }
  {  // M's vertex fp(f), corners 4t + 2: lanes 2, 6, 10, 14; in-neighbours the out-edge points of the lanes before
    const float* const q = xf + 128 + k;
    sV = sV + q[8];
    sV = sV + q[24];
    sV = sV + q[40];
    sV = sV + q[56];
    sV = sV + q[64 + 4];
    sV = sV + q[64 + 20];
    sV = sV + q[64 + 36];
    sV = sV + q[64 + 52];
    sV = (sV / 4.0f + xf[32 + k] * 2.0f) / 4.0f;
  }
  store_nt(out + (B.fM1 + c), fpt);
  outf[4 * (int64_t)(B.fM + t) + k] = sF;
  if (j == 0) outf[4 * (int64_t)(S.nv + f) + k] = sV;
  // M1 edges of corners 4c .. 4c + 3, then the four output quads
  const int32_t eX = B.eM1 + 4 * E1 + (x > xn ? 1 : 0), eY = B.eM1 + 4 * E1 + 2 + (t > G1 ? 1 : 0);
  const int32_t eZ = B.eM1 + 4 * E0 + 2 + (t > G0 ? 1 : 0), eW = B.eM1 + 4 * E0 + (x > xp ? 1 : 0);
  const int32_t fid = B.fM1 + c;
  Quads4 q;
  q.a = make_int4(x, eX, fid, eW);
  q.b = make_int4(B.eM + E1, eY, fid, eX);
  q.c = make_int4(B.fM + t, eZ, fid, eY);
  q.d = make_int4(B.eM + E0, eW, fid, eZ);
  return q;
}

// Edge items: 16 lanes per N edge e. Around X = ep(e), in turn: the M vertices
// A_j = v, fp(f), w, fp(g) and the M faces Z_j = t, next(t), s, next(s) between
// A_j and A_{j+1} (each passes A_j -> X -> A_{j+1}; t is the owner, so f < g and
// t, next(t) < s, next(s)); Y_j is the edge point of the M edge A_j X, M edge
// 4e + (v > w), 4e + 2, 4e + (w > v), 4e + 3. Around Y_j in turn: A_j, Z_j, X,
// Z_{j-1}, with the M1 faces
//   psi_0 = (A_j, Y_j, Z_j, Bin_j)        psi_1 = (X, Y_{j+1}, Z_j, Y_j)
//   psi_2 = (X, Y_j, Z_{j-1}, Y_{j-1})    psi_3 = (A_j, Bout_j, Z_{j-1}, Y_j)
// after each, Bin_j and Bout_j being the edge points of A_j's other M edges in
// Z_j and Z_{j-1}. Lane 4j + m loads the four corners of psi_m (the quads of
// lanes share lines; its neighbour of Y_j and Y_j itself are among them) and
// forms psi_m and the edge point of M1's edge from Y_j to its neighbour m,
// (neighbour + Y_j + psi_m + psi_{m-1}) / 4; the vertex points of the Y_j and of
// X are formed one component per lane, their terms picked in row order by
// address. What the kernel waits for is latency: seven waves a SIMD, each for
// its chain of half-edges, corners, positions and for the stores before its
// next loads (sending all positions' stores to a few lines, so without their
// HBM writes, gave 1.1 of 3.9 ms; half the vector instructions gave nothing).
// So a block takes two edges a row with every load before the first store:
// 4096 meshes 3.90 -> 3.69 ms. Four edges a row (79 registers instead of 61)
// 3.82, one or four without loads ahead 3.90.
constexpr int kRows = kBlock / 16;
constexpr int kEdgeIter = kDeepEdgeUnit / kRows;  // edges per row and unit
constexpr int kRowE = 33;                   // float4 of a row: neighbours of the Y 0-15, psi 16-31, one pad (rows start 4 banks apart)
constexpr int kRowX = 9 * kEdgeIter + 1;    // per edge: psi_1 and Y of j = 0 .. 3, X
constexpr int kEdgeLds = (kRowE + kRowX) * kRows;  // float4

__device__ __forceinline__ void deep_edges(const FinalView& V, const FinalMesh& S, int32_t first, int32_t cnt,
                                           float4* lds) {
  const DeepBase B(S);
  const int32_t cb = (int32_t)S.cb, vb = (int32_t)S.vb, emax = S.ne > 0 ? S.ne - 1 : 0;
  const float4* __restrict__ P1 = S.P1;
  float4* __restrict__ out = S.out_verts;
  float* __restrict__ outf = reinterpret_cast<float*>(S.out_verts);
  const int row = threadIdx.x >> 4, i = threadIdx.x & 15, m = i & 3, j = i >> 2;
  const bool odd = (j & 1) != 0, side = (j & 2) != 0;
  float4* const re = lds + row * kRowE;
  float4* const rx = lds + kRows * kRowE + row * kRowX;
  const float* const ref = reinterpret_cast<const float*>(re);
  uint32_t order = 0;  // per edge: t before next(t), s before next(s)
  // All loads of an edge come before the stores of the edge before it (a wait
  // for a load also waits for the stores issued before it): the half-edges and
  // their corners for the unit, the positions one edge ahead. A row beyond the
  // unit's edges repeats the last one and stores nothing.
  int32_t tq[kEdgeIter], sq[kEdgeIter], idq[kEdgeIter];
  int2 cq[kEdgeIter];
#pragma unroll
  for (int it = 0; it < kEdgeIter; ++it) {
    // (written whole for a closed mesh, and a replay whose edges differ stops before)
    const int2 o = V.own[S.eb + first + min(row + it * kRows, cnt - 1)];
    tq[it] = o.x - cb;
    sq[it] = o.y - cb;
  }
#pragma unroll
  for (int it = 0; it < kEdgeIter; ++it) {
    // the row's halves hold the face of t and the face of its twin, each quad
    // the face's corners from the half-edge's own on
    const int32_t a = side ? sq[it] : tq[it];
    const int32_t corner = cb + ((a & ~3) | ((a + m) & 3));
    idq[it] = V.ids[corner] - vb;
    cq[it] = V.ci[corner];
  }
  struct Row {
    int32_t Y_id;
    float4 r1, r2, r3, r4;  // the four corners of psi_m, in order
  };
  const bool even = (m & 1) == 0;
  auto load = [&](int it) __attribute__((always_inline)) {
    Row R;
    const int32_t e = first + min(row + it * kRows, cnt - 1);
    const int32_t a = side ? sq[it] : tq[it], h = a >> 2, id = idq[it];
    const int32_t ce = clampi(cq[it].x, emax), cg = (cq[it].y - cb) >> 2;  // edge, face across it
    const int32_t I0 = quad_lane_i<0>(id), I1 = quad_lane_i<1>(id), I2 = quad_lane_i<2>(id), I3 = quad_lane_i<3>(id);
    const int32_t C1 = quad_lane_i<1>(ce), C3 = quad_lane_i<3>(ce);
    const int32_t gc = quad_lane_i<1>(cg), gd = quad_lane_i<3>(cg);
    const int32_t Zc = odd ? ((a & ~3) | ((a + 1) & 3)) : a;
    R.Y_id = 4 * e + (odd ? (side ? 3 : 2) : (I0 > I1 ? 1 : 0));
    const int32_t across = row_ror_i<8>(4 * C1 + (I1 > I2 ? 1 : 0));  // the other half's
    const int32_t Bin = odd ? 4 * C1 + 2 + (h > gc ? 1 : 0) : 4 * C3 + (I0 > I3 ? 1 : 0);
    const int32_t Bout = odd ? 4 * C3 + 2 + (h > gd ? 1 : 0) : across;
    const int32_t Zq = row_ror_i<4>(Zc), Yn_id = row_ror_i<12>(R.Y_id), Yp_id = row_ror_i<4>(R.Y_id);
    R.r1 = P1[m == 0 || m == 3 ? (odd ? S.nv + h : I0) : B.epN + e];
    R.r2 = P1[B.eM + (even ? R.Y_id : m == 1 ? Yn_id : Bout)];
    R.r3 = P1[B.fM + (m < 2 ? Zc : Zq)];
    R.r4 = P1[B.eM + (!even ? R.Y_id : m == 0 ? Bin : Yp_id)];
    return R;
  };
  Row ahead = load(0);
#pragma unroll
  for (int it = 0; it < kEdgeIter; ++it) {
    const int r = row + it * kRows;
    const Row R = ahead;
    if (it + 1 < kEdgeIter) ahead = load(it + 1);
    if (r >= cnt) break;
    const bool tt = (tq[it] & 3) != 3, ss = (sq[it] & 3) != 3;
    order |= ((tt ? 1u : 0u) | (ss ? 2u : 0u)) << (2 * it);
    const float4 r1 = R.r1, r2 = R.r2, r3 = R.r3, r4 = R.r4;
    const int32_t Y_id = R.Y_id;
    const float4 psi = face_point(r1, r2, r3, r4);
    const float4 nbr = f4sel(even, r1, r3), Y = f4sel(even, r2, r4);
    const bool zfirst = j == 0 || (j == 1 && !tt) || (j == 3 && !ss);  // Z_j before Z_{j-1}
    const int32_t slot = m == 0 ? 0 : m == 2 ? 1 : ((m == 1) == zfirst ? 2 : 3);
    re[i] = nbr;
    re[16 + i] = psi;
    if (m) rx[9 * it + (m == 2 ? 8 : m == 3 ? 4 + j : j)] = f4sel(m == 1, psi, f4sel(m == 2, nbr, Y));
    const float4 q = f4mul(f4add(f4add(f4add(nbr, Y), psi), quad_prev(psi)), 0.25f);
    float4* const d = out + (B.eM1 + 4 * Y_id + slot);
    if (V.stream)
      store_nt(d, q);
    else
      *d = q;
    wave_lds_fence();
    // vertex point of Y_j, component m: the row's corners are those of the
    // lower M face first; in Z_j A_j's comes before X's, in Z_{j-1} when j is odd
    {
      const int f = 16 * j + m, g = 64 + f;
      const int r0 = odd ? 8 : 12, r1 = odd ? 12 : 8;
      const int n0 = odd ? f + 8 : f + 12, n1 = odd ? f + 12 : f + 8;  // X and Z_{j-1}
      float sum = 0.f;
      sum = sum + ref[g + (zfirst ? 0 : r0)];
      sum = sum + ref[g + (zfirst ? 4 : r1)];
      sum = sum + ref[g + (zfirst ? r0 : 0)];
      sum = sum + ref[g + (zfirst ? r1 : 4)];
      sum = sum + ref[zfirst ? f : n0];
      sum = sum + ref[zfirst ? f + 4 : n1];
      sum = sum + ref[zfirst ? n0 : f];
      sum = sum + ref[zfirst ? n1 : f + 4];
      const float y = m < 2 ? (m == 0 ? Y.x : Y.y) : (m == 2 ? Y.z : Y.w);
      outf[4 * (int64_t)(B.eM + Y_id) + m] = (sum / 4.0f + y * 2.0f) / 4.0f;
    }
    wave_lds_fence();  // read before the next edge writes
  }
  // vertex points of the X: lane i forms component m of the row's edge j
  const int r = row + j * kRows;
  if (j < kEdgeIter && r < cnt) {
    const float* const x = reinterpret_cast<const float*>(rx + 9 * j) + m;
    const int tt = (order >> (2 * j)) & 1 ? 0 : 4, ss = (order >> (2 * j)) & 2 ? 8 : 12;
    float sum = 0.f;
    sum = sum + x[tt];
    sum = sum + x[4 - tt];
    sum = sum + x[ss];
    sum = sum + x[20 - ss];
    sum = sum + x[16 + tt];
    sum = sum + x[20 - tt];
    sum = sum + x[16 + ss];
    sum = sum + x[36 - ss];
    outf[4 * (int64_t)(B.epN + first + r) + m] = (sum / 4.0f + x[32] * 2.0f) / 4.0f;
  }
}

// vertex point of a vertex v of N in the output: M corners 4t of its row's
// corners t, M1 faces (v, ep(4e1 + (v > w)), fp(M face t), ep(4e0 + (v > u)))
__device__ __forceinline__ void deep_vertex(const FinalView& V, const FinalMesh& S, int32_t v) {
  const DeepBase B(S);
  const int32_t cb = (int32_t)S.cb, vb = (int32_t)S.vb;
  const int32_t emax = S.ne > 0 ? S.ne - 1 : 0;
  const float4* __restrict__ P1 = S.P1;
  const int32_t* __restrict__ ids = V.ids + cb;
  const int2* __restrict__ ci = V.ci + cb;
  const int32_t p0 = V.tptr[vb + v];
  const int n = V.tptr[vb + v + 1] - p0;
  const int32_t* __restrict__ rx = V.trow_x ? V.trow_x + p0 : reinterpret_cast<const int32_t*>(V.trow + p0);
  const int rs = V.trow_x ? 1 : 2;
  const float4 Pv = P1[v];
  // M edges leaving v into its M face 4t, and entering it
  auto edges = [&](int32_t t, int32_t& out_e, int32_t& in_e) __attribute__((always_inline)) {
    const int32_t q0 = t & ~3;
    const int32_t tp = q0 | ((t + 3) & 3), tn = q0 | ((t + 1) & 3);
    out_e = 4 * clampi(ci[t].x, emax) + (v > ids[tn] - vb ? 1 : 0);
    in_e = 4 * clampi(ci[tp].x, emax) + (v > ids[tp] - vb ? 1 : 0);
  };
  int32_t tt[kVertexRegs], eo[kVertexRegs], ei[kVertexRegs];
  float4 a[kVertexRegs], b[kVertexRegs];
#pragma unroll
  for (int i = 0; i < kVertexRegs; ++i)
    if (i < n) tt[i] = rx[rs * i] - cb;
#pragma unroll
  for (int i = 0; i < kVertexRegs; ++i)
    if (i < n) edges(tt[i], eo[i], ei[i]);
#pragma unroll
  for (int i = 0; i < kVertexRegs; ++i)
    if (i < n) b[i] = P1[B.eM + ei[i]];
  // the out-edge's point from an in-edge already loaded, as in final_vertex
#pragma unroll
  for (int i = 0; i < kVertexRegs; ++i)
    if (i < n) {
      int k = -1;
#pragma unroll
      for (int j = 0; j < kVertexRegs; ++j)
        if (j < n && ei[j] == eo[i]) k = j;
      float4 e1 = b[0];
#pragma unroll
      for (int j = 1; j < kVertexRegs; ++j) e1 = f4sel(k == j, b[j], e1);
      if (k < 0) e1 = P1[B.eM + eo[i]];
      a[i] = face_point(Pv, e1, P1[B.fM + tt[i]], b[i]);
    }
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int i = 0; i < kVertexRegs; ++i)
    if (i < n) s = f4add(s, a[i]);
  for (int i = kVertexRegs; i < n; ++i) {
    const int32_t t = rx[rs * i] - cb;
    int32_t o, e;
    edges(t, o, e);
    s = f4add(s, face_point(Pv, P1[B.eM + o], P1[B.fM + t], P1[B.eM + e]));
  }
#pragma unroll
  for (int i = 0; i < kVertexRegs; ++i)
    if (i < n) s = f4add(s, b[i]);
  for (int i = kVertexRegs; i < n; ++i) {
    int32_t o, e;
    edges(rx[rs * i] - cb, o, e);
    s = f4add(s, P1[B.eM + e]);
  }
  const float nf = (float)n;
  S.out_verts[v] = f4div(f4add(f4div(s, nf), f4mul(Pv, nf - 2.0f)), nf);
}

// Blocks of one kind each: 256 M corners, kDeepEdgeUnit N edges, 256 N vertices
// (FinalSeg).
template <bool MULTI>
__global__ void __launch_bounds__(kBlock) k_final_deep(FinalView V) {
  if (stopped(V.stop)) return;
  const FinalSeg* seg;
  const FinalMesh S = block_mesh<MULTI>(V, seg);
  const int32_t b = (int32_t)block_index<kRemapFinal>() - (MULTI ? seg->block0 : 0);
  const int32_t before = share_of(b, seg->vratio), after = share_of(b + 1, seg->vratio);
  if (after > before) {
    int32_t end;
    const int32_t v = run_block(seg->runs, before, end) + (int32_t)threadIdx.x;
    if (v < end) deep_vertex(V, S, v);
    return;
  }
  const int32_t b1 = b - before, edges = share_of(b1, seg->eratio);
  __shared__ int4 stage[std::max(kStageStride * kBlock, kEdgeLds)];
  if (share_of(b1 + 1, seg->eratio) > edges) {
    static_assert(kEdgeIter <= 4, "a quad of the row's lanes per edge of its X");
    const int32_t first = edges * kDeepEdgeUnit;
    deep_edges(V, S, first, min(kDeepEdgeUnit, S.ne - first), reinterpret_cast<float4*>(stage));
    return;
  }
  const int32_t first = (b1 - edges) * kBlock, cnt = min(kBlock, 4 * S.nnz - first);
  Quads4 q4{};
  // (the exchange of a wave's rows lies in the LDS that the wave's own lanes stage their quads in)
  static_assert(4 * kRowEx <= 64 * kStageStride, "a wave's four rows in its staging area");
  float4* const ex = reinterpret_cast<float4*>(stage) + (threadIdx.x >> 6) * 64 * kStageStride + ((threadIdx.x >> 4) & 3) * kRowEx;
  if ((int)threadIdx.x < cnt) q4 = deep_corner(V, S, first + (int32_t)threadIdx.x, ex);
  wave_lds_fence();  // read before the quads overwrite it
  store_quads<MULTI>(S, q4, stage, first, cnt, 4 * S.nnz);
}


// The LAK form of the output quads of the meshes that share their last level's
// launch (createQuadColPtr / createQuadVals, LAKCatmullClarkKernels.cuh:396-431),
// whatever their levels: a block writes the 1024 quads of 256 items of its mesh,
// vals as int4 (1, 2, 3, 4), ptr as int4 16t + (0, 4, 8, 12). A pure streaming
// write, apart from the gathers and scattered stores of k_final. XCD-chunked
// block order: a fill of five 16-byte stores a thread reaches 6.6 TB/s that
// way, 5.8 to 6.2 with the blocks dealt round. One launch for all levels: two
// launches less on a batch of levels 1 to 4, about 6 us each when it is small.
__global__ void __launch_bounds__(kBlock) k_lak_form(const LakSeg* __restrict__ segs,
                                                     const int32_t* __restrict__ block_seg) {
  const int32_t b = (int32_t)block_index<kRemapFinal>();
  const LakSeg& seg = segs[block_seg[b]];
  const int32_t t0 = (b - seg.block0) * kBlock, cnt = min(kBlock, seg.n - t0);
  const int32_t t = t0 + (int32_t)threadIdx.x;
  const int nq = 4 * cnt;
  int32_t* __restrict__ vals = to_global(seg.vals) + 16 * (int64_t)t0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = j * kBlock + threadIdx.x;
    if (i < nq) store_nt(vals + 4 * i, 1, 2, 3, 4);
  }
  int32_t* const ptr = to_global(seg.ptr);
  if (!ptr) return;
  if ((int)threadIdx.x < cnt) store_nt(ptr + 4 * (int64_t)t, 16 * t, 16 * t + 4, 16 * t + 8, 16 * t + 12);
  if (t == seg.n - 1) store_nt(ptr + 4 * (int64_t)seg.n, 16 * seg.n);
}

// ---------------------------------------------------------------------------
// reduced / unreduced conversions of homogeneous meshes (GPU::CSCMesh::reduce /
// unreduce, include/Mesh.h:305-377): each face's (ids, vals) reordered by vals
// (reduce: ids in corner-position order) or by ids (unreduce), in place.

template <bool KEY_VALS>
__global__ void __launch_bounds__(kBlock) k_sort_faces(const int32_t* __restrict__ ptr, int32_t stride, int32_t nf,
                                                       int64_t nnz, int32_t* __restrict__ ids,
                                                       int32_t* __restrict__ vals, int* __restrict__ flags) {
  const int32_t f = (int32_t)(block_index() * blockDim.x + threadIdx.x);
  if (f >= nf) return;
  const int64_t s = ptr ? ptr[f] : (int64_t)stride * f;
  const int64_t e = ptr ? ptr[f + 1] : s + stride;
  const int n = (int)(e - s);
  if (s < 0 || e > nnz || n < 0 || n > 4) {  // homogeneous faces have 3 or 4 corners
    atomicOr(flags, kFlagBadPtr);
    return;
  }
  int32_t k[4], a[4], b[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (i < n) {
      a[i] = ids[s + i];
      b[i] = vals[s + i];
      k[i] = KEY_VALS ? b[i] : a[i];
    }
  // insertion sort by key, carrying (id, val)
#pragma unroll
  for (int i = 1; i < 4; ++i)
#pragma unroll
    for (int j = i; j > 0; --j)
      if (i < n && k[j - 1] > k[j]) {
        int32_t x = k[j]; k[j] = k[j - 1]; k[j - 1] = x;
        x = a[j]; a[j] = a[j - 1]; a[j - 1] = x;
        x = b[j]; b[j] = b[j - 1]; b[j - 1] = x;
      }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (i < n) {
      ids[s + i] = a[i];
      vals[s + i] = b[i];
    }
}

// vals[i] = 1-based corner position (i mod stride) + 1; ptr[f] = stride f
__global__ void k_fill_homogeneous(int32_t* __restrict__ ptr, int64_t nptr, int32_t* __restrict__ vals, int64_t nvals,
                                   int32_t stride) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (ptr && i < nptr) ptr[i] = (int32_t)(stride * i);
  if (vals && i < nvals) vals[i] = (int32_t)(i % stride) + 1;
}

// ---------------------------------------------------------------------------
// exclusive scan with total: out[i] = sum(in[0..i)), out[n] = sum(in)

constexpr int kScanItems = 8;
constexpr int kScanTile = kBlock * kScanItems;

__device__ __forceinline__ int64_t block_exclusive_scan(int64_t x, int64_t* lds, int64_t& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int64_t v = x;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    int64_t y = __shfl_up(v, d, 64);
    if (lane >= d) v += y;
  }
  if (lane == 63) lds[wave] = v;
  __syncthreads();
  int64_t off = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) {
    int64_t t = lds[w];
    off += (w < wave) ? t : 0;
    tot += t;
  }
  __syncthreads();
  total = tot;
  return off + v - x;
}

// Inputs up to kScanSmall items: one block of 1024 threads in one launch
// (instead of three).
constexpr int kScanSmallThreads = 1024;
constexpr int kScanSmallRounds = 8;  // int4 loads per thread
constexpr int kScanSmallRound = 4 * kScanSmallThreads;
constexpr int64_t kScanSmall = (int64_t)kScanSmallRounds * kScanSmallRound;

// Item (r, tid, j) = r * 4096 + 4 tid + j: every load and store instruction
// of a wave covers 1 KB of consecutive ints, all loads are in flight before
// the first add, the eight rounds are scanned side by side in registers, and
// wave 0 scans the 128 wave totals (rounds major) between two barriers.
__global__ void __launch_bounds__(kScanSmallThreads) k_scan_small(const int32_t* __restrict__ in, int64_t n,
                                                                  int32_t* __restrict__ out, int* __restrict__ flags) {
  constexpr int kWaves = kScanSmallThreads / 64;
  static_assert(kScanSmallRounds * kWaves == 128, "wave 0 scans two wave totals per lane");
  __shared__ int64_t wsum[kScanSmallRounds * kWaves];
  __shared__ int64_t total;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool vin = (reinterpret_cast<uintptr_t>(in) & 15) == 0;
  const bool vout = (reinterpret_cast<uintptr_t>(out) & 15) == 0;
  int4 x[kScanSmallRounds];
#pragma unroll
  for (int r = 0; r < kScanSmallRounds; ++r) {
    const int64_t i = (int64_t)r * kScanSmallRound + 4 * tid;
    if (vin && i + 3 < n) {
      x[r] = *reinterpret_cast<const int4*>(in + i);
    } else {
      x[r].x = i < n ? in[i] : 0;
      x[r].y = i + 1 < n ? in[i + 1] : 0;
      x[r].z = i + 2 < n ? in[i + 2] : 0;
      x[r].w = i + 3 < n ? in[i + 3] : 0;
    }
  }
  int64_t g[kScanSmallRounds], v[kScanSmallRounds];
#pragma unroll
  for (int r = 0; r < kScanSmallRounds; ++r) {
    g[r] = (int64_t)x[r].x + x[r].y + x[r].z + x[r].w;
    v[r] = wave_scan64(g[r]);
  }
  if (lane == 63) {
#pragma unroll
    for (int r = 0; r < kScanSmallRounds; ++r) wsum[r * kWaves + wave] = v[r];
  }
  __syncthreads();
  if (wave == 0) {  // 128 wave totals, two per lane: exclusive prefixes in place
    const int64_t a = wsum[2 * lane], b = wsum[2 * lane + 1];
    const int64_t inc = wave_scan64(a + b);
    wsum[2 * lane] = inc - a - b;
    wsum[2 * lane + 1] = inc - b;
    if (lane == 63) total = inc;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kScanSmallRounds; ++r) {
    const int64_t e0 = wsum[r * kWaves + wave] + v[r] - g[r];
    const int4 o = make_int4((int32_t)e0, (int32_t)(e0 + x[r].x), (int32_t)(e0 + x[r].x + x[r].y),
                             (int32_t)(e0 + x[r].x + x[r].y + x[r].z));
    const int64_t i = (int64_t)r * kScanSmallRound + 4 * tid;
    if (vout && i + 3 < n) {
      *reinterpret_cast<int4*>(out + i) = o;
    } else {
      if (i < n) out[i] = o.x;
      if (i + 1 < n) out[i + 1] = o.y;
      if (i + 2 < n) out[i + 2] = o.z;
      if (i + 3 < n) out[i + 3] = o.w;
    }
  }
  if (tid == 0) {
    const int64_t carry = total;
    if (carry > 0x7fffffffll) *flags = kFlagOverflow;
    out[n] = (int32_t)carry;
  }
}

// Tiles of kScanTile items: item (r, tid, j) of a tile is r * 4 kBlock + 4 tid
// + j (r < kScanRounds, j < 4), so that every load and store instruction of a
// wave covers 1 KB of consecutive ints.
constexpr int kScanRounds = kScanItems / 4;
// up to this many tiles (8 M items) the down pass sums the preceding tile
// sums itself (at most 16 per lane) instead of a partials launch
constexpr int64_t kScanFoldTiles = 4096;
static_assert(kScanRounds * 4 * kBlock == kScanTile, "tile layout");

__device__ __forceinline__ int4 scan_load4(const int32_t* __restrict__ in, int64_t i, int64_t n, bool vec) {
  if (vec && i + 3 < n) return *reinterpret_cast<const int4*>(in + i);
  return make_int4(i < n ? in[i] : 0, i + 1 < n ? in[i + 1] : 0, i + 2 < n ? in[i + 2] : 0, i + 3 < n ? in[i + 3] : 0);
}

__global__ void __launch_bounds__(kBlock) k_scan_reduce(const int32_t* __restrict__ in, int64_t n,
                                                        int64_t* __restrict__ partial) {
  __shared__ int64_t lds[kBlock / 64];
  const bool vec = (reinterpret_cast<uintptr_t>(in) & 15) == 0;
  const int64_t base = (int64_t)blockIdx.x * kScanTile + 4 * threadIdx.x;
  int4 x[kScanRounds];
#pragma unroll
  for (int r = 0; r < kScanRounds; ++r) x[r] = scan_load4(in, base + (int64_t)r * 4 * kBlock, n, vec);
  int64_t s = 0;
#pragma unroll
  for (int r = 0; r < kScanRounds; ++r) s += (int64_t)x[r].x + x[r].y + x[r].z + x[r].w;
  int64_t tot;
  block_exclusive_scan(s, lds, tot);
  if (threadIdx.x == 0) partial[blockIdx.x] = tot;
}

__global__ void __launch_bounds__(kBlock) k_scan_partials(int64_t* __restrict__ partial, int64_t ntiles,
                                                          int32_t* __restrict__ out, int64_t n, int* __restrict__ flags) {
  __shared__ int64_t lds[kBlock / 64];
  int64_t carry = 0;
  for (int64_t b = 0; b < ntiles; b += kBlock) {
    int64_t i = b + threadIdx.x;
    int64_t x = i < ntiles ? partial[i] : 0;
    int64_t tot;
    int64_t ex = block_exclusive_scan(x, lds, tot);
    if (i < ntiles) partial[i] = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0) {
    if (carry > 0x7fffffffll) *flags = kFlagOverflow;
    out[n] = (int32_t)carry;
  }
}

// FOLD: partial holds the tile sums (no partials pass); each block adds up
// the sums of the tiles before it, and block 0 also forms the total
// (out[n], the overflow flag). Without FOLD partial holds the
// exclusive tile prefixes.
template <bool FOLD>
__global__ void __launch_bounds__(kBlock) k_scan_down(const int32_t* __restrict__ in, int64_t n,
                                                      const int64_t* __restrict__ partial, int32_t* __restrict__ out,
                                                      int64_t ntiles, int* __restrict__ flags) {
  constexpr int kWaves = kBlock / 64;
  __shared__ int64_t wsum[kScanRounds * kWaves];
  __shared__ int64_t red[kBlock / 64];
  int64_t prefix = 0;
  if (FOLD) {
    int64_t acc = 0;
    for (int64_t i = threadIdx.x; i < (int64_t)blockIdx.x; i += kBlock) acc += partial[i];
    block_exclusive_scan(acc, red, prefix);
    if (blockIdx.x == 0) {
      int64_t all = 0, carry;
      for (int64_t i = threadIdx.x; i < ntiles; i += kBlock) all += partial[i];
      block_exclusive_scan(all, red, carry);
      if (threadIdx.x == 0) {
        if (carry > 0x7fffffffll) *flags = kFlagOverflow;
        out[n] = (int32_t)carry;
      }
    }
  } else {
    (void)ntiles;
    (void)flags;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool vin = (reinterpret_cast<uintptr_t>(in) & 15) == 0;
  const bool vout = (reinterpret_cast<uintptr_t>(out) & 15) == 0;
  const int64_t base = (int64_t)blockIdx.x * kScanTile + 4 * threadIdx.x;
  int4 x[kScanRounds];
#pragma unroll
  for (int r = 0; r < kScanRounds; ++r) x[r] = scan_load4(in, base + (int64_t)r * 4 * kBlock, n, vin);
  int64_t g[kScanRounds], v[kScanRounds];
#pragma unroll
  for (int r = 0; r < kScanRounds; ++r) {
    g[r] = (int64_t)x[r].x + x[r].y + x[r].z + x[r].w;
    v[r] = wave_scan64(g[r]);
  }
  if (lane == 63)
#pragma unroll
    for (int r = 0; r < kScanRounds; ++r) wsum[r * kWaves + wave] = v[r];
  __syncthreads();
  if (threadIdx.x == 0) {  // the wave totals, rounds major: exclusive prefixes in place
    int64_t run = FOLD ? prefix : partial[blockIdx.x];
    for (int k = 0; k < kScanRounds * kWaves; ++k) {
      const int64_t t = wsum[k];
      wsum[k] = run;
      run += t;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kScanRounds; ++r) {
    const int64_t e0 = wsum[r * kWaves + wave] + v[r] - g[r];
    const int4 o = make_int4((int32_t)e0, (int32_t)(e0 + x[r].x), (int32_t)(e0 + x[r].x + x[r].y),
                             (int32_t)(e0 + x[r].x + x[r].y + x[r].z));
    const int64_t i = base + (int64_t)r * 4 * kBlock;
    if (vout && i + 3 < n) {
      *reinterpret_cast<int4*>(out + i) = o;
    } else {
      if (i < n) out[i] = o.x;
      if (i + 1 < n) out[i + 1] = o.y;
      if (i + 2 < n) out[i + 2] = o.z;
      if (i + 3 < n) out[i + 3] = o.w;
    }
  }
}

}  // namespace

void init_device_options() {
  static std::once_flag once;
  std::call_once(once, [] {
    const char* e = std::getenv("SLAK_XCD_REMAP");
    int on = e ? std::atoi(e) : (kRemapLevel | kRemapFinal);
    (void)hipMemcpyToSymbol(HIP_SYMBOL(g_xcd_remap), &on, sizeof(int));
  });
}

// ---------------------------------------------------------------------------
// launchers

void launch_fill_i32(int32_t* p, int64_t n, int32_t value, hipStream_t st) {
  if (n <= 0) return;
  int64_t g = (n + kBlock - 1) / kBlock;
  if (g > 65536) g = 65536;
  k_fill_i32<<<(unsigned)g, kBlock, 0, st>>>(p, n, value);
}

// row slots by the block's vertex window (default); SLAK_COUNT_WINDOW=0 takes
// one device atomic per corner (read once)
static bool count_window() {
  static const bool on = [] {
    const char* e = std::getenv("SLAK_COUNT_WINDOW");
    return !e || std::atoi(e) != 0;
  }();
  return on;
}

void launch_gather(bool quad, const SegTable& seg, bool use_vals, int32_t* ids_pos, const LevelView& L,
                   hipStream_t st) {
  if (L.nf <= 0) return;
  const RowBuild rb{L.cnt, L.slots, L.head, L.next};
  const int vals = use_vals ? 1 : 0, window = count_window() ? 1 : 0;
  int32_t* const fptr = const_cast<int32_t*>(L.fptr);
  int32_t* const cface = const_cast<int32_t*>(L.cface);
  const bool one = seg.n == 1;
#define SLAK_GATHER(Q, O) \
  k_gather<Q, O><<<grid_for(L.nf), kBlock, 0, st>>>(seg, L.nf, vals, ids_pos, fptr, cface, L.flags, rb, window)
  if (quad) {
    if (one) SLAK_GATHER(true, true);
    else SLAK_GATHER(true, false);
  } else {
    if (one) SLAK_GATHER(false, true);
    else SLAK_GATHER(false, false);
  }
#undef SLAK_GATHER
}

void launch_setup(const void* src_pinned, void* dst, int64_t bytes, int32_t* zero, int64_t nzero, hipStream_t st) {
  if (bytes <= 0 && nzero <= 0) return;
  if ((bytes & 15) || (nzero & 3)) throw Error(5, "setup of partial 16-byte pieces");  // SLAK_ERR_INTERNAL
  void* src = nullptr;
  if (bytes > 0) SLAK_HIP_CHECK(hipHostGetDevicePointer(&src, const_cast<void*>(src_pinned), 0));
  const int64_t n = bytes / 16, nz = nzero / 4;
  const unsigned g = std::min<unsigned>(4096, grid_for(std::max(n, nz)));
  k_setup<<<g, kBlock, 0, st>>>(static_cast<const int4*>(src), static_cast<int4*>(dst), n,
                                reinterpret_cast<int4*>(zero), nz);
}

void launch_gather_verts(const SegTable& seg, int32_t nv_total, float4* P, hipStream_t st) {
  if (nv_total <= 0) return;
  k_gather_verts<<<grid_for(nv_total), kBlock, 0, st>>>(seg, nv_total, P);
}

void launch_copy_probe(const float4* a, float4* b, int64_t n, hipStream_t st) {
  if (n <= 0) return;
  if (n > 0x7fffffffll) throw Error(1, "copy probe too large");  // SLAK_ERR_INVALID_ARGUMENT
  k_copy_probe<<<grid_for(n), kBlock, 0, st>>>(a, b, n);
}

void launch_digest(const void* p, int64_t bytes, uint64_t* out, hipStream_t st) {
  k_fill_i32<<<1, 64, 0, st>>>(reinterpret_cast<int32_t*>(out), 2, 0);
  if (bytes <= 0) return;
  const int64_t nw = (bytes + 3) / 4;
  const unsigned g = (unsigned)std::min<int64_t>(kDigestBlocks, (nw + kBlock - 1) / kBlock);
  k_digest<<<g, kBlock, 0, st>>>(static_cast<const uint8_t*>(p), bytes, reinterpret_cast<unsigned long long*>(out));
}

void launch_faces(bool quad, const int32_t* ids, const int32_t* fptr, const float4* P, int32_t nf, const SegTable& seg,
                  const int* stop, hipStream_t st) {
  if (nf <= 0) return;
  const bool one = seg.n == 1;
  if (quad) {
    if (one) k_faces<true, true><<<grid_for(nf), kBlock, 0, st>>>(ids, fptr, P, nf, seg, stop);
    else k_faces<true, false><<<grid_for(nf), kBlock, 0, st>>>(ids, fptr, P, nf, seg, stop);
  } else {
    if (one) k_faces<false, true><<<grid_for(nf), kBlock, 0, st>>>(ids, fptr, P, nf, seg, stop);
    else k_faces<false, false><<<grid_for(nf), kBlock, 0, st>>>(ids, fptr, P, nf, seg, stop);
  }
}

// rows per block (64, 128 or 256) and LDS tile (even, 256..kRowTileMax
// entries) of the numbering
static void check_row_tiling(const LevelView& L) {
  if (L.rows_per_block != 64 && L.rows_per_block != 128 && L.rows_per_block != kBlock)
    throw Error(5, "rows per block must be 64, 128 or 256");  // SLAK_ERR_INTERNAL
  if (L.tile_entries < 256 || L.tile_entries > kRowTileMax || (L.tile_entries & 1))
    throw Error(5, "row tile out of range");  // SLAK_ERR_INTERNAL
}

void launch_symbolic(bool quad, int scheme, const LevelView& L, hipStream_t st) {
  if (L.nv <= 0) return;
  const unsigned g = grid_for(L.nv);
  if (quad) {
    if (scheme == kLAK) k_symbolic<true, kLAK><<<g, kBlock, 0, st>>>(L);
    else k_symbolic<true, kSLAK><<<g, kBlock, 0, st>>>(L);
  } else {
    if (scheme == kLAK) k_symbolic<false, kLAK><<<g, kBlock, 0, st>>>(L);
    else k_symbolic<false, kSLAK><<<g, kBlock, 0, st>>>(L);
  }
}

void launch_seg_bounds(const LevelView& L, hipStream_t st) {
  if (L.nv <= 0) return;
  k_seg_bounds<<<grid_for((int64_t)(L.seg.n + 1) * 64), kBlock, 0, st>>>(L);
}

void launch_number_faces(bool quad, int scheme, const LevelView& L, bool faces, hipStream_t st) {
  check_row_tiling(L);
  const int32_t nbn = L.nv > 0 ? (int32_t)grid_for(L.nv, L.rows_per_block) : 0;
  const size_t smem = (size_t)L.tile_entries * sizeof(int2);
  const int32_t nbf = faces && L.nf > 0 ? (int32_t)grid_for(L.nf) : 0;
  const bool one = L.seg.n == 1;
  const unsigned g = (unsigned)(nbn + nbf + (one && L.report ? 1 : 0));  // the first block reports
  if (g == 0) return;
#define SLAK_NUMBER(Q, S)                                                    \
  do {                                                                       \
    if (one) k_number_faces<Q, S, true><<<g, kBlock, smem, st>>>(L, nbn);    \
    else k_number_faces<Q, S, false><<<g, kBlock, smem, st>>>(L, nbn);       \
  } while (0)
  if (quad) {
    if (scheme == kLAK) SLAK_NUMBER(true, kLAK);
    else SLAK_NUMBER(true, kSLAK);
  } else {
    if (scheme == kLAK) SLAK_NUMBER(false, kLAK);
    else SLAK_NUMBER(false, kSLAK);
  }
#undef SLAK_NUMBER
}

void launch_report(const LevelView& L, hipStream_t st) { k_report<<<1, kBlock, 0, st>>>(L); }

bool first_level_is_small(const LevelView& L) {
  return L.seg.n == 1 && L.nv <= kSmallItems && L.nf <= kSmallItems && L.nnz <= 4 * kSmallItems;
}

void launch_first_small(bool quad, int scheme, bool use_vals, const LevelView& L, bool faces, hipStream_t st) {
  if (!first_level_is_small(L) || !L.report) throw Error(5, "not a small first level");  // SLAK_ERR_INTERNAL
  const int vals = use_vals ? 1 : 0, fp = faces ? 1 : 0;
  const int threads = (std::max({L.nv, L.nf, 1}) + 63) & ~63;  // one per vertex and face
  if (quad) {
    if (scheme == kLAK) k_first_small<true, kLAK><<<1, threads, 0, st>>>(L, vals, fp);
    else k_first_small<true, kSLAK><<<1, threads, 0, st>>>(L, vals, fp);
  } else {
    if (scheme == kLAK) k_first_small<false, kLAK><<<1, threads, 0, st>>>(L, vals, fp);
    else k_first_small<false, kSLAK><<<1, threads, 0, st>>>(L, vals, fp);
  }
}

void launch_spgemm_fde(bool quad, const LevelView& L, hipStream_t st) {
  if (L.nv <= 0) return;
  if (quad)
    k_spgemm_fde<true><<<grid_for(L.nv), kBlock, 0, st>>>(L);
  else
    k_spgemm_fde<false><<<grid_for(L.nv), kBlock, 0, st>>>(L);
}

// block counts and ratios of vertex runs over nv vertices; one run when they
// are not wanted or do not cover the vertices
static void plan_runs(VertexRuns& R, bool wanted, int64_t nv) {
  if (!wanted || R.n <= 0 || R.n > kMaxVSeg || R.first[0] != 0 || R.first[R.n] != nv) {
    R.n = 1;
    R.first[0] = 0;
    R.first[1] = (int32_t)nv;
  }
  int64_t total = 0;
  for (int s = 0; s < R.n; ++s) {
    const int64_t n = (int64_t)R.first[s + 1] - R.first[s];
    if (n < 0) throw Error(5, "vertex runs out of order");  // SLAK_ERR_INTERNAL
    R.nb[s] = (int32_t)((n + kBlock - 1) / kBlock);
    total += R.nb[s];
  }
  R.blocks = (int32_t)total;
  for (int s = 0; s < R.n; ++s) {
    R.ratio[s] = share_ratio(R.nb[s], total);
    total -= R.nb[s];
  }
}

template <bool QUAD, int SCHEME, bool ONE>
void launch_level_t(const RefineView& R, unsigned g, hipStream_t st) {
  const bool next = R.ntptr != nullptr, bnd = R.blk != nullptr;
  if (next) {
    if (bnd) k_level<QUAD, SCHEME, true, true, ONE><<<g, kBlock, 0, st>>>(R);
    else k_level<QUAD, SCHEME, true, false, ONE><<<g, kBlock, 0, st>>>(R);
  } else {
    if (bnd) k_level<QUAD, SCHEME, false, true, ONE><<<g, kBlock, 0, st>>>(R);
    else k_level<QUAD, SCHEME, false, false, ONE><<<g, kBlock, 0, st>>>(R);
  }
}

template <bool QUAD, int SCHEME>
void launch_level_t(const RefineView& R, unsigned g, hipStream_t st) {
  if (R.seg.n == 1) launch_level_t<QUAD, SCHEME, true>(R, g, st);
  else launch_level_t<QUAD, SCHEME, false>(R, g, st);
}

void launch_level(bool quad, int scheme, const RefineView& R0, hipStream_t st) {
  RefineView R = R0;
  static const bool runs = [] {  // SLAK_LEVEL_RUNS=0: vertex items in plain order
    const char* e = std::getenv("SLAK_LEVEL_RUNS");
    return !e || std::atoi(e) != 0;
  }();
  plan_runs(R.runs, runs, R.nv);
  const int64_t nbr = R.nnz > 0 ? grid_for(R.nnz) : 0;
  const int64_t T = nbr + R.runs.blocks;
  if (T == 0) return;
  R.vratio = share_ratio(R.runs.blocks, T);
  const unsigned g = (unsigned)T;
  if (quad) {
    if (scheme == kLAK) launch_level_t<true, kLAK>(R, g, st);
    else launch_level_t<true, kSLAK>(R, g, st);
  } else {
    if (scheme == kLAK) launch_level_t<false, kLAK>(R, g, st);
    else launch_level_t<false, kSLAK>(R, g, st);
  }
}

int64_t plan_final_blocks(FinalSeg& S, bool quad, bool deep) {
  static const bool runs = [] {  // SLAK_FINAL_RUNS=0: vertex items in plain order
    const char* e = std::getenv("SLAK_FINAL_RUNS");
    return !e || std::atoi(e) != 0;
  }();
  const FinalMesh& m = S.m;
  if (quad ? (int64_t)m.nnz != 4 * (int64_t)m.nf : deep)
    throw Error(5, "final level: the mesh it starts from must be quads");  // SLAK_ERR_INTERNAL
  if (deep && (2 * (int64_t)m.ne != m.nnz || 4ll * m.nnz > 0x7fffffff))
    throw Error(5, "deep final level: a closed mesh expected");  // SLAK_ERR_INTERNAL
  // Vertices that fit one block are one run: a block a class costs more than
  // the order of the classes gives (three levels of 40000 tetrahedra 741 -> 510
  // us, cubes 867 -> 629; four levels 1455 -> 994, 2064 -> 1556). The faces of
  // polygons (final_face) stay a run of their own: waves that do both kinds of
  // items take longer (two levels of 20000 tori of 32 triangles 421 -> 454 us).
  plan_runs(S.runs, runs && !(quad && m.nv <= kBlock), (int64_t)m.nv + (quad ? 0 : m.nf));
  const int64_t corners = m.nnz > 0 ? grid_for((deep ? 4ll : 1ll) * m.nnz) : 0;  // (a mesh without faces)
  const int64_t edges = deep ? ((int64_t)m.ne + kDeepEdgeUnit - 1) / kDeepEdgeUnit : 0;
  const int64_t total = corners + edges + S.runs.blocks;
  S.blocks = (int32_t)total;
  S.vratio = share_ratio(S.runs.blocks, total);
  S.eratio = share_ratio(edges, corners + edges);
  return total;
}

// blocks of a launch of V's meshes (a mesh without faces has vertex blocks
// alone, one without vertices none)
static unsigned final_grid(const FinalView& V) {
  if (V.segs && !V.block_seg) throw Error(5, "final level: no blocks planned");  // SLAK_ERR_INTERNAL
  const int64_t n = V.segs ? V.nblocks : V.one.blocks;
  if (n * kBlock > 0xffffffffll) throw Error(1, "level too large for one launch");
  return (unsigned)n;
}

template <bool QUAD, int SCHEME, bool BND>
static void launch_final_t(const FinalView& V, bool ids, unsigned g, hipStream_t st) {
  if (V.segs) {
    if (ids) k_final<QUAD, SCHEME, BND, true, true><<<g, kBlock, 0, st>>>(V);
    else k_final<QUAD, SCHEME, BND, true, false><<<g, kBlock, 0, st>>>(V);
  } else {
    if (ids) k_final<QUAD, SCHEME, BND, false, true><<<g, kBlock, 0, st>>>(V);
    else k_final<QUAD, SCHEME, BND, false, false><<<g, kBlock, 0, st>>>(V);
  }
}

template <bool QUAD>
static void launch_final_t(int scheme, const FinalView& V, bool ids, unsigned g, hipStream_t st) {
  const bool bnd = V.blk != nullptr;
  if (scheme == kLAK) {
    if (bnd) launch_final_t<QUAD, kLAK, true>(V, ids, g, st);
    else launch_final_t<QUAD, kLAK, false>(V, ids, g, st);
  } else {
    if (bnd) launch_final_t<QUAD, kSLAK, true>(V, ids, g, st);
    else launch_final_t<QUAD, kSLAK, false>(V, ids, g, st);
  }
}

void launch_final(int scheme, const FinalView& V, bool ids, hipStream_t st) {
  const unsigned g = final_grid(V);
  if (g == 0) return;
  if (V.fptr) launch_final_t<false>(scheme, V, ids, g, st);
  else launch_final_t<true>(scheme, V, ids, g, st);
}

void launch_final_deep(const FinalView& V, hipStream_t st) {
  if (!V.own || V.blk) throw Error(5, "deep final level: closed meshes with edge owners only");  // SLAK_ERR_INTERNAL
  const unsigned g = final_grid(V);
  if (g == 0) return;
  if (V.segs)
    k_final_deep<true><<<g, kBlock, 0, st>>>(V);
  else
    k_final_deep<false><<<g, kBlock, 0, st>>>(V);
}

void launch_lak_form(const LakSeg* segs, const int32_t* block_seg, int64_t nblocks, hipStream_t st) {
  if (nblocks <= 0) return;
  if (!segs || !block_seg) throw Error(5, "LAK form: no blocks planned");  // SLAK_ERR_INTERNAL
  if (nblocks * kBlock > 0xffffffffll) throw Error(1, "LAK form too large for one launch");
  k_lak_form<<<(unsigned)nblocks, kBlock, 0, st>>>(segs, block_seg);
}

void launch_sort_faces(bool by_vals, const int32_t* ptr, int32_t stride, int32_t nf, int64_t nnz, int32_t* ids,
                       int32_t* vals, int* flags, hipStream_t st) {
  if (nf <= 0) return;
  if (by_vals)
    k_sort_faces<true><<<grid_for(nf), kBlock, 0, st>>>(ptr, stride, nf, nnz, ids, vals, flags);
  else
    k_sort_faces<false><<<grid_for(nf), kBlock, 0, st>>>(ptr, stride, nf, nnz, ids, vals, flags);
}

void launch_fill_homogeneous(int32_t* ptr, int64_t nptr, int32_t* vals, int64_t nvals, int32_t stride, hipStream_t st) {
  const int64_t n = std::max(ptr ? nptr : 0, vals ? nvals : 0);
  if (n <= 0) return;
  k_fill_homogeneous<<<grid_for(n), kBlock, 0, st>>>(ptr, nptr, vals, nvals, stride);
}

int64_t scan_partials_len(int64_t n) { return (n + kScanTile - 1) / kScanTile + 1; }

// ---------------------------------------------------------------------------
// Scratch of the entry points that allocate nothing: one file-scope device
// array (each GPU holds its own copy from module load to process exit).
// Layout: the flags word in the first 256 bytes, then the int64 scan
// partials. Host code uses the per-device address hipGetSymbolAddress
// returns, never the array's name.

static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

NoAllocScratch noalloc_scratch() {
  static std::mutex mu;
  static std::vector<void*> per_dev;
  int dev = 0;
  SLAK_HIP_CHECK(hipGetDevice(&dev));
  std::lock_guard<std::mutex> g(mu);
  if ((int)per_dev.size() <= dev) per_dev.resize(dev + 1, nullptr);
  if (!per_dev[dev]) {
    void* p = nullptr;
    SLAK_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    per_dev[dev] = p;
  }
  char* base = static_cast<char*>(per_dev[dev]);
  NoAllocScratch s;
  s.flags = reinterpret_cast<int*>(base);
  s.partial = reinterpret_cast<int64_t*>(base + 256);
  s.partial_len = (int64_t)((kNoAllocScratchBytes - 256) / sizeof(int64_t));
  return s;
}

int64_t noalloc_scan_max_items() {
  const int64_t partials = (int64_t)((kNoAllocScratchBytes - 256) / sizeof(int64_t));
  return (partials - 1) * kScanTile;  // scan_partials_len(n) <= partials
}

void launch_scan(const int32_t* in, int32_t* out, int64_t n, int64_t* partial, int* flags, hipStream_t st) {
  if (n <= kScanSmall) {
    k_scan_small<<<1, kScanSmallThreads, 0, st>>>(in, n, out, flags);
    return;
  }
  int64_t ntiles = (n + kScanTile - 1) / kScanTile;
  k_scan_reduce<<<(unsigned)ntiles, kBlock, 0, st>>>(in, n, partial);
  if (ntiles <= kScanFoldTiles) {  // two launches: each tile adds up the sums before it
    k_scan_down<true><<<(unsigned)ntiles, kBlock, 0, st>>>(in, n, partial, out, ntiles, flags);
    return;
  }
  k_scan_partials<<<1, kBlock, 0, st>>>(partial, ntiles, out, n, flags);
  k_scan_down<false><<<(unsigned)ntiles, kBlock, 0, st>>>(in, n, partial, out, ntiles, flags);
}

}  // namespace slak
