// Paged-KV block gather/scatter for gfx950 (MI355X).
//
// Pure data movement, bound by HBM bandwidth: no MFMA, no LDS on the data
// itself. Every lane of a 256-lane workgroup (four wave64s) keeps kUnroll
// independent 16-byte loads in flight before it stores, which is what saturates
// HBM on a streaming copy. Large launches of blocks that are whole KiB go in
// slices of several blocks to a workgroup; otherwise blocks of 8 KiB (gathered:
// 16 KiB) and more get a workgroup each. The block id and
// the storage base are workgroup-uniform, so the compiler reads them with
// scalar loads into SGPRs: the id table is read once per block, broadcast
// through SGPRs instead of an LDS round trip and barrier. Smaller blocks (one
// KV head of a tensor-parallel rank, side tables such as per-head fp8 scales)
// are packed many to a workgroup, every lane with up to 8 vectors in flight.
//
// Between device buffers every piece takes the widest vectors its blocks hold
// (16 bytes, or what a smaller block allows) at any address: gfx950 serves
// unaligned accesses about as fast as aligned ones. A block that is no whole
// number of vectors ends with one stepped back to its last byte, which
// rewrites a few bytes with the same values. Launches with host memory on one
// side take one aligned width for all pieces.
//
// Loads and stores are non-temporal: a gathered block is read once and the
// staging copy is next read by the DMA engine, so neither should displace
// L2/MALL lines.
//
// Bad block ids (outside [0, pool_blocks)) are skipped and reported through
// an optional device flag; no lane ever forms an address from one.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>

#include "block_copy.h"

namespace kvx {
namespace {

constexpr int kThreads = 256;
constexpr int kUnroll = 8;  // vectors a lane has in flight
// Blocks per workgroup on the small-block path: the LDS address table holds
// 16 bytes per block (4 KiB, which leaves the occupancy of 8 workgroups per
// CU untouched).
constexpr uint32_t kSmallMaxBlocks = 256;

// A vector of V bytes at any byte address.
template <int V> struct VecT;
template <> struct VecT<16> {
  typedef uint32_t T __attribute__((ext_vector_type(4), aligned(1)));
};
template <> struct VecT<8> {
  typedef uint32_t T __attribute__((ext_vector_type(2), aligned(1)));
};
template <> struct VecT<4> { typedef uint32_t T __attribute__((aligned(1))); };
template <> struct VecT<2> { typedef uint16_t T __attribute__((aligned(1))); };
template <> struct VecT<1> { typedef uint8_t T; };

// Explicit address spaces: data goes through global_load/global_store (not
// flat), and workgroup-uniform table reads through the constant address
// space so they become scalar loads.
#define KVX_GLOBAL __attribute__((address_space(1)))
#define KVX_CONST __attribute__((address_space(4)))

template <typename T>
__device__ __forceinline__ KVX_GLOBAL T* gptr(uint64_t addr) {
  return (KVX_GLOBAL T*)addr;
}

template <typename T>
__device__ __forceinline__ T uniform_load(uint64_t table, uint32_t idx) {
  return ((const KVX_CONST T*)table)[idx];
}

struct KPiece {
  uint64_t storages;
  uint64_t staging;
  uint64_t others;
  int64_t stride_w;
  int64_t stride_i;
  int64_t pool_blocks;
  int64_t other_blocks;
  uint64_t bytes;     // bytes per block
  uint64_t magic;     // small blocks: floor(2^32 / elems) + 1
  uint32_t f0;
  uint32_t nblocks;
  uint32_t vec;       // vector bytes
  uint32_t elems;     // vectors per block: small blocks with the last, partial
                      // one; whole blocks without it
  uint32_t rest;      // bytes past a block's whole vectors
  uint32_t bpw;       // blocks per workgroup
  uint32_t wg_begin;  // first workgroup of the piece
  uint32_t whole;     // 1: every lane works on one block at a time
  uint32_t across;    // small blocks: > 0: of this many storages, from w0 on, the
  uint32_t w0;        // same id of each, then the next id (0: storage by storage)
};

// A kernel's one argument: its parameters and, with kCap > 0, the block ids
// themselves instead of a device table, so that a call needs no upload before
// its kernel.
template <typename P, int kCap>
struct Args {
  P p;
  uint32_t ids[kCap];
};
template <typename P>
struct Args<P, 0> {
  P p;
};

struct KParams {
  KPiece p[kMaxPieces];
  const int64_t* ids;
  const int64_t* ids2;
  int32_t* error;
  uint32_t n;
  int32_t npieces;
};

template <int V>
__device__ __forceinline__ typename VecT<V>::T ld(uint64_t base, uint64_t off) {
  return __builtin_nontemporal_load(
      (const KVX_GLOBAL typename VecT<V>::T*)(gptr<const uint8_t>(base) + off));
}

template <int V>
__device__ __forceinline__ void st(typename VecT<V>::T v, uint64_t base, uint64_t off) {
  __builtin_nontemporal_store(v, (KVX_GLOBAL typename VecT<V>::T*)(gptr<uint8_t>(base) + off));
}

// Copy of `elems` vectors by all lanes of the workgroup.
template <int V>
__device__ __forceinline__ void copy_whole_block(uint64_t src, uint64_t dst, uint32_t elems) {
  typedef typename VecT<V>::T T;
  uint32_t k = threadIdx.x;
  auto at = [](uint32_t i) { return static_cast<uint64_t>(i) * V; };
  for (; k + (kUnroll - 1) * kThreads < elems; k += kUnroll * kThreads) {
    T r[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) r[u] = ld<V>(src, at(k + u * kThreads));
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) st<V>(r[u], dst, at(k + u * kThreads));
  }
  // The tail (all of a 16 KiB block) still keeps 4, then 2 loads in flight.
  if (k + 3 * kThreads < elems) {
    T r[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) r[u] = ld<V>(src, at(k + u * kThreads));
#pragma unroll
    for (int u = 0; u < 4; ++u) st<V>(r[u], dst, at(k + u * kThreads));
    k += 4 * kThreads;
  }
  if (k + kThreads < elems) {
    const T r0 = ld<V>(src, at(k));
    const T r1 = ld<V>(src, at(k + kThreads));
    st<V>(r0, dst, at(k));
    st<V>(r1, dst, at(k + kThreads));
    k += 2 * kThreads;
  }
  if (k < elems) st<V>(ld<V>(src, at(k)), dst, at(k));
}

__device__ __forceinline__ KPiece select_piece(const KParams& P, uint32_t wg) {
  // Pieces are sorted by wg_begin; the choice is workgroup-uniform. Each
  // candidate is copied by a constant index so the kernel argument block is
  // read in place rather than spilled to scratch.
  KPiece p = P.p[0];
  if (P.npieces > 1 && wg >= P.p[1].wg_begin) p = P.p[1];
  if (P.npieces > 2 && wg >= P.p[2].wg_begin) p = P.p[2];
  if (P.npieces > 3 && wg >= P.p[3].wg_begin) p = P.p[3];
  return p;
}

// Address of a kernel's ids: its table, or where they lie in the kernel
// arguments (taken from the argument segment itself, so that an indexed read
// stays a load from there).
template <typename P, int kCap>
__device__ __forceinline__ uint64_t ids_address(const int64_t* table) {
  if constexpr (kCap == 0) {
    return reinterpret_cast<uint64_t>(table);
  } else {
    typedef Args<P, kCap> A;
    return reinterpret_cast<uint64_t>(__builtin_amdgcn_kernarg_segment_ptr()) +
           __builtin_offsetof(A, ids);
  }
}

// Id i, the same for the whole workgroup.
template <int kCap>
__device__ __forceinline__ int64_t uniform_id(uint64_t ids, uint32_t i) {
  if constexpr (kCap == 0) return uniform_load<int64_t>(ids, i);
  return uniform_load<uint32_t>(ids, i);
}

// Id i of a lane.
template <int kCap>
__device__ __forceinline__ int64_t lane_id(uint64_t ids, uint32_t i) {
  if constexpr (kCap == 0) return gptr<const int64_t>(ids)[i];
  return gptr<const uint32_t>(ids)[i];
}

__device__ __forceinline__ bool bad_id(int64_t id, int64_t limit) {
  return static_cast<uint64_t>(id) >= static_cast<uint64_t>(limit);
}

// Up to kSteps vectors a lane of the workgroup's small blocks, every load
// issued before the first store. Lane e moves vector (e % elems) of block
// (e / elems), its last one stepped back to the block's end; lanes past the
// end re-read the last vector and store nothing.
template <int V, int kSteps>
__device__ __forceinline__ void move_small(const uint64_t* s_src, const uint64_t* s_dst,
                                           uint32_t total, uint32_t elems, uint64_t magic,
                                           uint32_t bytes) {
  typename VecT<V>::T r[kSteps];
  uint64_t dst[kSteps];
#pragma unroll
  for (int u = 0; u < kSteps; ++u) {
    uint32_t e = threadIdx.x + u * kThreads;
    const bool in = e < total;
    e = in ? e : total - 1;
    const uint32_t b = static_cast<uint32_t>((e * magic) >> 32);
    const uint32_t sub = e - b * elems;
    const uint32_t off = sub + 1 < elems ? sub * V : bytes - V;
    r[u] = ld<V>(s_src[b], off);
    const uint64_t d = s_dst[b];
    dst[u] = in && d != 0 ? d + off : 0;
  }
#pragma unroll
  for (int u = 0; u < kSteps; ++u) {
    if (dst[u] != 0) st<V>(r[u], dst[u], 0);
  }
}

template <int V>
__device__ __forceinline__ void move_small_blocks(const uint64_t* s_src, const uint64_t* s_dst,
                                                  uint32_t total, uint32_t elems,
                                                  uint64_t magic, uint32_t bytes) {
  if (total > 4 * kThreads) {
    move_small<V, 8>(s_src, s_dst, total, elems, magic, bytes);
  } else if (total > kThreads) {
    move_small<V, 4>(s_src, s_dst, total, elems, magic, bytes);
  } else {
    move_small<V, 1>(s_src, s_dst, total, elems, magic, bytes);
  }
}

// Many small blocks per workgroup. The workgroup first resolves its blocks --
// id, table entries, bounds check -- with one pass of independent, coalesced
// loads, one block per lane, and stages each block's source and destination
// address in LDS, so that no lane waits on a chain of dependent table loads
// before its data loads. A bad id gets no destination and a source that can
// be read. g: the workgroup's number in the piece. Bound by HBM: 768 random
// 4 KiB blocks of 160 storages gathered in 177 us (5.7 TB/s; 242 with one
// vector in flight a lane), 2 KiB blocks with a 4-byte scale per (layer, block)
// scattered in 95 us (114 at the scales' 4-byte vectors for the whole launch).
template <bool kGather, int kCap>
__device__ __forceinline__ void copy_small_blocks(const KPiece& p, uint64_t ids,
                                                  const int64_t* ids2, int32_t* error,
                                                  uint32_t n, uint32_t g) {
  const uint32_t b0 = g * p.bpw;
  const uint32_t bytes = static_cast<uint32_t>(p.bytes);
  __shared__ uint64_t s_src[kSmallMaxBlocks];
  __shared__ uint64_t s_dst[kSmallMaxBlocks];
  const uint32_t left = p.nblocks - b0;
  const uint32_t nb = left < p.bpw ? left : p.bpw;
  for (uint32_t b = threadIdx.x; b < nb; b += kThreads) {
    const uint32_t f = (p.across != 0 ? 0 : p.f0) + b0 + b;
    const uint32_t d = p.across != 0 ? p.across : n;
    const uint32_t q = f / d;
    const uint32_t r = f - q * d;
    const uint32_t w = p.across != 0 ? p.w0 + r : q;
    const uint32_t i = p.across != 0 ? q : r;
    const int64_t id = lane_id<kCap>(ids, i);
    const uint64_t base = gptr<const uint64_t>(p.storages)[w];
    bool bad = bad_id(id, p.pool_blocks);
    uint64_t other;
    if (p.others != 0) {
      const int64_t id2 = gptr<const int64_t>(reinterpret_cast<uint64_t>(ids2))[i];
      const uint64_t obase = gptr<const uint64_t>(p.others)[w];
      const bool bad2 = bad_id(id2, p.other_blocks);
      bad = bad || bad2;
      other = obase + static_cast<uint64_t>(bad2 ? 0 : id2) * p.bytes;
    } else {
      other = p.staging + w * static_cast<uint64_t>(p.stride_w) +
              i * static_cast<uint64_t>(p.stride_i);
    }
    const uint64_t pool = base + static_cast<uint64_t>(id) * p.bytes;
    if (bad && error != nullptr) atomicOr(error, 1);
    s_src[b] = bad || !kGather ? other : pool;
    s_dst[b] = bad ? 0 : (kGather ? other : pool);
  }
  __syncthreads();
  const uint32_t total = nb * p.elems;
  switch (p.vec) {
    case 16: move_small_blocks<16>(s_src, s_dst, total, p.elems, p.magic, bytes); break;
    case 8: move_small_blocks<8>(s_src, s_dst, total, p.elems, p.magic, bytes); break;
    case 4: move_small_blocks<4>(s_src, s_dst, total, p.elems, p.magic, bytes); break;
    case 2: move_small_blocks<2>(s_src, s_dst, total, p.elems, p.magic, bytes); break;
    default: move_small_blocks<1>(s_src, s_dst, total, p.elems, p.magic, bytes); break;
  }
}

template <int V, bool kGather, int kCap>
__global__ __launch_bounds__(kThreads) void block_copy_kernel(Args<KParams, kCap> args) {
  const KParams& P = args.p;
  const uint32_t wg = blockIdx.x;
  const uint64_t ids = ids_address<KParams, kCap>(P.ids);
  const KPiece p = select_piece(P, wg);
  const uint32_t n = P.n;

  if (p.whole) {
    const uint32_t b0 = (wg - p.wg_begin) * p.bpw;
    // All lanes move one block at a time; the workgroup walks a run of
    // consecutive flat blocks (one block unless the grid is capped).
    const uint32_t left = p.nblocks - b0;
    const uint32_t nb = left < p.bpw ? left : p.bpw;
    for (uint32_t b = 0; b < nb; ++b) {
      const uint32_t f = p.f0 + b0 + b;
      const uint32_t w = f / n;
      const uint32_t i = f - w * n;
      const int64_t id = uniform_id<kCap>(ids, i);
      uint64_t other;
      bool bad = bad_id(id, p.pool_blocks);
      if (p.others != 0) {
        const int64_t id2 = uniform_load<int64_t>(reinterpret_cast<uint64_t>(P.ids2), i);
        bad = bad || bad_id(id2, p.other_blocks);
        other = uniform_load<uint64_t>(p.others, w) + static_cast<uint64_t>(id2) * p.bytes;
      } else {
        other = p.staging + w * static_cast<uint64_t>(p.stride_w) +
                i * static_cast<uint64_t>(p.stride_i);
      }
      if (bad) {
        if (threadIdx.x == 0 && P.error != nullptr) atomicOr(P.error, 1);
        continue;
      }
      const uint64_t base = uniform_load<uint64_t>(p.storages, w);
      const uint64_t pool = base + static_cast<uint64_t>(id) * p.bytes;
      const uint64_t src = kGather ? pool : other;
      const uint64_t dst = kGather ? other : pool;
      copy_whole_block<V>(src, dst, p.elems);
      if (p.rest != 0 && threadIdx.x == 0) {
        st<V>(ld<V>(src, p.bytes - V), dst, p.bytes - V);
      }
    }
    return;
  }

  copy_small_blocks<kGather, kCap>(p, ids, P.ids2, P.error, n, wg - p.wg_begin);
}

// The common launch (one piece of large blocks, no second paged side, one
// block per workgroup) without the piece selection: the workgroup reads the
// block id and the storage base with two independent scalar loads and starts
// its vector loads after one wait. Over whole storages the workgroup order
// is chosen by measurement (random ids, 64 storages of 512 MiB):
//   kAllStorages (scatter): consecutive workgroups take the same block index
//     of consecutive storages, so the writes in flight spread over every
//     storage instead of crowding one (+1 to +3 points of HBM bandwidth);
//   kStoragePairs (gather): the same block index of storages 2q and 2q + 1,
//     then the next index (+1.5 points against storage-major order; wider
//     groups measured slower).
struct FastParams {
  uint64_t storages;
  uint64_t staging;
  const int64_t* ids;
  int32_t* error;
  int64_t stride_w;
  int64_t stride_i;
  int64_t pool_blocks;
  uint64_t bytes;      // bytes per block
  uint32_t f0;
  uint32_t n;
  uint32_t elems;      // whole vectors per block
  uint32_t rest;       // bytes past them
  uint32_t wstorages;  // whole-storage orders: storages in the launch
  uint32_t w0;         // whole-storage orders: first storage (f0 = w0 * n)
  uint32_t pieces;     // workgroups per block (1, or blocks above kUnroll * kThreads vectors)
  uint32_t piece_elems;  // vectors per workgroup when pieces > 1
};

enum FastOrder : int { kStorageMajor = 0, kStoragePairs = 1, kAllStorages = 2 };

// Workgroup g of a fast launch: one whole block, or with pieces > 1 one
// piece of piece_elems vectors of a block, the pieces of a block on
// consecutive workgroups (so a large block's writes are in flight together).
template <bool kGather, int kOrder, int kCap>
__device__ __forceinline__ void fast_block(const FastParams& P, uint64_t ids, uint32_t g) {
  constexpr int V = 16;
  uint32_t piece = 0;
  if (P.pieces > 1) {
    const uint32_t b = g / P.pieces;
    piece = g - b * P.pieces;
    g = b;
  }
  uint32_t w, i;
  if (kOrder == kAllStorages) {
    i = g / P.wstorages;
    w = P.w0 + (g - i * P.wstorages);
  } else if (kOrder == kStoragePairs) {
    const uint32_t q = g / (2 * P.n);
    const uint32_t r = g - q * 2 * P.n;
    i = r >> 1;
    w = P.w0 + 2 * q + (r & 1);
  } else {
    const uint32_t f = P.f0 + g;
    w = f / P.n;
    i = f - w * P.n;
  }
  // Both table loads go out together (the base first: issued in the other
  // order, the compiler waits for the id before loading the base) and nothing
  // branches on the id before the copy: a workgroup waits for one scalar
  // round trip before its first vector load. A bad id turns the copy into no
  // work. (Measured against the branching form in one process on the same
  // allocations: equal, within 0.3 %.)
  const uint64_t base = uniform_load<uint64_t>(P.storages, w);
  const int64_t id = uniform_id<kCap>(ids, i);
  const bool bad = bad_id(id, P.pool_blocks);
  const uint32_t first = piece * P.piece_elems;  // 0 unless the block is split
  const uint32_t left = P.elems - first;
  const uint32_t span = P.pieces > 1 && left > P.piece_elems ? P.piece_elems : left;
  const uint32_t elems = bad ? 0u : span;
  const uint64_t pool = base + static_cast<uint64_t>(bad ? 0 : id) * P.bytes;
  const uint64_t stg = P.staging + w * static_cast<uint64_t>(P.stride_w) +
                       i * static_cast<uint64_t>(P.stride_i);
  const uint64_t src = kGather ? pool : stg;
  const uint64_t dst = kGather ? stg : pool;
  const uint64_t off = static_cast<uint64_t>(first) * V;
  copy_whole_block<V>(src + off, dst + off, elems);
  if (P.rest != 0 && !bad && piece + 1 == P.pieces && threadIdx.x == 0) {
    st<V>(ld<V>(src, P.bytes - V), dst, P.bytes - V);
  }
  if (bad && threadIdx.x == 0 && P.error != nullptr) atomicOr(P.error, 1);
}

template <bool kGather, int kOrder, int kCap>
__global__ __launch_bounds__(kThreads) void block_copy_fast_kernel(Args<FastParams, kCap> args) {
  fast_block<kGather, kOrder, kCap>(args.p, ids_address<FastParams, kCap>(args.p.ids), blockIdx.x);
}

// Blocks of a whole number of KiB over whole storages, in pieces: a workgroup
// moves one piece of kPiece KiB of each of 32 / kPiece blocks with consecutive
// ids of one storage, a wave 8 KiB of them. A workgroup's bytes are thus short
// pieces of several blocks, which the random side's DRAM serves better than one
// block at a time. Bound by HBM.
//   kPiece = 1 (gathers, most scatters): consecutive workgroups take the other
//     slices of the same 32 blocks, storage after storage. 512 random 32 KiB
//     blocks of 64 storages gathered in 336 us a launch (a whole block to a
//     workgroup: 356, sliced in four), 768 x 160 of 4 KiB in 163 (packed: 177),
//     0.54 GB of 8 KiB blocks in 172 (a workgroup a block: 197).
//   kPiece = 2, 4 and 8 (scatters of 4 to 32 KiB to ids spread over a pool):
//     consecutive workgroups take the same piece of the same ids in the next
//     storage, then the next piece. Writes want every storage in flight on some
//     allocations (512 random 32 KiB blocks of 64 storages, us: a block to a
//     workgroup, so ordered, 328; this 327; 1 KiB slices storage by storage 396) and
//     pieces on the others (391, 369, 415).
// The last ids of a storage (fewer than a group) are cut into 1 KiB slices with
// the id running fastest, 32 to a workgroup, so that every workgroup is full.
// The ids and the base are scalar loads, all in flight at once; nothing goes
// through LDS. A side piece (a scale table) takes the first workgroups.
constexpr uint32_t kSliceBytes = 1024;                      // 64 lanes x 16 bytes
constexpr uint32_t kSlices = kUnroll * (kThreads / 64);     // slices per workgroup
struct SlicedParams {
  uint64_t storages;
  uint64_t staging;
  const int64_t* ids;
  int32_t* error;
  int64_t stride_w;
  int64_t stride_i;
  int64_t pool_blocks;
  uint64_t bytes;      // bytes per block
  uint32_t n;
  uint32_t w0;           // first storage
  uint32_t slices;       // slices per block
  uint32_t side_wgs;     // workgroups of the side piece and, after them, of
  uint32_t last_wgs;     // every storage's last ids, in the first
  uint32_t extra_planes; // extra_planes values of blockIdx.z
  uint32_t last_per;     // workgroups of one storage's last ids
  KPiece side;
};

// Grid: kPiece = 1: (slices, id groups, extra planes + storages); kPiece > 1:
// (storages, pieces, extra planes + id groups).
template <bool kGather, int kPiece, int kCap>
__global__ __launch_bounds__(kThreads, 4) void block_copy_sliced_kernel(
    Args<SlicedParams, kCap> args) {
  constexpr int V = 16;
  constexpr uint32_t kIds = kSlices / kPiece;  // ids of a group
  constexpr uint32_t kPer = kUnroll / kPiece;  // ids of a wave's piece of it
  const SlicedParams& P = args.p;
  const uint64_t ids = ids_address<SlicedParams, kCap>(P.ids);
  const uint32_t plane = blockIdx.z - P.extra_planes;
  uint32_t wl = kPiece > 1 ? blockIdx.x : plane;                   // the storage
  const uint32_t group = kPiece > 1 ? plane : blockIdx.y;
  const uint32_t piece = kPiece > 1 ? blockIdx.y : blockIdx.x;
  uint32_t last = 0;                                               // workgroup of its last ids
  const bool whole = blockIdx.z >= P.extra_planes;
  if (!whole) {
    uint32_t g = (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
    if (g < P.side_wgs) {
      copy_small_blocks<kGather, kCap>(P.side, ids, nullptr, P.error, P.n, g);
      return;
    }
    g -= P.side_wgs;
    if (g >= P.last_wgs) return;
    wl = g / P.last_per;
    last = g - wl * P.last_per;
  }
  const uint32_t w = P.w0 + wl;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const uint32_t lane = (threadIdx.x % 64) * V;
  // The group's first id.
  const uint32_t first = whole ? group * kIds : P.n / kIds * kIds;
  const uint64_t stg_w = P.staging + w * static_cast<uint64_t>(P.stride_w);
  typename VecT<V>::T v[kUnroll];
  uint64_t pool_at[kUnroll], stg_at[kUnroll];
  bool ok[kUnroll];
  bool all_ok = true, any_bad = false;
  if (whole) {
    const uint32_t i0 = first + wave * kPer;
    const uint32_t off = piece * (kPiece * kSliceBytes);
    const uint64_t base = uniform_load<uint64_t>(P.storages, w) + off;
    const uint64_t stg = stg_w + i0 * static_cast<uint64_t>(P.stride_i) + off;
#pragma unroll
    for (uint32_t u = 0; u < kUnroll; ++u) {
      const uint32_t i = u / kPiece, sub = u % kPiece * kSliceBytes;
      const int64_t id = uniform_id<kCap>(ids, i0 + i);
      ok[u] = !bad_id(id, P.pool_blocks);
      all_ok = all_ok && ok[u];
      pool_at[u] = base + static_cast<uint64_t>(ok[u] ? id : 0) * P.bytes + sub;
      stg_at[u] = stg + i * static_cast<uint64_t>(P.stride_i) + sub;
    }
    any_bad = !all_ok;
  } else {
    // Unit k of the last `many` ids is slice k / many of id k % many.
    const uint32_t many = P.n - first;
    const uint32_t units = many * P.slices;
    const uint32_t k = last * kSlices + wave * kUnroll;
    if (k >= units) return;
    const uint64_t base = uniform_load<uint64_t>(P.storages, w);
    // Places first, then every id load, so that none waits for another; past
    // the end the last unit repeats.
    uint32_t id_at[kUnroll], off[kUnroll];
    uint32_t slice = k / many;
    uint32_t i = k - slice * many;
#pragma unroll
    for (uint32_t u = 0; u < kUnroll; ++u) {
      id_at[u] = first + i;
      off[u] = slice * kSliceBytes;
      const bool more = k + u + 1 < units;
      const bool wrap = i + 1 == many;
      i = more ? (wrap ? 0 : i + 1) : i;
      slice = more && wrap ? slice + 1 : slice;
    }
    int64_t id[kUnroll];
#pragma unroll
    for (uint32_t u = 0; u < kUnroll; ++u) id[u] = uniform_id<kCap>(ids, id_at[u]);
#pragma unroll
    for (uint32_t u = 0; u < kUnroll; ++u) {
      const bool in = k + u < units;
      const bool bad = bad_id(id[u], P.pool_blocks);
      ok[u] = in && !bad;
      all_ok = all_ok && ok[u];
      any_bad = any_bad || (in && bad);
      pool_at[u] = base + static_cast<uint64_t>(bad ? 0 : id[u]) * P.bytes + off[u];
      stg_at[u] = stg_w + id_at[u] * static_cast<uint64_t>(P.stride_i) + off[u];
    }
  }
  if (all_ok) {
#pragma unroll
    for (uint32_t u = 0; u < kUnroll; ++u) v[u] = ld<V>(kGather ? pool_at[u] : stg_at[u], lane);
#pragma unroll
    for (uint32_t u = 0; u < kUnroll; ++u) st<V>(v[u], kGather ? stg_at[u] : pool_at[u], lane);
    return;
  }
  // Fewer than 8 units, or a bad id.
#pragma unroll
  for (uint32_t u = 0; u < kUnroll; ++u) {
    if (ok[u]) v[u] = ld<V>(kGather ? pool_at[u] : stg_at[u], lane);
  }
#pragma unroll
  for (uint32_t u = 0; u < kUnroll; ++u) {
    if (ok[u]) st<V>(v[u], kGather ? stg_at[u] : pool_at[u], lane);
  }
  if (any_bad && threadIdx.x % 64 == 0 && P.error != nullptr) atomicOr(P.error, 1);
}

// The fast launch behind one leading small-block piece: the fp8 payload and
// its scale side table in one launch. The first side_wgs workgroups move the
// side piece (many blocks each, as in the general kernel), the rest take the
// payload blocks in the fast kernel's order.
struct FastSideParams {
  FastParams fast;
  KPiece side;
  uint32_t side_wgs;
};

template <bool kGather, int kOrder, int kCap>
__global__ __launch_bounds__(kThreads) void block_copy_fast_side_kernel(
    Args<FastSideParams, kCap> args) {
  const FastSideParams& P = args.p;
  const uint64_t ids = ids_address<FastSideParams, kCap>(P.fast.ids);
  if (blockIdx.x < P.side_wgs) {
    copy_small_blocks<kGather, kCap>(P.side, ids, nullptr, P.fast.error, P.fast.n, blockIdx.x);
    return;
  }
  fast_block<kGather, kOrder, kCap>(P.fast, ids, blockIdx.x - P.side_wgs);
}

// Two workgroups on each of the 256 CUs.
constexpr uint64_t kFillWorkgroups = 512;

// Packed blocks per workgroup: enough to give each lane up to 8 vectors, at most
// kSmallMaxBlocks.
uint32_t BlocksPerWorkgroup(uint64_t elems) {
  uint64_t bpw = (8 * kThreads) / (elems == 0 ? 1 : elems);
  if (bpw > kSmallMaxBlocks) bpw = kSmallMaxBlocks;
  return static_cast<uint32_t>(bpw < 1 ? 1 : bpw);
}

// Launches of fewer bytes have both their sides in the 256 MB last-level cache
// and no DRAM order to gain from: they keep the kernels that start faster (64 x
// 64 blocks of 32 KiB scattered in 46.6 us against 48.4 sliced, 256 x 160 of 4
// KiB, at the line, in 65.0 against 62.6).
constexpr uint64_t kSlicedMinBytes = 160 << 20;

// Whether a launch goes storage by storage: gathers, and scatters above the
// cache whose ids fill two fifths of their range (unknown: of the pool) or more.
// The neighbouring blocks of one storage are then in flight together, which most
// allocations serve better. Other scatters keep every storage in flight at once,
// which some allocations need. 512 32 KiB blocks of 64 storages, us, storage by
// storage and all at once: every id of a range, shuffled, 335 and 368 (five of
// seven allocations alike), 333 and 327 (the other two); every second 360 and
// 366, 354 and 329; every third 373 and 368, 363 and 328; random out of 16384 415
// and 370, 396 and 329. 16 KiB: 166 and 192, 166 and 168; 174 and 194, 173 and
// 167; 181 and 192, 181 and 167; 207 and 195, 200 and 168. One in two still gains
// more on the five than it loses on the two, one in three no longer. In the cache
// dense ids gain little on the five (12 KiB blocks, 80 MiB: 33.0 and 34.1) and lose on
// the two (32.7 and 29.3).
bool ByStorage(const CopyLaunch& l, CopyDir dir) {
  if (dir == CopyDir::kGather) return true;
  int64_t span = l.id_span;
  uint64_t total = 0;
  for (int k = 0; k < l.npieces && k < kMaxPieces; ++k) {
    const CopyPiece& c = l.pieces[k];
    if (c.nblocks <= 0 || c.block_bytes <= 0) return false;
    if (l.id_span <= 0) span = std::max(span, c.pool_blocks);
    uint64_t bytes = 0;
    if (__builtin_mul_overflow(static_cast<uint64_t>(c.nblocks),
                               static_cast<uint64_t>(c.block_bytes), &bytes) ||
        __builtin_add_overflow(total, bytes, &total)) {
      total = UINT64_MAX;
    }
  }
  return total >= kSlicedMinBytes && l.n > 0 && l.n <= INT32_MAX && span / 5 * 2 <= l.n;
}

// Whether a block of `elems` vectors goes whole to a workgroup (else packed):
// one of 2 and more vectors a lane (8 KiB), but copies between device buffers
// that go storage by storage pack up to 4 (16 KiB): 10 KB blocks of 64 storages
// gather in 190 us packed, 236 whole (0.54 GB a launch).
bool WholeBlock(uint64_t elems, bool paged, bool by_storage) {
  return elems >= (!paged && by_storage ? 4 : 2) * kThreads;
}

// Whether a piece's other side is a second paged buffer (host memory that the
// kernel reaches over PCIe).
bool Paged(const CopyLaunch& l) {
  bool paged = false;
  for (int k = 0; k < l.npieces; ++k) paged = paged || l.pieces[k].others != 0;
  return paged;
}

// Packed blocks of this size and more take the same id of every storage in turn
// where a scatter keeps every storage in flight: above the cache, and beside a
// scale table. us, storage by storage and so, on the two kinds of allocation: 7000
// bytes, 400 MiB, 178 and 178, 176 and 150; 4 KiB with 8-byte scales, 100 MiB, 44.5
// and 44.8, 44.9 and 40.1 (6 KiB with 12 43.8 and 44.4, 43.2 and 39.7). 4 KiB
// alone in the cache: 42.5 and 45.3, 41.6 and 40.1. Smaller ones do not mind
// (2 KiB with 4-byte scales 163 us on both, 400 MiB).
constexpr uint64_t kAcrossMinBytes = 4096;
bool BuildParams(const CopyLaunch& l, bool by_storage, int vec_bytes, KParams* P,
                 uint32_t* grid) {
  if (l.npieces < 1 || l.npieces > kMaxPieces ||
      (l.ids == nullptr && (l.inline_ids == nullptr || l.n > kMaxInlineIds || Paged(l))) ||
      l.n <= 0 || l.n > INT32_MAX || vec_bytes <= 0) {
    return false;
  }
  *P = KParams{};
  P->ids = l.ids;
  P->ids2 = l.ids2;
  P->error = l.error;
  P->n = static_cast<uint32_t>(l.n);
  P->npieces = l.npieces;
  // Vectors of a piece: the common width if a launch has a second paged side,
  // else the widest its blocks hold.
  const bool paged = Paged(l);
  auto vec_of = [&](uint64_t bytes) -> uint64_t {
    uint64_t v = static_cast<uint64_t>(vec_bytes);
    if (!paged) {
      for (v = 16; v > bytes;) v /= 2;
    }
    return v;
  };
  uint64_t total_blocks = 0, total_bytes = 0;
  for (int k = 0; k < l.npieces; ++k) {
    const uint64_t blocks = l.pieces[k].nblocks > 0 ? l.pieces[k].nblocks : 0;
    total_blocks += blocks;
    uint64_t bytes = 0;
    if (l.pieces[k].block_bytes <= 0 ||
        __builtin_mul_overflow(blocks, static_cast<uint64_t>(l.pieces[k].block_bytes), &bytes) ||
        __builtin_add_overflow(total_bytes, bytes, &total_bytes)) {
      total_bytes = UINT64_MAX;
    }
  }
  const bool across = !paged && !by_storage && (l.npieces > 1 || total_bytes >= kSlicedMinBytes);
  // Pieces of smaller blocks (side tables) take the first workgroups, so their
  // few workgroups run alongside the large blocks instead of after them.
  int order[kMaxPieces];
  for (int k = 0; k < l.npieces; ++k) {
    if (l.pieces[k].block_bytes <= 0) return false;
    int at = k;
    for (; at > 0 && l.pieces[order[at - 1]].block_bytes > l.pieces[k].block_bytes; --at) {
      order[at] = order[at - 1];
    }
    order[at] = k;
  }
  uint64_t wg = 0;
  for (int slot = 0; slot < l.npieces; ++slot) {
    const CopyPiece& c = l.pieces[order[slot]];
    if (c.storages == 0 || c.nblocks <= 0 || c.f0 < 0 || c.block_bytes <= 0 ||
        c.block_bytes % vec_bytes != 0 || c.pool_blocks <= 0) {
      return false;
    }
    if (c.others != 0 && (l.ids2 == nullptr || c.other_blocks <= 0)) return false;
    if (static_cast<uint64_t>(c.f0) + static_cast<uint64_t>(c.nblocks) >
        UINT32_MAX) {
      return false;
    }
    // The limit on a block is the common width's, so that what a launch
    // accepts does not depend on the vectors that move it.
    if (static_cast<uint64_t>(c.block_bytes) / vec_bytes > UINT32_MAX) return false;
    const uint64_t bytes = static_cast<uint64_t>(c.block_bytes);
    const uint64_t vec = vec_of(bytes);
    uint64_t elems = bytes / vec;
    const bool whole = WholeBlock(elems, paged, by_storage);
    if (!whole && bytes % vec != 0) ++elems;
    uint64_t bpw = whole ? 1 : BlocksPerWorkgroup(elems);
    // A launch that does not fill the chip has fewer vectors a lane instead (16
    // x 160 blocks of 4 KiB gathered in 6.5 against 7.3 us).
    while (!whole && !paged && bpw > 1 && bpw * elems > kThreads &&
           static_cast<uint64_t>(c.nblocks) < bpw * kFillWorkgroups) {
      bpw /= 2;
    }
    if (whole && l.max_workgroups > 0) {
      // This piece's share of the workgroup cap, at least one.
      uint64_t share = static_cast<uint64_t>(l.max_workgroups) *
                       static_cast<uint64_t>(c.nblocks) / total_blocks;
      if (share < 1) share = 1;
      const uint64_t need = (static_cast<uint64_t>(c.nblocks) + share - 1) / share;
      if (need > bpw) bpw = need;
    }
    if (bpw > UINT32_MAX) return false;
    KPiece& kp = P->p[slot];
    kp.storages = c.storages;
    kp.staging = c.staging;
    kp.others = c.others;
    kp.other_blocks = c.other_blocks;
    kp.stride_w = c.stride_w;
    kp.stride_i = c.stride_i;
    kp.pool_blocks = c.pool_blocks;
    kp.f0 = static_cast<uint32_t>(c.f0);
    kp.nblocks = static_cast<uint32_t>(c.nblocks);
    kp.bytes = bytes;
    kp.magic = (uint64_t{1} << 32) / elems + 1;
    kp.vec = static_cast<uint32_t>(vec);
    kp.elems = static_cast<uint32_t>(elems);
    kp.rest = static_cast<uint32_t>(bytes % vec);
    kp.bpw = static_cast<uint32_t>(bpw);
    kp.whole = whole ? 1u : 0u;
    const uint32_t n = P->n;
    if (!whole && across && bytes >= kAcrossMinBytes && kp.f0 % n == 0 && kp.nblocks % n == 0) {
      kp.across = kp.nblocks / n;
      kp.w0 = kp.f0 / n;
    }
    kp.wg_begin = static_cast<uint32_t>(wg);
    wg += (static_cast<uint64_t>(c.nblocks) + bpw - 1) / bpw;
    if (wg > INT32_MAX) return false;
  }
  *grid = static_cast<uint32_t>(wg);
  return true;
}

// The fast kernel's parameters when the launch qualifies (one whole-block
// piece, bpw 1, no second paged side).
bool BuildFastParams(const KParams& K, CopyDir dir, FastParams* F, int* order) {
  const KPiece& p = K.p[0];
  if (K.npieces != 1 || !p.whole || p.bpw != 1 || p.others != 0) return false;
  *F = FastParams{};
  F->storages = p.storages;
  F->staging = p.staging;
  F->ids = K.ids;
  F->error = K.error;
  F->stride_w = p.stride_w;
  F->stride_i = p.stride_i;
  F->pool_blocks = p.pool_blocks;
  F->f0 = p.f0;
  F->n = K.n;
  F->bytes = p.bytes;
  F->elems = p.elems;
  F->rest = p.rest;
  const bool whole_storages = p.f0 % K.n == 0 && p.nblocks % K.n == 0;
  const uint32_t W = p.nblocks / K.n;
  *order = kStorageMajor;
  if (whole_storages && W >= 2) {
    if (dir == CopyDir::kScatter) {
      *order = kAllStorages;
    } else if (W % 2 == 0) {
      *order = kStoragePairs;
    }
  }
  F->wstorages = W;
  F->w0 = p.f0 / K.n;
  F->pieces = 1;
  F->piece_elems = p.elems;
  return true;
}

// The fast-with-side-piece parameters when the launch is one small-block
// piece (no second paged side; BuildParams puts it first) followed by one
// whole-block piece that qualifies for the fast kernel.
bool BuildFastSideParams(const KParams& K, CopyDir dir, FastParams* F, KPiece* side,
                         uint32_t* side_wgs, int* order) {
  if (K.npieces != 2 || K.p[0].whole || K.p[0].others != 0) return false;
  KParams one = K;
  one.npieces = 1;
  one.p[0] = K.p[1];
  if (!BuildFastParams(one, dir, F, order)) return false;
  *side = K.p[0];
  *side_wgs = K.p[1].wg_begin;
  return true;
}

// KiB of the pieces a launch is cut into when it goes sliced, else 0. Over
// whole storages, at least 32 ids, and above the cache.
//   1 KiB: gathers of whole KiB from 2 to 256 KiB (512 KiB blocks measured 185
// us whole and 192 sliced, 0.54 GB, 256 KiB ones 184 and 177), scatters of dense
// ids up to 1 MiB (193 and 184), and scatters of 2 and 3 KiB, packed otherwise
// (480 MB of 3 KiB 170 and 163 us).
//   Other scatters: blocks of 4, 8, 16 and 32 KiB in halves of up to 8 KiB. us on
// the two kinds of allocation: 32 KiB whole 391 and so 370, 326 and 328; 16 KiB 202
// and 195, 168 and 168; 8 KiB 207 and 202, 166 and 168; 4 KiB storage by storage
// 163 and so 158, 162 and 140. The others stay whole or packed: 6, 12, 20 and
// 24 KiB in pieces lost on the second kind (141 and 147, 176 and 182, 175 and 181,
// 166 and 173) and gained little or nothing on the first, 64 KiB 329 and 339.
uint32_t PieceKib(const KPiece& p, uint32_t n, CopyDir dir, bool by_storage) {
  if (p.others != 0 || p.bytes % kSliceBytes != 0 || p.bytes < 2 * kSliceBytes) return 0;
  if (n < kSlices || p.f0 % n != 0 || p.nblocks % n != 0) return 0;
  if (p.bytes * p.nblocks < kSlicedMinBytes) return 0;
  const uint32_t kib = static_cast<uint32_t>(std::min<uint64_t>(p.bytes / kSliceBytes, 1u << 20));
  if (dir == CopyDir::kGather) return kib <= 256 ? 1 : 0;
  if (by_storage) return kib <= 1024 ? 1 : 0;
  if (kib < 4) return 1;
  return kib == 4 || kib == 8 ? kib / 2 : kib == 16 || kib == 32 ? 8 : 0;
}

// The sliced launch of one piece, or of one behind a side piece of smaller
// blocks; *grid receives its workgroups.
bool BuildSlicedParams(const KParams& K, CopyDir dir, bool by_storage, SlicedParams* S,
                       dim3* grid, uint32_t* piece_kib) {
  if (K.npieces > 2) return false;
  const KPiece& p = K.p[K.npieces - 1];
  const uint32_t kib = PieceKib(p, K.n, dir, by_storage);
  if (kib == 0) return false;
  if (K.npieces == 2 && (K.p[0].whole || K.p[0].others != 0)) return false;
  *S = SlicedParams{};
  S->storages = p.storages;
  S->staging = p.staging;
  S->ids = K.ids;
  S->error = K.error;
  S->stride_w = p.stride_w;
  S->stride_i = p.stride_i;
  S->pool_blocks = p.pool_blocks;
  S->bytes = p.bytes;
  S->n = K.n;
  S->w0 = p.f0 / K.n;
  S->slices = static_cast<uint32_t>(p.bytes / kSliceBytes);
  // Pieces, id groups and storages are the grid's dimensions, so that a
  // workgroup divides nothing to find its place (two divisions cost a gather 4 %:
  // 0.54 GB of 32 KiB blocks in 176.5 against 169.6 us). The side piece and the
  // last ids of the storages fill planes of their own before them.
  const uint64_t W = p.nblocks / K.n;
  const uint32_t ids = kSlices / kib;
  const uint64_t groups = K.n / ids;
  const uint64_t pieces = S->slices / kib;
  const uint64_t x = kib > 1 ? W : pieces, y = kib > 1 ? pieces : groups;
  const uint64_t z = kib > 1 ? groups : W;
  S->last_per = (K.n % ids * S->slices + kSlices - 1) / kSlices;
  const uint64_t last_wgs = W * S->last_per;
  if (K.npieces == 2) {
    S->side = K.p[0];
    S->side_wgs = K.p[1].wg_begin;
  }
  const uint64_t extra = (S->side_wgs + last_wgs + x * y - 1) / (x * y);
  const uint64_t planes = extra + z;
  S->last_wgs = static_cast<uint32_t>(last_wgs);
  S->extra_planes = static_cast<uint32_t>(extra);
  if (y > 65535 || planes > 65535 || x * y * planes > INT32_MAX) return false;
  *grid = dim3(static_cast<uint32_t>(x), static_cast<uint32_t>(y), static_cast<uint32_t>(planes));
  *piece_kib = kib;
  return true;
}

// LDS of one CU on gfx950.
constexpr uint32_t kLdsPerCu = 160u << 10;

// Launches of the packed and sliced kernels with fewer workgroups than this are
// not capped: they would run in a few unequal rounds (20 MB of 2 KiB blocks
// scattered in 9.7 us capped, 8.6 not).
constexpr uint32_t kCapGrid = 2048;

// LDS the kernels with the small-block path declare (its address tables).
constexpr uint32_t kStaticLds = 2 * kSmallMaxBlocks * sizeof(uint64_t);

// Whether a scatter that is neither sliced nor of one size of whole blocks takes
// the cap on workgroups per CU: if every piece goes packed. Capped and not, in one
// process: 2 KiB blocks with 4-byte scales 48.7 and 52.4 us (134 MB). Whole blocks
// with a scale table lose (us, 150 MiB, on two kinds of allocation: 8 KiB 69.6 and
// 64.9, 62.4 and 53.5; 12 KiB 69.2 and 64.2, 63.0 and 53.2), those of 16 KiB gain
// nothing on one (53.8 and 53.1) and 2 % on the other, and the cap takes the CUs'
// LDS from other streams.
bool CapScatter(const KParams& P) {
  for (int k = 0; k < P.npieces; ++k) {
    if (P.p[k].whole) return false;
  }
  return true;
}

// What a launch runs: its kernel, that kernel's parameters (the general kernel
// takes the KParams as they are), its grid and the LDS it reserves.
struct Choice {
  enum Kernel { kGeneral, kFast, kFastSide, kSliced } kernel = kGeneral;
  int order = kStorageMajor;  // fast kernels
  uint32_t piece_kib = 0;     // sliced kernel
  dim3 grid;
  uint32_t lds = 0;
  FastSideParams FS;
  SlicedParams S;
};

Choice Choose(const KParams& P, uint32_t grid, CopyDir dir, bool by_storage, int wg_per_cu,
              bool capped_grid) {
  const bool gather = dir == CopyDir::kGather;
  Choice c;
  c.grid = dim3(grid);
  FastParams& F = c.FS.fast;
  // Blocks above one workgroup's pass (kUnroll * kThreads vectors, 32 KiB at
  // 16-byte vectors) go to consecutive workgroups a pass each, unless the
  // launch's grid is capped (zero-copy copies keep their few workgroups).
  auto split = [&](uint32_t blocks) {
    const uint32_t pass = kUnroll * kThreads;
    if (capped_grid || F.elems <= pass) return;
    const uint64_t pieces = (static_cast<uint64_t>(F.elems) + pass - 1) / pass;
    if (static_cast<uint64_t>(blocks) * pieces + (grid - blocks) > INT32_MAX) return;
    F.pieces = static_cast<uint32_t>(pieces);
    F.piece_elems = pass;
    c.grid.x = grid - blocks + blocks * F.pieces;
  };
  // The reservation that leaves room for wg_per_cu workgroups on a CU.
  const uint32_t room = wg_per_cu > 0 ? kLdsPerCu / static_cast<uint32_t>(wg_per_cu) : 0;
  const uint32_t side_room = room > kStaticLds ? room - kStaticLds : 0;
  if (!capped_grid && BuildSlicedParams(P, dir, by_storage, &c.S, &c.grid, &c.piece_kib)) {
    c.kernel = Choice::kSliced;
    if (c.grid.x * c.grid.y * c.grid.z >= kCapGrid) c.lds = side_room;
    // All storages at once: half as many (512 x 64 random 32 KiB blocks in 369
    // us, 378 with 2 a CU; 327 and 327 on the other kind of allocation).
    if (c.piece_kib > 1 && wg_per_cu > 0) {
      c.lds = kLdsPerCu / static_cast<uint32_t>((wg_per_cu + 1) / 2) - kStaticLds;
    }
    return c;
  }
  if (BuildFastParams(P, dir, &F, &c.order)) {
    c.kernel = Choice::kFast;
    split(grid);
    if (gather) c.lds = room;
    return c;
  }
  // The kernels with the packed path: not the capped grids of zero-copy copies.
  const bool cap = !capped_grid && grid >= kCapGrid && (gather || CapScatter(P));
  if (cap) c.lds = side_room;
  if (BuildFastSideParams(P, dir, &F, &c.FS.side, &c.FS.side_wgs, &c.order)) {
    c.kernel = Choice::kFastSide;
    split(grid - c.FS.side_wgs);
  }
  return c;
}

// Few ids take kernels with smaller arguments: one block of 64 storages
// gathered in 13.0 us a call, 14.6 with room for kMaxInlineIds (copied twice
// on the way to the queue).
constexpr int kFewInlineIds = 64;

// A launch with its ids in a table (kCap = 0) or in its arguments.
template <int kCap>
struct Launcher {
  const uint32_t* inline_ids;
  uint32_t n;
  dim3 grid;
  uint32_t lds;
  hipStream_t stream;

  template <typename P>
  hipError_t Run(void (*kernel)(Args<P, kCap>), const P& p) const {
    Args<P, kCap> a{};
    a.p = p;
    if constexpr (kCap > 0) std::memcpy(a.ids, inline_ids, n * sizeof(uint32_t));
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), lds, stream, a);
    return hipGetLastError();
  }
  template <bool kGather, int kOrder>
  hipError_t Fast(const FastParams& F) const {
    return Run<FastParams>(block_copy_fast_kernel<kGather, kOrder, kCap>, F);
  }
  template <bool kGather, int kPiece>
  hipError_t Sliced(const SlicedParams& S) const {
    return Run<SlicedParams>(block_copy_sliced_kernel<kGather, kPiece, kCap>, S);
  }
  template <bool kGather, int kOrder>
  hipError_t FastSide(const FastSideParams& F) const {
    return Run<FastSideParams>(block_copy_fast_side_kernel<kGather, kOrder, kCap>, F);
  }
  template <int V>
  hipError_t General(const KParams& K, bool gather) const {
    return gather ? Run<KParams>(block_copy_kernel<V, true, kCap>, K)
                  : Run<KParams>(block_copy_kernel<V, false, kCap>, K);
  }
};

// whole_vec: vector bytes of the launch's whole-block pieces.
template <int kCap>
hipError_t Launch(const KParams& P, const uint32_t* inline_ids, uint32_t grid, CopyDir dir,
                  bool by_storage, int wg_per_cu, bool capped_grid, int whole_vec,
                  hipStream_t stream) {
  const bool gather = dir == CopyDir::kGather;
  const Choice c = Choose(P, grid, dir, by_storage, wg_per_cu, capped_grid);
  const Launcher<kCap> to{inline_ids, P.n, c.grid, c.lds, stream};
  const FastParams& F = c.FS.fast;
  if (c.kernel == Choice::kSliced) {
    if (gather) return to.template Sliced<true, 1>(c.S);
    return c.piece_kib == 8   ? to.template Sliced<false, 8>(c.S)
           : c.piece_kib == 4 ? to.template Sliced<false, 4>(c.S)
           : c.piece_kib == 2 ? to.template Sliced<false, 2>(c.S)
                              : to.template Sliced<false, 1>(c.S);
  }
  if (c.kernel == Choice::kFast) {
    if (gather) {
      return c.order == kStoragePairs ? to.template Fast<true, kStoragePairs>(F)
                                      : to.template Fast<true, kStorageMajor>(F);
    }
    return c.order == kAllStorages ? to.template Fast<false, kAllStorages>(F)
                                   : to.template Fast<false, kStorageMajor>(F);
  }
  if (c.kernel == Choice::kFastSide) {
    if (gather) {
      return c.order == kStoragePairs ? to.template FastSide<true, kStoragePairs>(c.FS)
                                      : to.template FastSide<true, kStorageMajor>(c.FS);
    }
    return c.order == kAllStorages ? to.template FastSide<false, kAllStorages>(c.FS)
                                   : to.template FastSide<false, kStorageMajor>(c.FS);
  }
  if constexpr (kCap == 0) {
    if (whole_vec == 4) return to.template General<4>(P, gather);
    if (whole_vec == 1) return to.template General<1>(P, gather);
  }
  return to.template General<16>(P, gather);
}

}  // namespace

int LaunchVectorBytes(const CopyLaunch& l, uint64_t extra_align) {
  uint64_t acc = extra_align;
  for (int k = 0; k < l.npieces && k < kMaxPieces; ++k) {
    const CopyPiece& c = l.pieces[k];
    acc |= static_cast<uint64_t>(c.block_bytes) | c.staging |
           static_cast<uint64_t>(c.stride_w) | static_cast<uint64_t>(c.stride_i);
  }
  if ((acc & 15) == 0) return 16;
  if ((acc & 3) == 0) return 4;
  return 1;
}

bool BlockCopyRouteOf(const CopyLaunch& l, CopyDir dir, int vec_bytes, BlockCopyRoute* route) {
  KParams P;
  uint32_t grid = 0;
  const bool by_storage = ByStorage(l, dir);
  if (!BuildParams(l, by_storage, vec_bytes, &P, &grid)) return false;
  const Choice c =
      Choose(P, grid, dir, by_storage, l.gather_workgroups_per_cu, l.max_workgroups > 0);
  static const char* const kNames[] = {"block_copy_kernel", "block_copy_fast_kernel",
                                       "block_copy_fast_side_kernel", "block_copy_sliced_kernel"};
  route->kernel = kNames[c.kernel];
  route->piece_kib = c.piece_kib;
  route->workgroups = static_cast<uint64_t>(c.grid.x) * c.grid.y * c.grid.z;
  route->lds_bytes = c.lds;
  return true;
}

hipError_t LaunchBlockCopy(const CopyLaunch& l, CopyDir dir, int vec_bytes,
                           hipStream_t stream) {
  KParams P;
  uint32_t grid = 0;
  const bool by_storage = ByStorage(l, dir);
  if (!BuildParams(l, by_storage, vec_bytes, &P, &grid)) return hipErrorInvalidValue;
  if (l.gather_workgroups_per_cu < 0 || l.gather_workgroups_per_cu > 32) {
    return hipErrorInvalidValue;
  }
  const int cap = l.gather_workgroups_per_cu;
  if (vec_bytes != 16 && vec_bytes != 4 && vec_bytes != 1) return hipErrorInvalidValue;
  const bool capped = l.max_workgroups > 0;
  if (l.ids == nullptr && l.n <= kFewInlineIds) {
    return Launch<kFewInlineIds>(P, l.inline_ids, grid, dir, by_storage, cap, capped, 16, stream);
  }
  if (l.ids == nullptr) {
    return Launch<kMaxInlineIds>(P, l.inline_ids, grid, dir, by_storage, cap, capped, 16, stream);
  }
  return Launch<0>(P, nullptr, grid, dir, by_storage, cap, capped, Paged(l) ? vec_bytes : 16,
                   stream);
}

}  // namespace kvx
