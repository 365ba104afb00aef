// Pack / unpack kernels for gfx950 (MI355X), compiled to a standalone code object
// (hipcc --genco) that the host library embeds and loads with hipModuleLoadData.
//
// One launch moves up to kMaxDesc "pieces" (a byte range of one tensor's payload) between
// strided tensor views and a dense staging payload. The payload is in storage order, so the
// tensor side is walked in address order too; nothing is transposed. The work is pure data
// movement and HBM-bound: every path aims at 128-bit coalesced loads and stores.
//
//   CONTIG  the piece is one contiguous run and 16-byte aligned: kUnroll x 16 B in flight
//           per lane, no index arithmetic.
//   RUNS    contiguous runs whose length, start and strides are multiples of 16 B: each
//           16-byte chunk is located with fast division over the canonical dimensions.
//   ROWS    contiguous runs off that grid (misaligned bases, odd run lengths or strides): each
//           16-byte payload chunk is one unaligned 128-bit access of its run; a chunk that
//           crosses into the next run moves element by element.
//   ELEM    an element-strided innermost dimension: elements are gathered one by one into LDS
//           and the tile is written to the payload with 128-bit stores (pack), or read from the
//           payload with 128-bit loads into LDS and scattered from there (unpack).
//   NARROW  a contiguous float32 tensor whose values are exactly bfloat16: the payload holds
//           the high 16 bits of each element (pack reads 32 B and writes 16 B a chunk; unpack
//           writes the halves back with zero low bits), so the same bits cross the host link
//           in half the bytes.
//
// Grid: one 256-lane workgroup per 16 KiB tile of payload; tiles of all pieces of the
// launch are numbered consecutively and a workgroup finds its piece from the launch's array
// of piece start tiles.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mo_kdesc.h"
#include "mo_wire.h"

// The scratch of mo_pack_to_host (size kNoAllocScratchBytes). External linkage with a C name:
// the host finds it in the loaded code object with hipModuleGetGlobal, once per device, and
// passes that address to the pack kernel like any payload buffer (a static array would have no
// symbol in the code object). Only the pack kernel writes it and the DMA reads it.
extern "C" {
__device__ __align__(256) unsigned char mo_noalloc_scratch[mo::kNoAllocScratchBytes];
}

namespace mo {

__device__ __forceinline__ uint32_t fdiv(uint32_t n, uint32_t m, uint32_t s) {
  const uint64_t t = __umulhi(m, n);
  return (uint32_t)((t + n) >> s);
}

// Address offset (bytes, relative to the tensor base) of unit `u` of a piece's tensor side.
// A unit is a 16-byte chunk (RUNS) or an element (ROWS, ELEM).
__device__ __forceinline__ uint64_t unit_offset(const KDesc& d, uint32_t u) {
  uint32_t q = fdiv(u, d.inner.m, d.inner.s);
  uint64_t off = (uint64_t)(u - q * d.inner.d) * d.inner_stride;
  const uint32_t nouter = d.nouter;
#pragma unroll
  for (int k = 0; k < kMaxOuter; ++k) {
    if (k < (int)nouter) {
      const uint32_t q2 = fdiv(q, d.outer[k].m, d.outer[k].s);
      off += (uint64_t)(q - q2 * d.outer[k].d) * d.ostride[k];
      q = q2;
    }
  }
  return off;
}

// Every device pointer reaches the kernels as an integer inside a descriptor, so the compiler
// cannot infer its address space and would emit flat (generic) memory instructions. The
// accessors below name the space: global (HBM or pinned host memory).
#define MO_GLOBAL __attribute__((address_space(1)))
#define MO_LDS __attribute__((address_space(3)))

// 16-byte values move as a native vector: uint4 is a class whose copy constructor takes a
// generic reference, which would turn the access back into a flat one.
typedef unsigned int mo_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int mo_u32x2 __attribute__((ext_vector_type(2)));

template <typename T>
__device__ __forceinline__ T ld(const char* p) {
  return *(const MO_GLOBAL T*)p;
}
template <typename T>
__device__ __forceinline__ void st(char* p, T v) {
  *(MO_GLOBAL T*)p = v;
}
template <>
__device__ __forceinline__ uint4 ld<uint4>(const char* p) {
  const mo_u32x4 x = *(const MO_GLOBAL mo_u32x4*)p;
  return make_uint4(x.x, x.y, x.z, x.w);
}
template <>
__device__ __forceinline__ void st<uint4>(char* p, uint4 v) {
  *(MO_GLOBAL mo_u32x4*)p = mo_u32x4{v.x, v.y, v.z, v.w};
}

__device__ __forceinline__ void copy_elem(char* dst, const char* src, uint32_t eb) {
  switch (eb) {
    case 1: st(dst, ld<uint8_t>(src)); break;
    case 2: st(dst, ld<uint16_t>(src)); break;
    case 4: st(dst, ld<uint32_t>(src)); break;
    case 8: st(dst, ld<uint64_t>(src)); break;
    default: st(dst, ld<uint4>(src)); break;
  }
}

__device__ __forceinline__ uint4 ld16(const char* p) { return ld<uint4>(p); }
__device__ __forceinline__ void st16(char* p, uint4 v) { st(p, v); }

// Streaming store for the staging payload: it is written once and next read by a DMA engine,
// so the write is marked non-temporal (no reuse expected in the GPU caches).
__device__ __forceinline__ void st16_stream(char* p, uint4 v) {
  const mo_u32x4 x = {v.x, v.y, v.z, v.w};
  __builtin_nontemporal_store(x, (MO_GLOBAL mo_u32x4*)p);
}

// Full tiles whose cache policy the launch picks at run time (KDesc.cache) use buffer
// instructions, whose cache-policy operand is an immediate of the instruction: the policy arms of
// a switch then stay separate code paths. With ordinary loads and stores the arms differ only in a
// non-temporal hint, which the optimizer treats as metadata: it merges the arms into one and drops
// the hint. The resource spans one tile: raw access, stride 0, num_records = the tile's bytes,
// word 3 = DATA_FORMAT 32 (untyped buffer access on gfx9-family targets).
constexpr int kAuxNt = 2;  // cache-policy operand: bit 1 = nt on gfx940-family targets
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const char* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)bytes, 0x00020000);
}

// A full CONTIG tile: kUnroll 16-byte loads a lane in flight, then the stores.
template <bool kNtLoad, bool kNtStore>
__device__ __forceinline__ void contig_tile(char* dst, const char* src, uint32_t tid) {
  const __amdgpu_buffer_rsrc_t s = tile_rsrc(src, kTileBytes), t = tile_rsrc(dst, kTileBytes);
  mo_u32x4 v[kUnroll];
#pragma unroll
  for (int k = 0; k < kUnroll; ++k)
    v[k] = __builtin_amdgcn_raw_buffer_load_b128(s, (uint32_t)(k * kThreads + tid) * 16, 0, kNtLoad ? kAuxNt : 0);
#pragma unroll
  for (int k = 0; k < kUnroll; ++k)
    __builtin_amdgcn_raw_buffer_store_b128(v[k], t, (uint32_t)(k * kThreads + tid) * 16, 0, kNtStore ? kAuxNt : 0);
}

// A full NARROW unpack tile: 8 contiguous payload bytes (4 bfloat16 values) <-> 16 contiguous
// float32 tensor bytes a lane and round, so each instruction covers one span.
template <bool kNtLoad, bool kNtStore>
__device__ __forceinline__ void widen_tile(char* tensor32, const char* payload, uint32_t tid) {
  constexpr int kRounds = 2 * kUnroll;
  const __amdgpu_buffer_rsrc_t p = tile_rsrc(payload, kTileBytes), t = tile_rsrc(tensor32, 2 * kTileBytes);
  mo_u32x2 v[kRounds];
#pragma unroll
  for (int k = 0; k < kRounds; ++k)
    v[k] = __builtin_amdgcn_raw_buffer_load_b64(p, (uint32_t)(k * kThreads + tid) * 8, 0, kNtLoad ? kAuxNt : 0);
#pragma unroll
  for (int k = 0; k < kRounds; ++k)
    __builtin_amdgcn_raw_buffer_store_b128(mo_u32x4{v[k].x << 16, v[k].x & 0xffff0000u, v[k].y << 16, v[k].y & 0xffff0000u},
                                           t, (uint32_t)(k * kThreads + tid) * 16, 0, kNtStore ? kAuxNt : 0);
}

// Payload-side store: streaming when packing (the payload is the staging buffer).
template <bool kPack>
__device__ __forceinline__ void st16_out(char* p, uint4 v) {
  if (kPack) st16_stream(p, v);
  else st16(p, v);
}

// NARROW: 8 float32 elements (two 16-byte words a, b) <-> their 8 high halves (one 16-byte word;
// element j's bits at payload bytes 2j, 2j+1, little-endian).
__device__ __forceinline__ uint4 high_halves(uint4 a, uint4 b) {
  return make_uint4((a.x >> 16) | (a.y & 0xffff0000u), (a.z >> 16) | (a.w & 0xffff0000u),
                    (b.x >> 16) | (b.y & 0xffff0000u), (b.z >> 16) | (b.w & 0xffff0000u));
}
__device__ __forceinline__ void widen(uint4 v, uint4& a, uint4& b) {
  a = make_uint4(v.x << 16, v.x & 0xffff0000u, v.y << 16, v.y & 0xffff0000u);
  b = make_uint4(v.z << 16, v.z & 0xffff0000u, v.w << 16, v.w & 0xffff0000u);
}
template <bool kPack>
__device__ __forceinline__ void narrow_chunk(char* payload16, char* tensor32) {
  if (kPack) {
    const uint4 a = ld16(tensor32), b = ld16(tensor32 + 16);
    st16_stream(payload16, high_halves(a, b));
  } else {
    uint4 a, b;
    widen(ld16(payload16), a, b);
    st16(tensor32, a);
    st16(tensor32 + 16, b);
  }
}

// `body` with a value of the element type of `eb` bytes.
template <typename F>
__device__ __forceinline__ void with_element(uint32_t eb, F&& body) {
  switch (eb) {
    case 1: body(uint8_t()); break;
    case 2: body(uint16_t()); break;
    case 4: body(uint32_t()); break;
    case 8: body(uint64_t()); break;
    default: body(mo_u32x4{0, 0, 0, 0}); break;
  }
}

// 16 bytes at any byte address (global accesses of any alignment are one instruction under the
// unaligned access mode every HSA kernel runs in).
typedef unsigned int mo_u32x4_any __attribute__((ext_vector_type(4), aligned(1)));

// Address offsets of the units u[0 .. N - 1], and the units of their innermost runs from them on:
// unit_offset with the dimensions outermost, so that N chains run side by side in little code.
template <int N>
__device__ __forceinline__ void unit_offsets(const KDesc& d, const uint32_t (&u)[N], uint64_t (&off)[N], uint32_t (&left)[N]) {
  uint32_t q[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    q[i] = fdiv(u[i], d.inner.m, d.inner.s);
    const uint32_t at = u[i] - q[i] * d.inner.d;
    off[i] = (uint64_t)at * d.inner_stride;
    left[i] = d.inner.d - at;
  }
#pragma unroll 1
  for (uint32_t k = 0; k < d.nouter; ++k) {
    const KFastDiv f = d.outer[k];
    const uint64_t stride = d.ostride[k];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const uint32_t q2 = fdiv(q[i], f.m, f.s);
      off[i] += (uint64_t)(q[i] - q2 * f.d) * stride;
      q[i] = q2;
    }
  }
}

// The 16 payload bytes of chunk `c`, whose elements cross from one run into the next (runs hold at
// least 16 bytes): `n0` elements at `t0`, the others at `t1`, all in flight together.
template <bool kPack, typename T>
__device__ __forceinline__ void split_chunk(char* payload16, char* t0, char* t1, uint32_t n0) {
  constexpr uint32_t kPer = 16 / sizeof(T);
  union {
    mo_u32x4 v;
    T e[kPer];
  } x;
  if (!kPack) x.v = *(const MO_GLOBAL mo_u32x4*)payload16;
  char* const second = t1 - (uint64_t)n0 * sizeof(T);
#pragma unroll
  for (uint32_t j = 0; j < kPer; ++j) {
    char* const at = (j < n0 ? t0 : second) + j * sizeof(T);
    if (kPack) x.e[j] = *(const MO_GLOBAL T*)at;
    else *(MO_GLOBAL T*)at = x.e[j];
  }
  if (kPack) __builtin_nontemporal_store(x.v, (MO_GLOBAL mo_u32x4*)payload16);
}

// ROWS: one tile of contiguous runs off the 16-byte grid. Every lane locates its kUnroll chunks of
// 16 payload bytes and has them in flight together; chunks that cross into the next run follow.
// Memory-bound where runs are long; taken element by element, such a tile was bound by its
// dependent round trips (32 a lane for 2-byte elements, 64 for bytes). Pack and unpack of 2 693 rows
// of 6 144 bytes from an odd element on: 14.4 and 15.3 us, now 5.4 and 6.4 (6.2 and 5.2 TB/s); rows
// of 67 bytes: 22.0 and 19.9, now 6.7 and 7.1.
template <bool kPack>
__device__ __forceinline__ void rows_tile(const KDesc& d, uint32_t e0, uint32_t tile_bytes, char* payload, char* tensor,
                                          uint32_t eb, uint32_t tid) {
  const uint32_t nchunk = tile_bytes / 16, per = 16 / eb;
  uint32_t e[kUnroll], left[kUnroll];
  uint64_t off[kUnroll];
  mo_u32x4 v[kUnroll];
  bool split = false;
#pragma unroll
  for (int k = 0; k < kUnroll; ++k) e[k] = e0 + (k * kThreads + tid) * per;
  unit_offsets(d, e, off, left);
#pragma unroll
  for (int k = 0; k < kUnroll; ++k) {
    const uint32_t c = k * kThreads + tid;
    if (c >= nchunk) continue;
    if (left[k] < per) split = true;
    else v[k] = kPack ? *(const MO_GLOBAL mo_u32x4_any*)(tensor + off[k]) : *(const MO_GLOBAL mo_u32x4*)(payload + 16 * (size_t)c);
  }
#pragma unroll
  for (int k = 0; k < kUnroll; ++k) {
    const uint32_t c = k * kThreads + tid;
    if (c >= nchunk || left[k] < per) continue;
    if (kPack) __builtin_nontemporal_store(v[k], (MO_GLOBAL mo_u32x4*)(payload + 16 * (size_t)c));
    else *(MO_GLOBAL mo_u32x4_any*)(tensor + off[k]) = v[k];
  }
  if (__builtin_amdgcn_ballot_w64(split) != 0) {
#pragma unroll 1
    for (uint32_t c = tid; c < nchunk; c += kThreads) {
      const uint32_t first = e0 + c * per;
      const uint32_t n0 = d.inner.d - (first - fdiv(first, d.inner.m, d.inner.s) * d.inner.d);
      if (n0 >= per) continue;
      const uint32_t both[2] = {first, first + n0};
      uint32_t unused[2];
      uint64_t at[2];
      unit_offsets(d, both, at, unused);
      with_element(eb, [&](auto zero) {
        split_chunk<kPack, decltype(zero)>(payload + 16 * (size_t)c, tensor + at[0], tensor + at[1], n0);
      });
    }
  }
  for (uint32_t b = nchunk * 16 + tid * eb; b < tile_bytes; b += kThreads * eb) {
    char* const t = tensor + unit_offset(d, e0 + b / eb);
    if (kPack) copy_elem(payload + b, t, eb);
    else copy_elem(t, payload + b, eb);
  }
}

// ELEM: one tile of a view whose innermost stride is not its element size (or whose runs are under
// 16 bytes), staged in LDS. The payload side moves in 16-byte chunks; on the tensor side
// consecutive lanes take consecutive elements, kInFlight of them a lane at a time (one at a time, a
// tile was as many dependent round trips; more than four take registers from the other tiles of a
// launch). Every other one of 2 693 x 256 halves: 11.3 and 10.4 us, now 6.9 and 5.1.
template <bool kPack, typename T>
__device__ __forceinline__ void elem_tile(const KDesc& d, uint32_t e0, uint32_t tile_bytes, char* payload, char* tensor,
                                          uint32_t tid, MO_LDS char* lds) {
  constexpr int kInFlight = 4;
  const uint32_t nelem = tile_bytes / sizeof(T), nvec = tile_bytes / 16;
  MO_LDS T* const el = (MO_LDS T*)lds;
  MO_LDS mo_u32x4* const vec = (MO_LDS mo_u32x4*)lds;
  if (!kPack) {
    mo_u32x4 p[kUnroll];
#pragma unroll
    for (int k = 0; k < kUnroll; ++k) {
      const uint32_t c = k * kThreads + tid;
      if (c < nvec) p[k] = *(const MO_GLOBAL mo_u32x4*)(payload + 16 * (size_t)c);
    }
#pragma unroll
    for (int k = 0; k < kUnroll; ++k)
      if (k * kThreads + tid < nvec) vec[k * kThreads + tid] = p[k];
    for (uint32_t j = nvec * 16 / sizeof(T) + tid; j < nelem; j += kThreads) el[j] = *(const MO_GLOBAL T*)(payload + j * sizeof(T));
    __syncthreads();
  }
#pragma unroll 1
  for (uint32_t j0 = tid; j0 < nelem; j0 += kThreads * kInFlight) {
    T v[kInFlight];
    uint32_t e[kInFlight], unused[kInFlight];
    uint64_t off[kInFlight];
#pragma unroll
    for (int k = 0; k < kInFlight; ++k) e[k] = e0 + j0 + k * kThreads;
    unit_offsets(d, e, off, unused);
#pragma unroll
    for (int k = 0; k < kInFlight; ++k) {
      const uint32_t j = j0 + k * kThreads;
      if (j >= nelem) continue;
      if (kPack) v[k] = *(const MO_GLOBAL T*)(tensor + off[k]);
      else *(MO_GLOBAL T*)(tensor + off[k]) = el[j];
    }
    if (!kPack) continue;
#pragma unroll
    for (int k = 0; k < kInFlight; ++k)
      if (j0 + k * kThreads < nelem) el[j0 + k * kThreads] = v[k];
  }
  if (kPack) {
    __syncthreads();
    for (uint32_t c = tid; c < nvec; c += kThreads) __builtin_nontemporal_store(vec[c], (MO_GLOBAL mo_u32x4*)(payload + 16 * (size_t)c));
    for (uint32_t j = nvec * 16 / sizeof(T) + tid; j < nelem; j += kThreads) *(MO_GLOBAL T*)(payload + j * sizeof(T)) = el[j];
  }
}

// One 16 KiB tile (`tile`, numbered within the launch) of piece `d`. kElem: the launch may hold
// ROWS and ELEM pieces, for which every workgroup of the launch then reserves the LDS staging
// buffer and more registers; launches without them use the instantiation without either.
template <bool kPack, bool kElem>
__device__ __forceinline__ void copy_tile(const KDesc& d, uint32_t tile) {
  const uint32_t tid = threadIdx.x;
  const uint64_t tile_off = (uint64_t)(tile - d.tile0) * kTileBytes;  // bytes into the piece
  const uint64_t left = d.nbytes - tile_off;
  const uint32_t tile_bytes = left < kTileBytes ? (uint32_t)left : kTileBytes;
  char* const payload = (char*)d.payload + tile_off;
  char* const tensor = (char*)d.tensor;
  const uint32_t eb = d.eb;

  if (d.path == kPathContig) {
    char* const t = tensor + d.first + tile_off;
    const char* src = kPack ? t : payload;
    char* dst = kPack ? payload : t;
    if (tile_bytes == kTileBytes) {
      switch (d.cache & (kCacheNtLoad | kCacheNtStore)) {
        case 0: contig_tile<false, false>(dst, src, tid); break;
        case kCacheNtLoad: contig_tile<true, false>(dst, src, tid); break;
        case kCacheNtStore: contig_tile<false, true>(dst, src, tid); break;
        default: contig_tile<true, true>(dst, src, tid); break;
      }
    } else {
      const uint32_t nvec = tile_bytes / 16;
      for (uint32_t c = tid; c < nvec; c += kThreads) st16_out<kPack>(dst + (size_t)c * 16, ld16(src + (size_t)c * 16));
      for (uint32_t b = nvec * 16 + tid * eb; b < tile_bytes; b += kThreads * eb) copy_elem(dst + b, src + b, eb);
    }
    return;
  }

  if (d.path == kPathNarrow) {
    // payload offsets count bfloat16 bits; the float32 tensor side is twice as far in. A full
    // tile, measured both ways on the block microbench: pack keeps 16-byte streaming stores (a
    // lane reads the 32 tensor bytes of one payload chunk); unpack is widen_tile.
    char* const t = tensor + 2 * (d.first + tile_off);
    if (tile_bytes == kTileBytes) {
      if (kPack) {
        uint4 a[kUnroll], b[kUnroll];
#pragma unroll
        for (int k = 0; k < kUnroll; ++k) {
          a[k] = ld16(t + (size_t)(k * kThreads + tid) * 32);
          b[k] = ld16(t + (size_t)(k * kThreads + tid) * 32 + 16);
        }
#pragma unroll
        for (int k = 0; k < kUnroll; ++k) st16_stream(payload + (size_t)(k * kThreads + tid) * 16, high_halves(a[k], b[k]));
      } else {
        switch (d.cache & (kCacheNtLoad | kCacheNtStore)) {
          case 0: widen_tile<false, false>(t, payload, tid); break;
          case kCacheNtLoad: widen_tile<true, false>(t, payload, tid); break;
          case kCacheNtStore: widen_tile<false, true>(t, payload, tid); break;
          default: widen_tile<true, true>(t, payload, tid); break;
        }
      }
    } else {
      const uint32_t nvec = tile_bytes / 16;
      for (uint32_t c = tid; c < nvec; c += kThreads) narrow_chunk<kPack>(payload + (size_t)c * 16, t + (size_t)c * 32);
      for (uint32_t b = nvec * 16 + tid * 2; b < tile_bytes; b += kThreads * 2) {
        if (kPack)
          st(payload + b, (uint16_t)(ld<uint32_t>(t + (size_t)b * 2) >> 16));
        else
          st(t + (size_t)b * 2, (uint32_t)ld<uint16_t>(payload + b) << 16);
      }
    }
    return;
  }

  if (d.path == kPathRuns) {
    const uint32_t c0 = (uint32_t)(tile_off / 16);
    const uint32_t nchunk = tile_bytes / 16;
    const uint32_t first = (uint32_t)d.first;
    uint4 v[kUnroll];
    uint64_t toff[kUnroll];
#pragma unroll
    for (int k = 0; k < kUnroll; ++k) {
      const uint32_t c = k * kThreads + tid;
      if (c < nchunk) {
        toff[k] = unit_offset(d, first + c0 + c);
        v[k] = kPack ? ld16(tensor + toff[k]) : ld16(payload + (size_t)c * 16);
      }
    }
#pragma unroll
    for (int k = 0; k < kUnroll; ++k) {
      const uint32_t c = k * kThreads + tid;
      if (c < nchunk) {
        if (kPack) st16_stream(payload + (size_t)c * 16, v[k]);
        else st16(tensor + toff[k], v[k]);
      }
    }
    return;
  }

  if constexpr (kElem) {
    __shared__ uint4 lds[kTileBytes / 16];
    const uint32_t e0 = (uint32_t)d.first + (uint32_t)(tile_off / eb);
    if (d.path == kPathRows) {
      rows_tile<kPack>(d, e0, tile_bytes, payload, tensor, eb, tid);
    } else {
      with_element(eb, [&](auto zero) {
        elem_tile<kPack, decltype(zero)>(d, e0, tile_bytes, payload, tensor, tid, (MO_LDS char*)lds);
      });
    }
  }
}

// Several pieces: the workgroup's piece is the last one starting at or before its tile. The
// starts are one contiguous array (unused entries UINT32_MAX), compared without branches.
template <bool kPack, bool kElem>
__device__ __forceinline__ void copy_body(const LaunchArgs& args) {
  const uint32_t tile = blockIdx.x;
  uint32_t i = 0;
#pragma unroll
  for (int k = 1; k < kMaxDesc; ++k) i += args.tile0[k] <= tile ? 1u : 0u;
  copy_tile<kPack, kElem>(args.d[i], tile);
}

}  // namespace mo

extern "C" __global__ __launch_bounds__(mo::kThreads) void mo_pack_kernel(const mo::LaunchArgs args) {
  mo::copy_body<true, false>(args);
}

extern "C" __global__ __launch_bounds__(mo::kThreads) void mo_unpack_kernel(const mo::LaunchArgs args) {
  mo::copy_body<false, false>(args);
}

// The same with ROWS or ELEM pieces in the launch (16 KiB of LDS a workgroup).
extern "C" __global__ __launch_bounds__(mo::kThreads) void mo_pack_elem_kernel(const mo::LaunchArgs args) {
  mo::copy_body<true, true>(args);
}

extern "C" __global__ __launch_bounds__(mo::kThreads) void mo_unpack_elem_kernel(const mo::LaunchArgs args) {
  mo::copy_body<false, true>(args);
}

// One piece (tile0 == 0): the same work with a single descriptor as the kernel argument, which
// cuts the argument block a launch carries from sizeof(LaunchArgs) to sizeof(KDesc). Most
// launches move one saved tensor.
extern "C" __global__ __launch_bounds__(mo::kThreads) void mo_pack1_kernel(const mo::KDesc d) {
  mo::copy_tile<true, false>(d, blockIdx.x);
}

extern "C" __global__ __launch_bounds__(mo::kThreads) void mo_unpack1_kernel(const mo::KDesc d) {
  mo::copy_tile<false, false>(d, blockIdx.x);
}

extern "C" __global__ __launch_bounds__(mo::kThreads) void mo_pack1_elem_kernel(const mo::KDesc d) {
  mo::copy_tile<true, true>(d, blockIdx.x);
}

extern "C" __global__ __launch_bounds__(mo::kThreads) void mo_unpack1_elem_kernel(const mo::KDesc d) {
  mo::copy_tile<false, true>(d, blockIdx.x);
}

// Byte equality of two ranges (both 16-byte aligned), one 16 KiB tile per workgroup. Lanes
// that see a difference write 1 to *flag (pinned host memory the host cleared before the
// launch); equal ranges write nothing. The host reads the flag once an event recorded after
// the launch has completed.
extern "C" __global__ __launch_bounds__(mo::kThreads) void mo_equal_kernel(const char* a, const char* b,
                                                                            uint64_t nbytes, uint32_t* flag) {
  using namespace mo;
  const uint32_t tid = threadIdx.x;
  const uint64_t tile_off = (uint64_t)blockIdx.x * kTileBytes;
  const uint64_t left = nbytes - tile_off;
  const char* const x = a + tile_off;
  const char* const y = b + tile_off;
  uint32_t diff = 0;
  if (left >= kTileBytes) {
    uint4 u[kUnroll], v[kUnroll];
#pragma unroll
    for (int k = 0; k < kUnroll; ++k) {
      u[k] = ld16(x + (size_t)(k * kThreads + tid) * 16);
      v[k] = ld16(y + (size_t)(k * kThreads + tid) * 16);
    }
#pragma unroll
    for (int k = 0; k < kUnroll; ++k) diff |= (u[k].x ^ v[k].x) | (u[k].y ^ v[k].y) | (u[k].z ^ v[k].z) | (u[k].w ^ v[k].w);
  } else {
    const uint32_t nvec = (uint32_t)(left / 16);
    for (uint32_t c = tid; c < nvec; c += kThreads) {
      const uint4 u = ld16(x + (size_t)c * 16), v = ld16(y + (size_t)c * 16);
      diff |= (u.x ^ v.x) | (u.y ^ v.y) | (u.z ^ v.z) | (u.w ^ v.w);
    }
    for (uint32_t i = nvec * 16 + tid; i < (uint32_t)left; i += kThreads)
      diff |= (uint32_t)(ld<uint8_t>(x + i) ^ ld<uint8_t>(y + i));
  }
  if (diff) st((char*)flag, 1u);
}

// Device <-> pinned-host copy through the shader engines instead of a DMA engine.
// Each lane keeps kLinkUnroll 16-byte transfers in flight; the grid strides over the buffer.
extern "C" __global__ __launch_bounds__(mo::kThreads) void mo_link_copy_kernel(char* __restrict__ dst,
                                                                                const char* __restrict__ src,
                                                                                uint64_t nbytes) {
  using namespace mo;
  const uint64_t nvec = nbytes / 16;
  const uint64_t lanes = (uint64_t)gridDim.x * kThreads;
  const uint64_t step = lanes * kLinkUnroll;
  uint64_t base = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  for (; base + (kLinkUnroll - 1) * lanes < nvec; base += step) {
    uint4 v[kLinkUnroll];
#pragma unroll
    for (int k = 0; k < kLinkUnroll; ++k) v[k] = ld16(src + (base + k * lanes) * 16);
#pragma unroll
    for (int k = 0; k < kLinkUnroll; ++k) st16(dst + (base + k * lanes) * 16, v[k]);
  }
  for (; base < nvec; base += lanes) st16(dst + base * 16, ld16(src + base * 16));
  if (blockIdx.x == 0) {
    for (uint64_t b = nvec * 16 + threadIdx.x; b < nbytes; b += kThreads) st(dst + b, ld<uint8_t>(src + b));
  }
}


// ------------------------------------------------------------------------------------------
// Wire coding of a staging segment (format in mo_wire.h). Three kernels code a segment into a
// wire buffer: each tile's exponent model and rANS stream into the working space, with its coded
// size (a wave per tile, four a workgroup, which share no LDS and never wait for each other); a
// scan of the tile sizes into offsets plus the header and the raw tail (one workgroup, whose waves
// meet once per 4 096 tiles); then each tile assembled at its offset (a workgroup per tile). Two
// kernels decode one, a workgroup of one wave per tile: one looks a slot's rank up first, the
// other its whole entry, for segments whose tiles are all resident with that table.
// Stores into the wire buffer go through a buffer resource bounded by the buffer's capacity, those
// of a tile's stream words through one over the 32 KiB that the working space keeps for them: the
// callers pass at least wire_capacity(raw_bytes), which covers both (mo_wire_encode checks it). The
// decoder reads the coded stream through a resource too, so a stream that arrives damaged cannot
// make it touch memory outside its buffers.
namespace mo {
constexpr int kWireWaves = kThreads / 64;
constexpr uint32_t kWireOob = 0x80000000u;  // a buffer offset past every wire buffer: the access is dropped
static_assert(kWireWaves == (int)kWireTilesPerGroup, "one wave per tile");

__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, m, 64));
  return v;
}
__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += (uint32_t)__shfl_xor((int)v, m, 64);
  return v;
}
// Inclusive prefix sum over the wave's lanes.
__device__ __forceinline__ uint32_t wave_scan(uint32_t v, uint32_t lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = (uint32_t)__shfl_up((int)v, d, 64);
    if (lane >= (uint32_t)d) v += y;
  }
  return v;
}
// Inclusive prefix maximum over the wave's lanes (values >= 0), by DPP moves: shifts by 1, 2, 4
// and 8 lanes within each row of 16, then row 0's last lane into row 1 and row 2's into row 3,
// then lane 31 into rows 2 and 3. Lanes a move has no source for take 0.
__device__ __forceinline__ uint32_t wave_scan_max_dpp(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false));  // row_shr:1
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false));  // row_shr:2
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false));  // row_shr:4
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false));  // row_shr:8
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));  // row_bcast:15
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));  // row_bcast:31
  return v;
}
// Lanes below this one whose bit is set in `mask`.
__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}
__device__ __forceinline__ uint32_t word_of(const uint4& v, int k) {
  const uint32_t w = k < 2 ? v.x : k < 4 ? v.y : k < 6 ? v.z : v.w;
  return (k & 1) ? w >> 16 : w & 0xffffu;
}
__device__ __forceinline__ uint32_t exponent_of(uint32_t word) { return (word >> 7) & 0xffu; }
__device__ __forceinline__ uint32_t sign_mantissa_of(uint32_t word) { return ((word >> 8) & 0x80u) | (word & 0x7fu); }
__device__ __forceinline__ __amdgpu_buffer_rsrc_t wire_rsrc(const char* p, uint64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)(bytes < 0x7fffffffull ? bytes : 0x7fffffffull),
                                           0x00020000);
}
// Orders the wave's own LDS accesses (a wave's LDS operations execute in order; this keeps the
// compiler from moving them across).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
// Coder table entry of one exponent of frequency f and cumulative frequency c: {f << 20, less one (a
// state above it emits a word first); f and 4096 - f as the halves of a word; the float just under
// 1 / f by which a state is divided; c}. With 1 / f * (1 - 2^-22) rounded, trunc(float(x) * that)
// is floor(x / f) or one less for every x < f << 20: four roundings of at most 2^-24 each (of 1 / f,
// of it times 1 - 2^-22, of float(x), of their product) keep the product above x / f * (1 - 2^-21),
// which is less than a half below x / f under 2^20, and (1 - 2^-22)(1 + 2^-24)^4 < 1 keeps it below.
__device__ __forceinline__ float coder_rcp(uint32_t f) { return (1.0f / (float)f) * (1.0f - 0x1p-22f); }
}  // namespace mo

// Pass 1: each tile's exponent frequencies, normalised, its rANS stream and final states in the
// working space, and the tile's coded size into the stream's tile table. One wave per tile, 8 KiB
// of LDS a wave: the counts, and in their place afterwards each exponent's coder entry and
// reciprocal and two groups' exponents. State l codes the tile's words 64 j + l, so a group of 8
// rounds is 1 KiB of consecutive words: one 16-byte load a lane, moved to LDS, read back one byte
// a round.
// Bound by instruction issue, four cycles a wave and instruction: 13.5 waves a CU for a 113 MB
// segment, each counting 16 384 words and walking 256 rounds (of 66 us, by leaving parts out: the
// rounds 36, the counts 18, the table and the loads 12). The counts are LDS atomics on 8 copies of
// each bin (a wave's words share a few exponents, and atomics on one address serialise; 8 copies
// leave about three lanes an address): three instructions a word where adding once per distinct
// value of a lane's 8 words took 21. A round divides by a float reciprocal with one correction
// step, where the multiply-high and the low product take four times the issue of the others each;
// the entries it needs are read a group ahead of the coding chain. A 113 MB segment of activations,
// warm: 92 us before, 64 now (105 and 85 from memory); a 256 KiB segment 45 us before, 28 now.
extern "C" __global__ __launch_bounds__(mo::kThreads) void mo_wire_sizes_kernel(const char* raw, uint64_t raw_bytes,
                                                                                 char* wire, uint64_t wire_capacity) {
  using namespace mo;
  typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
  constexpr uint32_t kCopies = 8;
  __shared__ __attribute__((aligned(256 * 4 * kCopies))) uint32_t space[kWireWaves][256 * kCopies];
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint64_t tile = (uint64_t)blockIdx.x * kWireTilesPerGroup + wave;
  if (tile >= wire_tiles(raw_bytes)) return;  // wave-uniform; the waves never synchronise
  const uint32_t n = wire_tile_words(raw_bytes, tile), J = n / kWireLanes, nb = n / kWireBlockVals;
  const char* src = raw + tile * kWireTileRaw;
  const __amdgpu_buffer_rsrc_t w = wire_rsrc(wire, wire_capacity);
  const uint32_t rec = (uint32_t)(wire_scratch_offset(raw_bytes) + tile * kWireScratchTile);
  MO_LDS uint32_t* const cnt = (MO_LDS uint32_t*)space[wave];
  MO_LDS mo_u32x4* const cod = (MO_LDS mo_u32x4*)space[wave];                                     // 4 KiB
  MO_LDS unsigned char* const grp = (MO_LDS unsigned char*)space[wave] + 256 * sizeof(mo_u32x4);  // 1 KiB
  for (uint32_t b = lane; b < 256 * kCopies / 4; b += 64) *(MO_LDS mo_u32x4*)(cnt + 4 * b) = mo_u32x4{0, 0, 0, 0};
  wave_lds_fence();
  // Histogram, 8 loads of 16 bytes a lane in flight (n / 8 is a multiple of 64, so a load is taken
  // by all lanes or by none).
  // A bin's address: the exponent field moved to bits 5-12, or-ed into the lane's copy of bin 0.
  const uint32_t mine = (uint32_t)(uintptr_t)(cnt + (lane & (kCopies - 1)));
  auto count = [&](uint32_t field) {
    __hip_atomic_fetch_add((MO_LDS uint32_t*)(uintptr_t)((field & (255u * 4 * kCopies)) | mine), 1u, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WAVEFRONT);
  };
  for (uint32_t c0 = 0; c0 < n / 8; c0 += 8 * 64) {
    uint4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (c0 + 64 * i < n / 8) v[i] = ld16(src + 16 * (uint64_t)(c0 + 64 * i + lane));
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (c0 + 64 * i >= n / 8) continue;
      const uint32_t d[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        count(d[k] >> 2);   // bits 7-14
        count(d[k] >> 18);  // bits 23-30
      }
    }
  }
  wave_lds_fence();
  // Normalised frequencies: lane l owns exponents 4l .. 4l + 3.
  uint32_t f[4], fsum = 0, best = 0, pres = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t e = 4 * lane + k;
    const mo_u32x4 a = *(const MO_LDS mo_u32x4*)(cnt + kCopies * e), b = *(const MO_LDS mo_u32x4*)(cnt + kCopies * e + 4);
    const uint32_t c = a.x + a.y + a.z + a.w + b.x + b.y + b.z + b.w;
    f[k] = c ? max(1u, 8u * c / nb) : 0u;  // floor(c * 4096 / n), n = 512 nb
    fsum += f[k];
    pres += c ? 1u : 0u;
    best = max(best, (c << 8) | (255u - e));  // most frequent, the smallest exponent on ties
  }
  fsum = wave_sum(fsum);
  best = wave_max(best);
  const uint32_t top_e = 255u - (best & 0xffu);
  uint32_t most = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (4 * lane + k == top_e) most = f[k];
  const int adjusted = (int)__shfl((int)most, (int)(top_e >> 2), 64) + (int)(1u << kWireProbBits) - (int)fsum;
  bool raw_tile = adjusted < 1;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (4 * lane + k == top_e) f[k] = (uint32_t)adjusted;
  // cumulative frequencies, the table (ascending exponents) and the coder entries
  const uint32_t lsum = f[0] + f[1] + f[2] + f[3];
  uint32_t cum = wave_scan(lsum, lane) - lsum;
  const uint32_t rank_incl = wave_scan(pres, lane);
  const uint32_t nsym = (uint32_t)__shfl((int)rank_incl, 63, 64);
  uint32_t rank = rank_incl - pres;
  wave_lds_fence();  // every lane has read its counts
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t e = 4 * lane + k;
    if (f[k]) {
      __builtin_amdgcn_raw_buffer_store_b32(e | (f[k] << 8), w, (int)(rec + kWireScratchTable + 4 * rank), 0, 0);
      ++rank;
      cod[e] = mo_u32x4{(f[k] << 20) - 1, f[k] | ((1u << kWireProbBits) - f[k]) << 16,
                        __builtin_bit_cast(uint32_t, coder_rcp(f[k])), cum};
    }
    cum += f[k];
  }
  wave_lds_fence();
  // rANS over j = J-1 .. 0; the stream fills the working space from its end downwards
  uint32_t x = kWireStateLow, top = J * kWireLanes;
  const __amdgpu_buffer_rsrc_t out = wire_rsrc(wire + rec + kWireScratchStream, 2 * kWireTileVals);
  if (!raw_tile) {
    const int ngroups = (int)(J / 8);
    auto load = [&](int g) { return ld16(src + 1024 * (uint64_t)(g > 0 ? g : 0) + 16 * lane); };  // past 0: a spare
    uint4 next = load(ngroups - 1);
    // The entries of a group's 8 rounds, read while the group before is coded (buffer: group parity).
    auto entries = [&](int g, mo_u32x4(&t)[8], uint32_t buffer) {
      auto pair = [](uint32_t d) { return (d >> 7) & 0x00ff00ffu; };  // a dword's exponents, bytes 0 and 2
      const u32x2 e8 = {__builtin_amdgcn_perm(pair(next.y), pair(next.x), 0x06040200u),
                        __builtin_amdgcn_perm(pair(next.w), pair(next.z), 0x06040200u)};
      next = load(g - 1);
      MO_LDS unsigned char* const to = grp + 512 * buffer;
      *(MO_LDS u32x2*)(to + 8 * lane) = e8;
      wave_lds_fence();
#pragma unroll
      for (int r = 0; r < 8; ++r) t[r] = cod[to[64 * r + lane]];
    };
    auto code = [&](const mo_u32x4(&t)[8]) {
#pragma unroll
      for (int r = 7; r >= 0; --r) {
        // elements read into scalars first: a bit cast of the vector element itself reads the first
        const uint32_t bound = t[r][0], freqs = t[r][1], rcp = t[r][2], c = t[r][3];
        const uint32_t fr = freqs & 0xffffu;
        const bool emit = x > bound;
        const uint64_t bal = __ballot(emit);
        top -= (uint32_t)__popcll(bal);
        // every lane stores, a lane that emits nothing at an offset the buffer drops: a fixed
        // number of stores a group, which keeps the compiler's wait for `next` exact
        const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, top));
        __builtin_amdgcn_raw_buffer_store_b16((unsigned short)(x & 0xffffu), out, (int)(2 * (emit ? at : kWireOob / 2)), 0, 0);
        x = emit ? x >> 16 : x;
        uint32_t q = (uint32_t)((float)x * __builtin_bit_cast(float, rcp));  // floor(x / fr), or one less
        q += x - __umul24(q, fr) >= fr ? 1u : 0u;
        x = __umul24(q, freqs >> 16) + (x + c);  // (q << 12) + x % fr + c
      }
    };
    mo_u32x4 even[8], odd[8];
    entries(ngroups - 1, even, 0);
    for (int g = ngroups - 1; g >= 0; g -= 2) {  // past group 0 the entries are spares
      entries(g - 1, odd, 1);
      code(even);
      if (g == 0) break;
      entries(g - 2, even, 0);
      code(odd);
    }
  }
  const uint32_t nwords = J * kWireLanes - top;
  __builtin_amdgcn_raw_buffer_store_b32(x, w, (int)(rec + kWireScratchStates + 4 * lane), 0, 0);
  const uint32_t rans = wire_rans_tile(n, nsym, nwords), plain = wire_raw_tile(n);
  raw_tile = raw_tile || rans >= plain;
  if (lane == 0) {
    const uint32_t size = raw_tile ? plain : rans;
    __builtin_amdgcn_raw_buffer_store_b128(
        mo_u32x4{raw_tile ? kWireModeRaw : (kWireModeRans | (nsym << 8)), raw_tile ? 0u : nwords, top, size}, w,
        (int)rec, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b32(size, w, (int)(kWireHeader + 4 * tile), 0, 0);
  }
}

// Pass 2 (one workgroup of kWireScanThreads): tile sizes -> tile offsets (exclusive scan from
// tiles_start), the header, the raw tail; the total also to `host_total` (pinned host memory,
// may be null), where the copy engine's issuer reads it once this kernel has completed.
// Latency-bound: a lane takes four tiles and the waves' sums meet once per 4 096 tiles (a 113 MB
// segment has 3 456); with one tile a lane and a scan through LDS in ten rounds it took 8.5 us, now 4.9.
extern "C" __global__ __launch_bounds__(mo::kWireScanThreads) void mo_wire_scan_kernel(const char* raw,
                                                                                        uint64_t raw_bytes, char* wire,
                                                                                        uint64_t wire_capacity,
                                                                                        uint64_t* host_total) {
  using namespace mo;
  constexpr uint32_t kWaves = kWireScanThreads / 64, kChunk = 4 * kWireScanThreads;
  __shared__ uint32_t sums[2][kWaves];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const __amdgpu_buffer_rsrc_t w = wire_rsrc(wire, wire_capacity);
  const uint64_t tiles = wire_tiles(raw_bytes);
  const uint64_t tail = raw_bytes % kWireBlockBytes, tail_src = wire_blocks(raw_bytes) * kWireBlockBytes;
  const uint64_t data_start = wire_data_start(raw_bytes);
  for (uint64_t i = tid; i < tail; i += kWireScanThreads)
    __builtin_amdgcn_raw_buffer_store_b8(ld<uint8_t>(raw + tail_src + i), w, (int)(data_start + i), 0, 0);
  uint64_t carry = wire_tiles_start(raw_bytes);
  for (uint64_t base = 0; base < tiles; base += kChunk) {
    const uint64_t t = base + 4 * tid;
    uint32_t v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      v[k] = t + k < tiles ? __builtin_amdgcn_raw_buffer_load_b32(w, (int)(kWireHeader + 4 * (t + k)), 0, 0) : 0u;
    const uint32_t mine = v[0] + v[1] + v[2] + v[3], upto = wave_scan(mine, lane);
    // two sets of sums in turn: a wave may still read the last chunk's
    const uint32_t set = (uint32_t)(base / kChunk) & 1;
    if (lane == 63) sums[set][wave] = upto;
    __syncthreads();
    uint32_t before = 0, chunk = 0;
#pragma unroll
    for (uint32_t k = 0; k < kWaves; ++k) {
      const uint32_t s = sums[set][k];
      before += k < wave ? s : 0u;
      chunk += s;
    }
    uint32_t at = (uint32_t)carry + before + upto - mine;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (t + k < tiles) __builtin_amdgcn_raw_buffer_store_b32(at, w, (int)(kWireHeader + 4 * (t + k)), 0, 0);
      at += v[k];
    }
    carry += chunk;
  }
  if (tid == 0) {
    __builtin_amdgcn_raw_buffer_store_b32((uint32_t)carry, w, 0, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b32((uint32_t)(carry >> 32), w, 4, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b32((uint32_t)raw_bytes, w, 8, 0, 0);
    __builtin_amdgcn_raw_buffer_store_b32((uint32_t)tiles, w, 12, 0, 0);
    if (host_total) st((char*)host_total, carry);
  }
}

// Pass 3: assemble each tile at its offset (header, then the raw words, or the sign-mantissa
// bytes, table, final states and stream from the working space). One workgroup a tile: HBM-bound
// (the raw words once more, the stream, 0.67 of the raw bytes out), so every lane has its 8 loads
// of raw words in flight before it knows the tile's record, and stores and loads are coalesced
// runs of a wave. A 113 MB segment: 56 us with one wave a tile and 4-byte stream copies, now 32.7
// (113 MB of raw words and 19 of stream in, 76 of coded bytes out: 6.4 TB/s); 58 and 35 from memory.
extern "C" __global__ __launch_bounds__(mo::kThreads) void mo_wire_encode_kernel(const char* raw, uint64_t raw_bytes,
                                                                                  char* wire, uint64_t wire_capacity) {
  using namespace mo;
  const uint32_t tid = threadIdx.x;
  const uint64_t tile = blockIdx.x;
  const uint32_t n = wire_tile_words(raw_bytes, tile);
  const char* src = raw + tile * kWireTileRaw;
  const __amdgpu_buffer_rsrc_t w = wire_rsrc(wire, wire_capacity);
  const uint32_t rec = (uint32_t)(wire_scratch_offset(raw_bytes) + tile * kWireScratchTile);
  constexpr uint32_t kLoads = kWireTileVals / 8 / kThreads;  // 8
  uint4 v[kLoads];
#pragma unroll
  for (uint32_t i = 0; i < kLoads; ++i) {
    const uint32_t c = i * kThreads + tid;
    v[i] = c < n / 8 ? ld16(src + 16 * (uint64_t)c) : make_uint4(0, 0, 0, 0);
  }
  const uint32_t toff = __builtin_amdgcn_raw_buffer_load_b32(w, (int)(kWireHeader + 4 * tile), 0, 0);
  const mo_u32x4 r = __builtin_amdgcn_raw_buffer_load_b128(w, (int)rec, 0, 0);
  const uint32_t head = r[0], nwords = r[1], first = r[2];
  if (tid == 0) __builtin_amdgcn_raw_buffer_store_b128(mo_u32x4{head, nwords, 0u, 0u}, w, (int)toff, 0, 0);
  const uint32_t body = toff + kWireTileHeader;
  if ((head & 3u) == kWireModeRaw) {
#pragma unroll
    for (uint32_t i = 0; i < kLoads; ++i) {
      const uint32_t c = i * kThreads + tid;
      if (c < n / 8)
        __builtin_amdgcn_raw_buffer_store_b128(mo_u32x4{v[i].x, v[i].y, v[i].z, v[i].w}, w, (int)(body + 16 * c), 0, 0);
    }
    return;
  }
  // sign-mantissa bytes: 8 words in, 8 bytes out a lane and load
#pragma unroll
  for (uint32_t i = 0; i < kLoads; ++i) {
    const uint32_t c = i * kThreads + tid;
    auto pair = [](uint32_t x) { return (x & 0x007f007fu) | ((x >> 8) & 0x00800080u); };  // bytes 0 and 2
    auto four = [&](uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(pair(b), pair(a), 0x06040200u); };
    if (c < n / 8)
      __builtin_amdgcn_raw_buffer_store_b64(mo_u32x2{four(v[i].x, v[i].y), four(v[i].z, v[i].w)}, w, (int)(body + 8 * c),
                                            0, 0);
  }
  // table, zero-padded to 16 bytes (nsym is at most 256, one entry a lane)
  const uint32_t nsym = head >> 8, tab = body + n, tab_words = (uint32_t)wire_align16(4 * nsym) / 4;
  if (tid < tab_words) {
    const uint32_t e = tid < nsym ? __builtin_amdgcn_raw_buffer_load_b32(w, (int)(rec + kWireScratchTable + 4 * tid), 0, 0) : 0u;
    __builtin_amdgcn_raw_buffer_store_b32(e, w, (int)(tab + 4 * tid), 0, 0);
  }
  // final states
  const uint32_t states = tab + 4 * tab_words;
  if (tid < kWireLanes)
    __builtin_amdgcn_raw_buffer_store_b32(
        __builtin_amdgcn_raw_buffer_load_b32(w, (int)(rec + kWireScratchStates + 4 * tid), 0, 0), w,
        (int)(states + 4 * tid), 0, 0);
  // the stream, 8 words (16 bytes) a lane, zero-padded to 16 bytes: it starts at word `first` of the
  // working space, so a lane reads the five aligned dwords around its words and shifts them
  const uint32_t stream = states + 4 * kWireLanes, at = rec + kWireScratchStream + 4 * (first / 2);
  const uint32_t shift = 16 * (first & 1);
  for (uint32_t c = tid; c < (nwords + 7) / 8; c += kThreads) {
    const mo_u32x4 lo = __builtin_amdgcn_raw_buffer_load_b128(w, (int)(at + 16 * c), 0, 0);
    const uint32_t hi = __builtin_amdgcn_raw_buffer_load_b32(w, (int)(at + 16 * c + 16), 0, 0);
    mo_u32x4 o;
    const uint32_t left = nwords - 8 * c;  // words of this piece and after
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
      const uint32_t x = __builtin_amdgcn_alignbit(k < 3 ? lo[k < 3 ? k + 1 : 0] : hi, lo[k], shift);
      o[k] = left >= 2 * k + 2 ? x : left == 2 * k + 1 ? x & 0xffffu : 0u;
    }
    __builtin_amdgcn_raw_buffer_store_b128(o, w, (int)(stream + 16 * c), 0, 0);
  }
}

// Decode a coded stream of `raw_bytes` into `raw`. Grid: max(tiles, 1) workgroups of one wave, a tile
// each; the first also copies the raw tail. In LDS: the slots' table, the entries by rank (2 KiB), a
// ring of the stream's next 512 words, and one group's exponents: state l decodes the tile's words
// 64 j + l, so the exponents of 8 rounds are 1 KiB of consecutive words, written out as one 16-byte
// store a lane.
// Bound by a round's chain of LDS reads and the vector instructions between them, and where a CU
// holds many tiles nearly as much by the issue of those: so a round is kept short. A wave is its own
// workgroup (its arrays lie at fixed LDS addresses, and tiles spread evenly over the CUs); the ring
// repeats its first 256 words past its end, so that the four rounds between refills index it without
// wrapping; and a byte select brings a stream word in.
// kDirect: the slots' table holds whole entries (16 KiB; 20 KiB a tile, 8 tiles a CU), two LDS reads
// a round. Otherwise it holds ranks (4 KiB; 8 KiB a tile, 20 tiles a CU), whose entries a third read
// brings; an entry's parts sit where the multiply, the subtraction and the byte store take them as
// they are. 113 MB: 66 us with four tiles a workgroup and 26 instructions a round, 51 by ranks now; a
// 256 KiB segment 47 us, 33 by ranks, 30 direct. These are calls back to back, the stream in the
// cache; from memory every tile also waits for the chain of loads in front of its first round (tile
// offset, head, then table, states and stream): 80 and 76 us, 51 and 40 by ranks, 37 direct.
// Reads go through a resource over [wire, wire + wire_bytes), and writes stay inside
// [raw, raw + raw_bytes) whatever the stream holds: a damaged header is clamped, and table values
// only index the wave's own LDS arrays.
namespace mo {
template <bool kDirect>
__device__ __forceinline__ void wire_decode_body(const char* wire, uint64_t wire_bytes, uint64_t raw_bytes, char* raw) {
  constexpr uint32_t kSlots = 1u << kWireProbBits, kRing = 512, kAgain = 256;
  // a slot's rank (a byte), or with kDirect its entry: slot - c | exponent << 12 | f - 1 << 20
  __shared__ __attribute__((aligned(16))) unsigned char slots[kDirect ? 4 * kSlots : kSlots];
  __shared__ __attribute__((aligned(16))) mo_u32x2 rank_entry[256];  // {f, c | exponent << 16}
  __shared__ __attribute__((aligned(16))) unsigned short ring[kRing + kAgain];
  __shared__ __attribute__((aligned(16))) unsigned char group[8 * kWireLanes];
  const uint32_t lane = threadIdx.x;
  const __amdgpu_buffer_rsrc_t w = wire_rsrc(wire, wire_bytes);
  if (blockIdx.x == 0) {
    const uint64_t tail = raw_bytes % kWireBlockBytes, tail_dst = wire_blocks(raw_bytes) * kWireBlockBytes;
    const uint64_t data_start = wire_data_start(raw_bytes);
    for (uint64_t i = lane; i < tail; i += 64)
      st(raw + tail_dst + i, (uint8_t)__builtin_amdgcn_raw_buffer_load_b8(w, (int)(data_start + i), 0, 0));
  }
  const uint64_t tile = blockIdx.x;
  if (tile >= wire_tiles(raw_bytes)) return;
  const uint32_t n = wire_tile_words(raw_bytes, tile), J = n / kWireLanes;
  char* const dst = raw + tile * kWireTileRaw;
  const uint32_t toff = __builtin_amdgcn_raw_buffer_load_b32(w, (int)(kWireHeader + 4 * tile), 0, 0);
  const uint32_t head = __builtin_amdgcn_raw_buffer_load_b32(w, (int)toff, 0, 0);
  const uint32_t body = toff + kWireTileHeader;
  if ((head & 3u) != kWireModeRans) {
    for (uint32_t c = lane; c < n / 8; c += 64) {
      const mo_u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(w, (int)(body + 16 * c), 0, 0);
      st16(dst + 16 * (uint64_t)c, make_uint4(v.x, v.y, v.z, v.w));
    }
    return;
  }
  const uint32_t nsym = min((head >> 8) & 0x1ffu, 256u);
  MO_LDS unsigned char* const sr = (MO_LDS unsigned char*)slots;
  MO_LDS mo_u32x2* const re = (MO_LDS mo_u32x2*)rank_entry;
  MO_LDS unsigned short* const words = (MO_LDS unsigned short*)ring;
  MO_LDS unsigned char* const grp = (MO_LDS unsigned char*)group;
  // Table entries in rank order with their cumulative frequencies; each entry's first slot is
  // marked with its rank (rank 0 starts at slot 0, where every slot's mark starts).
  const uint32_t tab = body + n;
  for (uint32_t i = lane; i < sizeof(slots) / 16; i += 64) *(MO_LDS mo_u32x4*)(sr + 16 * i) = mo_u32x4{0, 0, 0, 0};
  wave_lds_fence();
  uint32_t carry = 0;
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    const uint32_t r = 64 * k + lane;
    const uint32_t e = r < nsym ? __builtin_amdgcn_raw_buffer_load_b32(w, (int)(tab + 4 * r), 0, 0) : 0u;
    const uint32_t f = r < nsym ? min((e >> 8) & 0x1fffu, kSlots) : 0u;
    const uint32_t incl = wave_scan(f, lane), c = carry + incl - f;
    carry += (uint32_t)__shfl((int)incl, 63, 64);
    re[r] = mo_u32x2{f, (c & 0xffffu) | ((e & 0xffu) << 16)};
    if (f && c < kSlots) sr[kDirect ? 4 * c : c] = (unsigned char)r;
  }
  wave_lds_fence();
  // Every slot's rank: the last mark at or before it (marks rise with the slot). Four consecutive
  // slots a lane: the maxima within them, a prefix maximum over the lanes' last ones, and the carry
  // of the rounds before.
  uint32_t before = 0;
  for (uint32_t row = 0; row < kSlots / 256; ++row) {
    uint32_t m[4];
    if (kDirect) {
      const mo_u32x4 four = *(const MO_LDS mo_u32x4*)(sr + 1024 * row + 16 * lane);
#pragma unroll
      for (int k = 0; k < 4; ++k) m[k] = four[k];
    } else {
      const uint32_t four = *(const MO_LDS uint32_t*)(sr + 256 * row + 4 * lane);
#pragma unroll
      for (int k = 0; k < 4; ++k) m[k] = (four >> (8 * k)) & 0xffu;
    }
#pragma unroll
    for (int k = 1; k < 4; ++k) m[k] = max(m[k - 1], m[k]);
    const uint32_t upto = wave_scan_max_dpp(m[3]);
    const uint32_t left = max(before, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)upto, 0x138, 0xf, 0xf, false));  // wave_shr:1
#pragma unroll
    for (int k = 0; k < 4; ++k) m[k] = max(left, m[k]);
    if (kDirect) {
      mo_u32x4 entries;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const mo_u32x2 t = re[m[k]];
        const uint32_t f = t[0], ce = t[1];
        entries[k] = ((256 * row + 4 * lane + k - ce) & 0xfffu) | ((ce >> 16) << 12) | ((f - 1) << 20);
      }
      *(MO_LDS mo_u32x4*)(sr + 1024 * row + 16 * lane) = entries;
    } else {
      *(MO_LDS uint32_t*)(sr + 256 * row + 4 * lane) = m[0] | (m[1] << 8) | (m[2] << 16) | (m[3] << 24);
    }
    before = max(before, (uint32_t)__builtin_amdgcn_readlane((int)upto, 63));
  }
  // States, and the stream's first 512 words into the ring (word i at i % 512, and again at
  // 512 + i % 512 where that is below 768); `next` holds the 2 words this lane brings in at the
  // next refill.
  const uint32_t states = tab + (uint32_t)wire_align16(4 * nsym);
  uint32_t x = __builtin_amdgcn_raw_buffer_load_b32(w, (int)(states + 4 * lane), 0, 0);
  const uint32_t stream = states + 4 * kWireLanes;
  auto refill = [&](uint32_t at, uint32_t v) {  // 128 words from ring word `at` on, a multiple of 128
    *(MO_LDS uint32_t*)(words + at + 2 * lane) = v;
    if (at < kAgain) *(MO_LDS uint32_t*)(words + kRing + at + 2 * lane) = v;
  };
#pragma unroll
  for (uint32_t q = 0; q < 4; ++q)
    refill(128 * q, __builtin_amdgcn_raw_buffer_load_b32(w, (int)(stream + 256 * q + 4 * lane), 0, 0));
  uint32_t next = __builtin_amdgcn_raw_buffer_load_b32(w, (int)(stream + 1024 + 4 * lane), 0, 0);
  wave_lds_fence();
  uint32_t ptr = 0, wb = 0;  // words read so far; the first word the ring still holds
  // the group's sign-mantissa bytes (words 8 l .. 8 l + 7 of its 512), one group ahead
  const uint32_t ngroups = J / 8;
  mo_u32x2 sm_next = __builtin_amdgcn_raw_buffer_load_b64(w, (int)(body + 8 * lane), 0, 0);
  for (uint32_t g = 0; g < ngroups; ++g) {
    const mo_u32x2 sm = sm_next;
    sm_next = __builtin_amdgcn_raw_buffer_load_b64(w, (int)(body + 512 * (g + 1) + 8 * lane), 0, 0);  // a spare past the last
    uint32_t at;  // the ring's byte at which the next word lies
    auto wrap = [&] {
      at = 2 * (ptr % kRing);
      asm("" : "+s"(at));  // a number of its own: known to be a double, it is doubled again each round
    };
    wrap();
#pragma unroll
    for (uint32_t r = 0; r < 8; ++r) {
      const uint32_t slot = x % kSlots, high = x >> kWireProbBits;
      uint32_t exponent;
      if (kDirect) {
        const uint32_t t = *(const MO_LDS uint32_t*)(sr + 4 * slot);
        x = __umul24(t >> 20, high) + (high + (t & 0xfffu));
        exponent = t >> 12;
      } else {
        const mo_u32x2 t = re[sr[slot]];
        const uint32_t f = t[0], ce = t[1];
        x = __umul24(f, high) + (slot - (ce & 0xffffu));
        exponent = ce >> 16;
      }
      const bool need = x < kWireStateLow;
      const uint64_t bal = __ballot(need);
      const uint32_t mine = __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
      const uint32_t word = *(const MO_LDS unsigned short*)((const MO_LDS unsigned char*)words + (2 * mine + at));
      x = __builtin_amdgcn_perm(x, word, need ? 0x05040100u : 0x07060504u);  // (x << 16) | word, or x
      ptr += (uint32_t)__popcll(bal);
      at += 2 * (uint32_t)__popcll(bal);
      grp[64 * r + lane] = (unsigned char)exponent;
      // Every four rounds, which read at most 256 words: the ring holds at least 512 - 127 of them.
      // Words [wb, wb + 128) are consumed: their ring quarter takes words [wb + 512, wb + 640).
      if (r % 4 == 3) {
        while (ptr - wb >= 128) {
          refill(wb % kRing, next);
          wb += 128;
          next = __builtin_amdgcn_raw_buffer_load_b32(w, (int)(stream + 2 * (wb + kRing) + 4 * lane), 0, 0);
          wave_lds_fence();
        }
        wrap();
      }
    }
    wave_lds_fence();
    const mo_u32x2 ex = *(const MO_LDS mo_u32x2*)(grp + 8 * lane);
    uint32_t o[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {  // words 2k and 2k + 1: their bytes spread to the halves, then shifted into place
      const uint32_t spread = k & 1 ? 0x0c070c06u : 0x0c050c04u;
      const uint32_t s = __builtin_amdgcn_perm(sm[k >> 1], 0u, spread), m = __builtin_amdgcn_perm(ex[k >> 1], 0u, spread);
      o[k] = ((s & 0x00800080u) << 8) | (m << 7) | (s & 0x007f007fu);
    }
    st16(dst + 1024 * (uint64_t)g + 16 * lane, make_uint4(o[0], o[1], o[2], o[3]));
    wave_lds_fence();  // the group buffer is read before the next group writes it
  }
}
}  // namespace mo

extern "C" __global__ __launch_bounds__(64) void mo_wire_decode_kernel(const char* wire, uint64_t wire_bytes,
                                                                       uint64_t raw_bytes, char* raw) {
  mo::wire_decode_body<false>(wire, wire_bytes, raw_bytes, raw);
}

extern "C" __global__ __launch_bounds__(64) void mo_wire_decode_direct_kernel(const char* wire, uint64_t wire_bytes,
                                                                              uint64_t raw_bytes, char* raw) {
  mo::wire_decode_body<true>(wire, wire_bytes, raw_bytes, raw);
}
