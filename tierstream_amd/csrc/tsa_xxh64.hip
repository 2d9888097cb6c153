// Device XXH64 (seed 0) for units already resident in HBM, in two ways:
//
//  * digest: XXH64 keeps four dependent 64-bit chains per input, each chain a sequence of rotl(v + w*P2, 31)*P1 steps.
//    There is no associative combine, so a unit's digest is bound by its chains: one wave runs only them, fed with the
//    products w*P2 by four others. With very many units a quad of lanes per unit does all of it.
//  * verify: checkpoint-parallel. The host hashes every unit once while it fills the pinned tier / the arena and keeps
//    the four accumulators at the start of every segment (a fixed byte count inside each extent). On the device each
//    (unit, segment) pair is an independent quad: start from the segment's checkpoint, run the segment's stripes over
//    the device bytes, and require the next checkpoint (or, for the unit's last segment, the finalized digest equal to
//    the descriptor's hash). All segments of all units run in parallel, so one launch is HBM-bound even for one unit.
//    If every segment agrees, the device bytes' XXH64 equals the descriptor hash exactly (the transitions compose).
//
// Byte order and the algorithm follow the published XXH64 description (reference src/xxh64.cpp:39-112 restates it).
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tsa_device.hpp"
#include "wave_search.hpp"

namespace tsa {
namespace dev {

constexpr uint64_t P1 = 0x9E3779B185EBCA87ull;
constexpr uint64_t P2 = 0xC2B2AE3D27D4EB4Full;
constexpr uint64_t P3 = 0x165667B19E3779F9ull;
constexpr uint64_t P4 = 0x85EBCA77C2B2AE63ull;
constexpr uint64_t P5 = 0x27D4EB2F165667C5ull;

typedef __attribute__((address_space(1))) const uint64_t gword_t;
typedef __attribute__((address_space(1))) uint64_t gout_t;
typedef __attribute__((address_space(1))) const unsigned char gbyte_t;

__device__ __forceinline__ uint64_t rotl64(uint64_t x, int r) { return (x << r) | (x >> (64 - r)); }
// rotl by 31 as two funnel shifts (v_alignbit_b32) on the 32-bit halves: hi' = (hi:lo) >> 1, lo' = (lo:hi) >> 1
__device__ __forceinline__ uint64_t rotl31(uint64_t x) {
  const uint32_t hi = uint32_t(x >> 32), lo = uint32_t(x);
  return uint64_t(__builtin_amdgcn_alignbit(hi, lo, 1u)) << 32 | __builtin_amdgcn_alignbit(lo, hi, 1u);
}
__device__ __forceinline__ uint64_t xround(uint64_t acc, uint64_t w) { return rotl31(acc + w * P2) * P1; }
// The same round on the state b = acc * P1^-1 (mod 2^64): b' = rotl(b * P1 + w * P2, 31), where the sum costs nothing
// (v_mad_u64_u32 adds the product on the way).
constexpr uint64_t inverse64(uint64_t x) {  // modulo 2^64, x odd (Newton: each step doubles the correct bits)
  uint64_t r = x;
  for (int i = 0; i < 6; ++i) r *= 2 - x * r;
  return r;
}
constexpr uint64_t P1inv = inverse64(P1);
__device__ __forceinline__ uint64_t bround(uint64_t b, uint64_t product) { return rotl31(b * P1 + product); }
__device__ __forceinline__ uint64_t xmerge(uint64_t h, uint64_t v) { return (h ^ xround(0, v)) * P1 + P4; }

// A unit's last (< 32) bytes in registers: whole words, then the rest (p is 8-byte aligned).
struct Tail {
  uint64_t word[3] = {0, 0, 0};
  uint64_t rest = 0;
  uint32_t len = 0;
};
__device__ __forceinline__ Tail load_tail(const unsigned char* p, uint32_t len) {
  Tail t;
  t.len = len;
  const uintptr_t at = reinterpret_cast<uintptr_t>(p);
#pragma unroll
  for (uint32_t i = 0; i < 3; ++i)
    if (8 * i + 8 <= len) t.word[i] = *reinterpret_cast<gword_t*>(at + 8 * i);
  if (const uint32_t n = len & 7u) {  // (all its bytes at once: one after the other, each was a memory latency)
#pragma unroll
    for (uint32_t b = 0; b < 7; ++b)
      t.rest |= uint64_t(*reinterpret_cast<gbyte_t*>(at + (len & ~7u) + (b < n ? b : n - 1))) << (8 * b);
    t.rest &= (1ull << (8 * n)) - 1;
  }
  return t;
}
__device__ __forceinline__ void store_tail(unsigned char* p, const Tail& t) {
#pragma unroll
  for (uint32_t i = 0; i < 3; ++i)
    if (8 * i + 8 <= t.len) *reinterpret_cast<uint64_t*>(p + 8 * i) = t.word[i];
  for (uint32_t b = t.len & ~7u; b < t.len; ++b) p[b] = static_cast<unsigned char>(t.rest >> (8 * (b & 7u)));
}

// Digest of the four accumulators, the total length and the tail. Runs on one lane.
__device__ __forceinline__ uint64_t xfinal(const uint64_t v[4], uint64_t total, const Tail& t) {
  uint64_t h;
  if (total >= 32) {
    h = rotl64(v[0], 1) + rotl64(v[1], 7) + rotl64(v[2], 12) + rotl64(v[3], 18);
    for (int k = 0; k < 4; ++k) h = xmerge(h, v[k]);
  } else {
    h = P5;  // seed 0
  }
  h += total;
#pragma unroll
  for (uint32_t i = 0; i < 3; ++i)
    if (8 * i + 8 <= t.len) {
      h ^= xround(0, t.word[i]);
      h = rotl64(h, 27) * P1 + P4;
    }
  uint64_t rest = t.rest;
  uint32_t n = t.len & 7u;
  if (n >= 4) {
    h ^= (rest & 0xFFFFFFFFull) * P1;
    h = rotl64(h, 23) * P2 + P3;
    rest >>= 32;
    n -= 4;
  }
  for (; n > 0; --n, rest >>= 8) {
    h ^= (rest & 0xFFu) * P5;
    h = rotl64(h, 11) * P1;
  }
  h ^= h >> 33;
  h *= P2;
  h ^= h >> 29;
  h *= P3;
  h ^= h >> 32;
  return h;
}

// One chain (lane q of the quad) over n stripes starting at p (p is 8-byte aligned: extents start 256-byte aligned
// in every caller, and every extent but the last is a multiple of 32 bytes). Each block of kBlock stripes is loaded
// (kBlock independent 8-byte loads per lane in flight), then run. The loads go through the global address space (the
// pointer is cast to it): a generic pointer makes flat loads, which also count on the LDS counter and cost 4 % here.
// They are ordinary cached loads: the quad reads 32 bytes of a 128-byte line per stripe and the next three stripes
// read the rest of it, so the line must stay in the CU's cache (a streaming hint that skips it cost 40 % on gfx950).
//
// Measured on one 336 MiB unit (8 KiB segments): this loop reads at 5.8 TB/s; the rounds alone (no loads) run at 17 TB/s, so
// it is bound by the read, not the multiplies. The streamed check below reads aligned segments at 6.4 TB/s. Sixteen stripes a
// block: with 8, 25 MB of 8-byte aligned units took 8.3 us against 7.6; with 32, 34 MB of ragged ones 12.0 against 10.7.
constexpr int kBlock = 16;

// kCopy: each word read is also stored at the same offset from d (the staged unit's bytes into their arena slot while
// they are hashed: the bytes cross HBM once each way).
template <bool kCopy>
__device__ __forceinline__ uint64_t chain_t(uint64_t v, const unsigned char* p, unsigned char* d, uint64_t n,
                                            uint32_t q) {
  gword_t* w = reinterpret_cast<gword_t*>(reinterpret_cast<uintptr_t>(p)) + q;
  gout_t* o = reinterpret_cast<gout_t*>(reinterpret_cast<uintptr_t>(d)) + q;
  uint64_t s = 0;
  for (; s + kBlock <= n; s += kBlock) {
    uint64_t buf[kBlock];
#pragma unroll
    for (int k = 0; k < kBlock; ++k) buf[k] = w[4 * (s + k)];
    if (kCopy) {
#pragma unroll
      for (int k = 0; k < kBlock; ++k) o[4 * (s + k)] = buf[k];
    }
#pragma unroll
    for (int k = 0; k < kBlock; ++k) v = xround(v, buf[k]);
  }
  for (; s < n; ++s) {
    const uint64_t x = w[4 * s];
    if (kCopy) o[4 * s] = x;
    v = xround(v, x);
  }
  return v;
}
__device__ __forceinline__ uint64_t chain(uint64_t v, const unsigned char* p, uint64_t n, uint32_t q) {
  return chain_t<false>(v, p, nullptr, n, q);
}

__device__ __forceinline__ void init_acc(uint64_t v[4]) {
  v[0] = P1 + P2;
  v[1] = P2;
  v[2] = 0;
  v[3] = 0 - P1;
}

// One unit per quad, its stripes in order by the quad itself (launches of very many units).
__global__ __launch_bounds__(256) void digest_quads_kernel(const TsaUnit* __restrict__ units, uint32_t n,
                                                           uint64_t* __restrict__ out) {
  const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t u = gid >> 2, q = gid & 3u;
  const bool live = u < n;
  uint64_t acc[4];
  init_acc(acc);
  uint64_t v = acc[q];
  uint64_t total = 0;
  const unsigned char* tail = nullptr;
  uint32_t tail_len = 0;
  if (live) {
    const TsaUnit un = units[u];
    for (uint32_t e = 0; e < un.n_ext; ++e) {
      const unsigned char* p = static_cast<const unsigned char*>(un.ext[e].ptr);
      const uint64_t b = un.ext[e].bytes;
      const uint64_t stripes = b / 32;
      v = chain(v, p, stripes, q);
      total += b;
      if (e + 1 == un.n_ext) {
        tail = p + stripes * 32;
        tail_len = uint32_t(b - stripes * 32);
      }
    }
  }
  // the quad's accumulators to its lane 0 (all lanes of the wave take part in the shuffles)
  uint64_t all[4];
  const uint32_t base = threadIdx.x & ~3u;
#pragma unroll
  for (int k = 0; k < 4; ++k) all[k] = __shfl(v, int(base + k), 64);
  if (live && q == 0) out[u] = xfinal(all, total, load_tail(tail, tail_len));
}

// ---- Whole-unit digests, one hashing wave fed by four ----
//
// A unit's digest is four serial chains, so a launch of few units lasts as long as its longest chain. What a round costs
// is everything the chain's wave issues: here it is only the chain. With b = rotl(acc + w P2, 31), the accumulator is
// b P1 and the next round is b' = rotl(b P1 + w' P2, 31): one v_mad_u64_u32 (the product's low half, w' P2 added on the
// way), two v_mul_lo_u32, an add and two funnel shifts: 25 cycles measured for one wave, 30 with its LDS reads (61 with
// the word's own product in the same wave). One 9 MiB unit: 11.6 -> 3.62 ms; 128 of them: 15.8 -> 3.66 ms. The products
// w P2 come from four other waves of the workgroup: they read the units' bytes in 16-byte pieces (whole lines), multiply,
// and lay each chain's products next to each other in LDS, so that the hashing wave takes two rounds with one ds_read_b128.
//
// A workgroup hashes kG units (4 kG lanes of its first wave); kG is a power of two, 512 / kG stripes of each unit make a
// chunk (16 KiB), and three chunk buffers go round: while chunk k is hashed, chunk k+1 is complete (the hashing wave
// reads its first stripes ahead) and the feeders write chunk k+2, with the loads of chunks k+3 and k+4 under way in
// their registers. One barrier per chunk. The hashing wave's higher priority keeps the feeder that shares its SIMD from
// taking its issue slots.
constexpr uint32_t kFeeders = 256;       // feeding lanes (four waves)
constexpr uint32_t kFeedStripes = 512;   // stripes of a chunk, all units of the workgroup
constexpr uint32_t kFeedLoads = kFeedStripes * 2 / kFeeders;  // 16-byte pieces per lane and chunk
constexpr uint32_t kHashAhead = 16;      // stripes the hashing wave holds in registers ahead
// A workgroup whose units have no more than this many stripes hashes them quad by quad from memory: one 64-byte unit 6.7
// us, fed 8.2; 512 units of 512 bytes 7.8 / 9.5; 12288 of 1 KiB 9.3 / 12.1. At 2 KiB feeding is even with it (7.6 / 8.5,
// after other reads 9.8 / 9.4).
constexpr uint32_t kDirect = 32;

typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
typedef u64x2 u64x2_a8 __attribute__((aligned(8)));
typedef __attribute__((address_space(1))) const u64x2_a8 gpiece_t;

// A unit's stripes: stripe s lies at base[e] + 32 s for the first extent e with s < end[e].
struct UnitStripes {
  uintptr_t base[TSA_MAX_EXTENTS];
  uint64_t end[TSA_MAX_EXTENTS];
  uint64_t bytes;
  const unsigned char* tail;  // the bytes after the last stripe
  uint32_t tail_len;
};

// kHashAhead rounds on the products r, from the state b to the state b (see above). Written out because its speed hangs
// on where the instructions lie: every one is 8 bytes long, and a lone wave issues one every 4 cycles as long as they
// start 8-byte aligned (25 cycles a round; 31 when they straddle, as they do behind the compiler's 4-byte waits). The
// reads of the next products stand between two such runs and cost about 5 cycles a round; spread over the rounds they
// cost 10, and with fewer than 33 lanes active the rounds themselves are slower (31), so all lanes take part.
#define TSA_ROUND(P)                                   \
  "v_mad_u64_u32 v[12:13], vcc, v10, %[lo], %[" P "]\n" \
  "v_mul_lo_u32 v14, v10, %[hi]\n"                     \
  "v_mul_lo_u32 v15, v11, %[lo]\n"                     \
  "v_add3_u32 v13, v15, v13, v14\n"                    \
  "v_alignbit_b32 v11, v13, v12, 1\n"                  \
  "v_alignbit_b32 v10, v12, v13, 1\n"
__device__ __forceinline__ uint64_t hash_ahead(uint64_t b, const u64x2* r) {
  uint64_t v;
  asm volatile(
      ".p2align 3\n"  //
      TSA_ROUND("p0") TSA_ROUND("p1") TSA_ROUND("p2") TSA_ROUND("p3")      //
      TSA_ROUND("p4") TSA_ROUND("p5") TSA_ROUND("p6") TSA_ROUND("p7")      //
      TSA_ROUND("p8") TSA_ROUND("p9") TSA_ROUND("p10") TSA_ROUND("p11")    //
      TSA_ROUND("p12") TSA_ROUND("p13") TSA_ROUND("p14") TSA_ROUND("p15")  //
      : "={v[10:11]}"(v)
      : "0"(b), [lo] "s"(uint32_t(P1)), [hi] "s"(uint32_t(P1 >> 32)),  //
        [p0] "v"(r[0].x), [p1] "v"(r[0].y), [p2] "v"(r[1].x), [p3] "v"(r[1].y), [p4] "v"(r[2].x), [p5] "v"(r[2].y),
        [p6] "v"(r[3].x), [p7] "v"(r[3].y), [p8] "v"(r[4].x), [p9] "v"(r[4].y), [p10] "v"(r[5].x), [p11] "v"(r[5].y),
        [p12] "v"(r[6].x), [p13] "v"(r[6].y), [p14] "v"(r[7].x), [p15] "v"(r[7].y)
      : "vcc", "v12", "v13", "v14", "v15");
  return v;
}
#undef TSA_ROUND

template <uint32_t kG>
__global__ __launch_bounds__(64 + kFeeders) void digest_fed_kernel(const TsaUnit* __restrict__ units, uint32_t n,
                                                                   uint64_t* __restrict__ out) {
  constexpr uint32_t kC = kFeedStripes / kG;         // stripes of one unit in a chunk
  constexpr uint32_t kRow = kC * 8 + 16;             // bytes of a chain's row (the pad spreads the rows over the banks)
  constexpr uint32_t kBuf = 4 * kG * kRow;
  static_assert(kC % (2 * kHashAhead) == 0, "whole register blocks per chunk");
  __shared__ __attribute__((aligned(16))) unsigned char lds[3 * kBuf];
  __shared__ UnitStripes table[kG];
  const uint32_t tid = threadIdx.x;
  const bool feeds = tid >= 64;
  const uint32_t mine = feeds ? (tid - 64) / (kFeeders / kG) : (tid & (4 * kG - 1)) >> 2;
  const uint32_t u = blockIdx.x * kG + mine;
  if (tid < kG) {
    const uint32_t v = blockIdx.x * kG + tid;
    const TsaUnit un = units[v < n ? v : n - 1];  // (whole: one memory latency)
    const uint32_t ext = v < n ? un.n_ext : 0;
    uint64_t at = 0, sum = 0;
    const unsigned char* tail = nullptr;
    uint32_t tail_len = 0;
#pragma unroll
    for (uint32_t e = 0; e < TSA_MAX_EXTENTS; ++e) {
      const uint64_t bytes = e < ext ? un.ext[e].bytes : 0;
      table[tid].base[e] = (e < ext ? reinterpret_cast<uintptr_t>(un.ext[e].ptr) : 0) - 32 * at;
      at += bytes / 32;
      table[tid].end[e] = at;
      sum += bytes;
      if (e < ext) {
        tail = static_cast<const unsigned char*>(un.ext[e].ptr) + bytes / 32 * 32;
        tail_len = uint32_t(bytes % 32);
      }
    }
    table[tid].bytes = sum;
    table[tid].tail = tail;
    table[tid].tail_len = tail_len;
  }
  __syncthreads();
  const UnitStripes& us = table[mine];
  const uint64_t total = us.end[TSA_MAX_EXTENTS - 1];
  uint64_t most = 0;
#pragma unroll
  for (uint32_t i = 0; i < kG; ++i) {
    const uint64_t t = table[i].end[TSA_MAX_EXTENTS - 1];
    most = t > most ? t : most;
  }
  const uint64_t chunks = __builtin_amdgcn_readfirstlane(uint32_t((most + kC - 1) / kC >> 32)) * (1ull << 32) +
                          __builtin_amdgcn_readfirstlane(uint32_t((most + kC - 1) / kC));

  if (feeds) {
    if (most <= kDirect) return;
    constexpr uint32_t kLanes = kFeeders / kG;  // of one unit: lane l moves half l & 1 of stripes l / 2 + j kLanes / 2
    const uint32_t l = (tid - 64) % kLanes;
    unsigned char* row = lds + (4 * mine + (l & 1u) * 2) * kRow + (l >> 1) * 8;
    uintptr_t base = us.base[0];
    uint64_t end = us.end[0];
    auto load = [&](uint64_t c, u64x2* r) {
      const uint64_t lo = c * kC;
      if (lo >= end && lo < total)
        for (uint32_t e = 1; e < TSA_MAX_EXTENTS && lo >= end; ++e) {
          base = us.base[e];
          end = us.end[e];
        }
      if (__all(lo + kC <= end || lo >= total)) {  // whole chunks of one extent; a unit that has ended reads its entry
        const bool ended = lo >= total;
        const uintptr_t p = ended ? reinterpret_cast<uintptr_t>(units) : base + 32 * (lo + (l >> 1)) + (l & 1u) * 16;
        const uint32_t step = ended ? 0 : kLanes * 16;
#pragma unroll
        for (uint32_t j = 0; j < kFeedLoads; ++j) r[j] = *reinterpret_cast<gpiece_t*>(p + j * step);
      } else {
#pragma unroll
        for (uint32_t j = 0; j < kFeedLoads; ++j) {
          const uint64_t s = lo + j * (kLanes / 2) + (l >> 1);
          uint32_t e = 0;
          while (e + 1 < TSA_MAX_EXTENTS && s >= us.end[e]) ++e;
          r[j] = u64x2{0, 0};
          if (s < total) r[j] = *reinterpret_cast<gpiece_t*>(us.base[e] + 32 * s + (l & 1u) * 16);
        }
      }
    };
    auto store = [&](uint32_t b, const u64x2* r) {
#pragma unroll
      for (uint32_t j = 0; j < kFeedLoads; ++j) {
        unsigned char* d = row + b * kBuf + j * (kLanes / 2) * 8;
        *reinterpret_cast<uint64_t*>(d) = r[j].x * P2;
        *reinterpret_cast<uint64_t*>(d + kRow) = r[j].y * P2;
      }
    };
    u64x2 r0[kFeedLoads], r1[kFeedLoads];
    load(0, r0);
    load(1, r1);
    store(0, r0);
    load(2, r0);
    store(1, r1);
    load(3, r1);
    __syncthreads();
    uint32_t b = 2;
    for (uint64_t k = 0; k < chunks; k += 2) {
      store(b, r0);
      load(k + 4, r0);
      __syncthreads();
      b = b == 2 ? 0 : b + 1;
      if (k + 1 == chunks) break;
      store(b, r1);
      load(k + 5, r1);
      __syncthreads();
      b = b == 2 ? 0 : b + 1;
    }
    return;
  }

  const uint32_t q = tid & 3u;
  const bool ends = tid < 4 * kG && q == 0 && u < n;
  Tail tail;  // (read ahead of the chains: at the end it would be one more memory latency)
  if (ends) tail = load_tail(us.tail, us.tail_len);
  if (most <= kDirect) {  // (the feeders have ended)
    uint64_t acc[4];
    init_acc(acc);
    uint64_t v = q == 0 ? acc[0] : q == 1 ? acc[1] : q == 2 ? acc[2] : acc[3], at = 0;
    for (uint32_t e = 0; e < TSA_MAX_EXTENTS && at < total; ++e) {
      v = chain(v, reinterpret_cast<const unsigned char*>(us.base[e] + 32 * at), us.end[e] - at, q);
      at = us.end[e];
    }
    uint64_t all[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) all[k] = __shfl(v, int((tid & ~3u) + k), 64);
    if (ends) out[u] = xfinal(all, us.bytes, tail);
    return;
  }
  __builtin_amdgcn_s_setprio(3);
  const unsigned char* row = lds + (4 * mine + q) * kRow;
  uint64_t acc[4];
  init_acc(acc);
  uint64_t b = (q == 0 ? acc[0] : q == 1 ? acc[1] : q == 2 ? acc[2] : acc[3]) * P1inv;
  auto fetch = [](const unsigned char* from, u64x2* r) {
#pragma unroll
    for (uint32_t j = 0; j < kHashAhead / 2; ++j) r[j] = *reinterpret_cast<const u64x2*>(from + j * 16);
  };
  __syncthreads();
  u64x2 a0[kHashAhead / 2], a1[kHashAhead / 2];
  uint32_t buf = 0;
  fetch(row, a0);
  for (uint64_t k = 0; k < chunks; ++k) {
    const uint32_t next = buf == 2 ? 0 : buf + 1;
    const uint64_t done = k * kC;
    const uint32_t left = total <= done ? 0u : total - done < kC ? uint32_t(total - done) : kC;
    if (__all(left == 0 || left == kC)) {
      uint64_t v = b;
#pragma unroll 1
      for (uint32_t s = 0; s < kC; s += 2 * kHashAhead) {
        const bool turn = s + 2 * kHashAhead == kC;
        const unsigned char* p = row + buf * kBuf + s * 8;
        fetch(p + kHashAhead * 8, a1);
        v = hash_ahead(v, a0);
        fetch(turn ? row + next * kBuf : p + kHashAhead * 16, a0);
        v = hash_ahead(v, a1);
      }
      b = left ? v : b;
    } else {  // units that end inside this chunk: blocks that all lanes hash whole or not at all, then single stripes
#pragma unroll 1
      for (uint32_t s = 0; s < kC && __any(s < left); s += kHashAhead) {
        if (__all(left <= s || left >= s + kHashAhead)) {
          fetch(row + buf * kBuf + s * 8, a0);
          const uint64_t v = hash_ahead(b, a0);
          b = s < left ? v : b;
        } else {
#pragma unroll 1
          for (uint32_t t = s; t < s + kHashAhead; ++t) {
            const uint64_t v = bround(b, *reinterpret_cast<const uint64_t*>(row + buf * kBuf + t * 8));
            b = t < left ? v : b;
          }
        }
      }
      fetch(row + next * kBuf, a0);
    }
    buf = next;
    __syncthreads();
  }
  const uint64_t v = b * P1;
  uint64_t all[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) all[k] = __shfl(v, int((tid & ~3u) + k), 64);
  if (ends) out[u] = xfinal(all, us.bytes, tail);
}

// ---- The LDS-streamed check ----
//
// The chain loop above reads 8 bytes per lane at a 32-byte stride: every load instruction of a wave touches 16 lines
// (one per quad) and relies on the CU cache to keep each line for the next three. Here every wave streams its 16
// segments through LDS instead, with direct-to-LDS 16-byte loads (global_load_lds_dwordx4): 64 lanes fill 1 KiB of
// LDS per instruction, eight whole 128-byte lines. The quads then run their chains from LDS. Only for waves whose
// segments are 16-byte aligned: pieces that straddle two lines' halves made 34 MB of 8-byte aligned units 12.1 us, the
// chain loop 10.7.
//
// Per wave: a chunk is 256 bytes (8 stripes) of each of its 16 segments, 4 KiB, four loads: load k carries segments
// 4k..4k+3, lanes 16i..16i+15 the 16 pieces of segment 4k+i. A segment's stripes are rotated by (its quad index mod 8)
// inside its 256 bytes, so that the wave's ds_read_b64 of one stripe of all 16 segments spreads over the LDS banks.
// Before the chunks goes one load of every quad's checkpoint and the one after it (64 contiguous bytes): read where it
// is used, the checkpoint held every chunk's loads back, and the next one cost a memory latency at the end.
// The loads are inline assembly, so the compiler neither waits for them nor knows them; each chunk waits for its own
// loads with an explicit vmcnt (loads complete in order, and a load or store of the compiler's among them only makes
// the wait longer). Lanes whose piece lies past their segment's stripes load an earlier piece again (never out of
// bounds), and every wave issues the same number of loads, which the vmcnt counts rely on. A chunk that every segment has
// whole or not at all is hashed without a select per round: waves at the end of a part are as fast as the others (with
// both costs in them they were the launch's last: 8 MB in 5.5 us instead of 6.3).
//
// What bounds it: reading, from about 50 MB on (336 MiB in 56.1 us on changing buffers, 6.4 TB/s); below, one launch and
// four or five memory latencies (192 KiB 5.0-5.2 us, of which a launch of nothing takes 3.7).
template <uint32_t kD>  // per wave: kD chunk buffers, and 64 bytes of checkpoints per quad behind them
constexpr uint32_t wave_lds_bytes() {
  return kD * 4096 + 64 * 16;
}

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) u32x4 gu32x4_t;

// M0 (the LDS destination) is restored for the compiler; s_nop: an M0 write before a load to LDS.
__device__ __forceinline__ void lds_load16(const unsigned char* g, uint32_t lds_addr) {
  uint32_t save;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, off nt\n\t"
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0"
      : "=&s"(save)
      : "v"(g), "s"(lds_addr)
      : "memory");
}
// A chunk: piece k of the lane at g[k] + kAt to lds_addr + 1024 k (the instruction's offset moves both addresses).
template <uint32_t kAt = 0>
__device__ __forceinline__ void lds_load_chunk(const unsigned char* const g[4], uint32_t lds_addr) {
  uint32_t save;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %5\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, off offset:%6 nt\n\t"
      "s_add_u32 m0, m0, 0x400\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %2, off offset:%6 nt\n\t"
      "s_add_u32 m0, m0, 0x400\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %3, off offset:%6 nt\n\t"
      "s_add_u32 m0, m0, 0x400\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %4, off offset:%6 nt\n\t"
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0"
      : "=&s"(save)
      : "v"(g[0]), "v"(g[1]), "v"(g[2]), "v"(g[3]), "s"(lds_addr - kAt), "n"(kAt)
      : "memory", "scc");
}

template <uint32_t kD, uint32_t kC = 0>
__device__ __forceinline__ void issue_all(const unsigned char* const g[4], uint32_t lds_off) {
  if constexpr (kC < kD) {
    lds_load_chunk<kC * 256>(g, lds_off + kC * 4096);
    issue_all<kD, kC + 1>(g, lds_off);
  }
}

template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Chunk by chunk, each when it has landed (the later ones' loads may still be in flight).
template <uint32_t kD, uint32_t kC = 0, class F>
__device__ __forceinline__ void drain(F&& hash) {
  if constexpr (kC < kD) {
    wait_loads<4 * (kD - 1 - kC)>();
    hash(kC);
    drain<kD, kC + 1>(hash);
  }
}

// One wave's 16 segments (quad j's lanes 4 j + q hold segment j): where it is read and (kCopy) written, its stripes (0
// hashes nothing and reads 16 bytes), its checkpoint (32 bytes, 64 when it is not the unit's last). Out: the
// accumulator after the segment, and the next checkpoint's. All 64 lanes call it, at least one of them live; the others
// go along with the first live segment and their results mean nothing. lds: the wave's wave_lds_bytes<kD>().
//
// kD 2 or 4: as many chunk buffers go round, chunk c + kD loaded when chunk c has been hashed (its LDS reads complete:
// lgkmcnt 0). kD 8: segments of up to 2 KiB, all their chunks in flight at once (not for the copy, whose stores the waits
// would wait for).
template <uint32_t kD>
__device__ __forceinline__ unsigned char* wave_lds(unsigned char* lds) {  // the wave's part of its workgroup's
  return lds + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * wave_lds_bytes<kD>();
}
template <uint32_t kD, bool kCopy>
__device__ __forceinline__ uint64_t lds_check(bool live, const unsigned char* from, unsigned char* to,
                                              uint32_t stripes, const uint64_t* state, bool last,
                                              unsigned char* lds, uint64_t* next) {
  const uint32_t lds_off = uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)(lds)));
  const uint32_t lane = threadIdx.x & 63u, q = lane & 3u, j = lane >> 2;
  const uint32_t i = lane >> 4, m = lane & 15u;
  const int first = __ffsll(static_cast<long long>(__ballot(live))) - 1;
  auto from_first = [&](uint64_t x, uint64_t mine) {
    const uint64_t f = __shfl(static_cast<unsigned long long>(x), first, 64);
    return live ? mine : f;
  };
  from = reinterpret_cast<const unsigned char*>(from_first(reinterpret_cast<uintptr_t>(from), reinterpret_cast<uintptr_t>(from)));
  state = reinterpret_cast<const uint64_t*>(from_first(reinterpret_cast<uintptr_t>(state), reinterpret_cast<uintptr_t>(state)));
  last = last || !live;
  constexpr bool kAll = kD == 8;
  static_assert(!kAll || !kCopy, "");
  uint32_t chunks = kD;
  if (!kAll) {  // as many rounds of the buffers as the wave's longest segment has
    uint32_t most = stripes;
#pragma unroll
    for (uint32_t d = 4; d < 64; d *= 2) most = max(most, uint32_t(__shfl_xor(int(most), int(d), 64)));
    chunks = max(kD, __builtin_amdgcn_readfirstlane((most + 8 * kD - 1) / (8 * kD) * kD));
  }
  const bool whole = __all(!live || stripes == 8 * chunks);
  lds_load16(reinterpret_cast<const unsigned char*>(state) + (last ? q & 1u : q) * 16, lds_off + kD * 4096);
  // The lane's piece of load k (of segment 4k + i: quad 4k + i's lane 0 holds its source) in chunk 0, and how far its
  // segment has later ones: past that the lane loads the last one again, or (no stripe of its own) the segment's first.
  const unsigned char* src[4];
  unsigned char* dst[4];
  uint32_t n[4], g0[4], lim[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int owner = int((4 * k + i) * 4);
    g0[k] = ((m >> 1) - ((4 * k + i) & 7u)) & 7u;  // its stripe in chunk 0
    n[k] = uint32_t(__shfl(int(stripes), owner, 64));
    const uint32_t at = g0[k] * 32 + (m & 1u) * 16;
    src[k] = reinterpret_cast<const unsigned char*>(
                 __shfl(static_cast<unsigned long long>(reinterpret_cast<uintptr_t>(from)), owner, 64)) +
             (whole || g0[k] < n[k] ? at : 0);
    lim[k] = g0[k] < n[k] ? (n[k] - 1 - g0[k]) / 8 * 256 : 0;
    if (kCopy)
      dst[k] = reinterpret_cast<unsigned char*>(
                   __shfl(static_cast<unsigned long long>(reinterpret_cast<uintptr_t>(to)), owner, 64)) +
               at;
  }
  auto issue = [&](uint32_t c, uint32_t buf) {
    if (whole) {
      lds_load_chunk(src, lds_off + buf * 4096);
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) src[k] += 256;
    } else {
      const unsigned char* g[4];
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) g[k] = src[k] + min(256 * c, lim[k]);
      lds_load_chunk(g, lds_off + buf * 4096);
    }
  };
  auto put = [](unsigned char* p, u32x4 x) {  // (a global store: a generic one would also count on the LDS counter)
    *reinterpret_cast<gu32x4_t*>(reinterpret_cast<uintptr_t>(p)) = x;
  };
  const bool full = kCopy && __all(live && stripes == 8 * chunks);
  auto store = [&](uint32_t c, uint32_t buf) {  // the lane's own four pieces, as they landed in LDS
    u32x4 x[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) x[k] = *reinterpret_cast<const u32x4*>(lds + buf * 4096 + k * 1024 + lane * 16);
    if (full) {
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k) put(dst[k] + c * 256, x[k]);
    } else {
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k)
        if (g0[k] + 8 * c < n[k]) put(dst[k] + c * 256, x[k]);
    }
  };
  const uint32_t rot = j & 7u;
  const unsigned char* rd = lds + (j >> 2) * 1024 + (j & 3u) * 256 + q * 8;
  uint64_t b = 0;
  auto hash = [&](uint32_t c, uint32_t buf) {
    uint64_t x[8];
#pragma unroll
    for (uint32_t t = 0; t < 8; ++t)
      x[t] = *reinterpret_cast<const uint64_t*>(rd + ((t + rot) & 7u) * 32 + buf * 4096);
    const bool in = 8 * c < stripes;
    if (whole || __all(!in || stripes >= 8 * c + 8)) {  // every segment has all of the chunk or none of it
      uint64_t r = b;
#pragma unroll
      for (uint32_t t = 0; t < 8; ++t) r = bround(r, x[t] * P2);
      b = whole || in ? r : b;
    } else {
#pragma unroll
      for (uint32_t t = 0; t < 8; ++t) {
        uint64_t r = bround(b, x[t] * P2);
        asm volatile("" : "+v"(r));  // (a select, not a branch around each round)
        b = 8 * c + t < stripes ? r : b;
      }
    }
  };
  if (kAll && whole) {
    issue_all<kD>(src, lds_off);
  } else {
#pragma unroll (kAll ? 1 : kD)
    for (uint32_t c = 0; c < kD; ++c) issue(c, c);
  }
  wait_loads<4 * kD>();
  const uint64_t* st = reinterpret_cast<const uint64_t*>(lds + kD * 4096 + j * 64);
  b = st[q] * P1inv;
  *next = st[4 + q];
  for (uint32_t c = 0; !kAll && c + kD < chunks; c += kD) {
#pragma unroll
    for (uint32_t i = 0; i < kD; ++i) {
      wait_loads<4 * (kD - 1)>();
      if (kCopy) store(c + i, i);
      hash(c + i, i);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      issue(c + i + kD, i);
    }
  }
  const uint32_t c = chunks - kD;
  drain<kD>([&](uint32_t i) {
    if (kCopy) store(c + i, i);
    hash(c + i, i);
  });
  return b * P1;
}

// The chain-loop kernels (dg_verify_kernel, dg_scatter_verify_kernel) are held to 8 waves per SIMD (at most 64
// VGPRs): unbounded, the compiler spends registers on scheduling (83-86 VGPRs, 5 waves per SIMD) and the kernel has
// 5/8 of the loads in flight it could; bounded it needs 52-58 with no spill, and one 336 MiB unit's check (3 parts,
// 2 KiB segments, timed alone in a fresh process) ran 67 -> 62 us. The LDS-streamed kernels keep their loads in LDS,
// not in registers.
#define TSA_VERIFY_BOUNDS __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8, 8)))

// A segment of a unit given by its extents: where it lies and what it must lead to.
struct HostSeg {
  const unsigned char* from = nullptr;
  const uint64_t* state = nullptr;
  uint64_t digest = 0, total = 0, stripes = 0;
  uint32_t ui = 0;
  bool live = false, last = false;
  Tail tail;
};
// shift: seg_bytes = 1 << shift, or 64 when it is no power of two (a 64-bit division is about 100 instructions).
__device__ __forceinline__ HostSeg host_segment(const TsaVerifyUnit& un, uint32_t ui, uint64_t s, uint64_t seg_bytes,
                                                uint32_t shift, uint32_t* fail, uint32_t q) {
  HostSeg g;
  g.ui = ui;
  const uint64_t local = s - un.seg_first;  // the unit's segment index (its checkpoint index)
  const uint32_t n_ext = un.n_ext;
  uint64_t k = local;
  bool found = false;
  const unsigned char* tail = nullptr;
  uint32_t tail_len = 0;
#pragma unroll
  for (uint32_t e = 0; e < TSA_MAX_EXTENTS; ++e) {
    if (e < n_ext && !found) {
      const uint64_t b = un.ext[e].bytes;
      const bool last_ext = e + 1 == n_ext;
      const uint64_t span = last_ext ? b / 32 * 32 : b;
      uint64_t nseg = shift < 64 ? (span + seg_bytes - 1) >> shift : (span + seg_bytes - 1) / seg_bytes;
      if (last_ext && nseg == 0) nseg = 1;
      if (k < nseg) {
        found = true;
        const unsigned char* p = static_cast<const unsigned char*>(un.ext[e].ptr);
        const uint64_t off = k * seg_bytes;
        const uint64_t end = off + seg_bytes < span ? off + seg_bytes : span;
        g.stripes = (end - off) / 32;
        g.from = p + off;
        g.last = last_ext && k + 1 == nseg;
        tail = p + span;
        tail_len = uint32_t(b - span);
      }
      k -= nseg;
    }
  }
  if (!found) {  // the launch's prefix sums disagree with the extents: reported, nothing read or checked
    if (q == 0) atomicOr(fail + ui, 2u);
    return g;
  }
  if (g.last && q == 0) g.tail = load_tail(tail, tail_len);
  g.live = true;
  g.state = un.states + 4 * local;
  g.digest = un.digest;
  g.total = un.total;
  return g;
}
// One (unit, segment) per quad. seg_first is the prefix sum of segments over the launch's units (ascending). kD: as for
// lds_check, in waves whose segments all start at a multiple of `mask` + 1; any other wave, and every one with kD 0, runs the
// chain loop from memory.
template <uint32_t kD>
__device__ __forceinline__ void verify_body(const TsaVerifyUnit* __restrict__ units, uint32_t n_units, uint64_t n_segments,
                                            uint64_t seg_bytes, uint32_t shift, uint64_t mask,
                                            uint32_t* __restrict__ fail) {
  const uint64_t s0 = (uint64_t(blockIdx.x) * 256 + __builtin_amdgcn_readfirstlane(threadIdx.x & ~63u)) >> 2;
  if (s0 >= n_segments) return;  // (the whole wave)
  const uint32_t q = threadIdx.x & 3u;
  const uint64_t s = s0 + ((threadIdx.x & 63u) >> 2);
  const uint64_t end = n_segments - s0 < 16 ? n_segments : s0 + 16;
  uint32_t ui = last_at_most(n_units, s0, [&](uint32_t i) { return units[i].seg_first; });
  HostSeg g;
  const uint64_t after = ui + 1 < n_units ? units[ui + 1].seg_first : ~0ull;
  TsaVerifyUnit un = units[ui];  // (whole and at once: with scalar loads, one memory latency)
  const bool one = after >= end;  // the wave's segments are one unit's
  if (!one) {
    // The quad's unit: the next 16 units' first segments in one read, counted up to the quad's own (unit by unit, 200
    // units of one segment each were 16 reads one behind the other: 8.6 us, 7.2 like this).
    const uint64_t base = ui + 1;
    for (uint64_t w = base, seen = after; seen < end; w += 16) {
      const uint64_t i = w + (threadIdx.x & 15u);
      const uint64_t f = i < n_units ? units[i].seg_first : ~0ull;
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        seen = uint64_t(uint32_t(__builtin_amdgcn_readlane(int(f >> 32), k))) << 32 |
               uint32_t(__builtin_amdgcn_readlane(int(f), k));
        ui += seen <= s;
      }
    }
  }
  if constexpr (kD != 0) {  // (one copy of the code for both: a first launch waits for it)
    if (!one) un = units[ui];
    if (s < end) g = host_segment(un, ui, s, seg_bytes, shift, fail, q);
  } else if (one) {  // (with the entry in scalar registers: 187 MB in 512-byte segments 31.7 us, 33.4 with it in vector ones)
    if (s < end) g = host_segment(un, ui, s, seg_bytes, shift, fail, q);
  } else if (s < end) {
    const TsaVerifyUnit mine = units[ui];
    g = host_segment(mine, ui, s, seg_bytes, shift, fail, q);
  }
  if (__ballot(g.live) == 0) return;
  uint64_t v = 0, next = 0;
  bool streamed = false;
  if constexpr (kD != 0) {
    streamed = __all(!g.live || (reinterpret_cast<uintptr_t>(g.from) & mask) == 0);
    __shared__ __attribute__((aligned(16))) unsigned char lds[4 * wave_lds_bytes<kD>()];
    if (streamed)
      v = lds_check<kD, false>(
          g.live, g.stripes ? g.from : reinterpret_cast<const unsigned char*>(g.state), nullptr, uint32_t(g.stripes), g.state,
          g.last, wave_lds<kD>(lds), &next);
  }
  if (!streamed && g.live) {
    // (global loads: with a generic one under way the compiler waits for all of a block's words before its first round)
    gword_t* const state = reinterpret_cast<gword_t*>(reinterpret_cast<uintptr_t>(g.state));
    next = g.last ? 0 : state[4 + q];
    v = chain(state[q], g.from, g.stripes, q);
  }
  uint64_t all[4];
  const uint32_t base = threadIdx.x & ~3u;
#pragma unroll
  for (int k = 0; k < 4; ++k) all[k] = __shfl(v, int(base + k), 64);
  if (!g.live) return;
  if (!g.last) {
    if (v != next) atomicOr(fail + g.ui, 1u);
  } else if (q == 0) {
    if (xfinal(all, g.total, g.tail) != g.digest) atomicOr(fail + g.ui, 1u);
  }
}
template <uint32_t kD>
__global__ __launch_bounds__(256) void verify_lds_kernel(const TsaVerifyUnit* __restrict__ units, uint32_t n_units,
                                                         uint64_t n_segments, uint64_t seg_bytes, uint32_t shift,
                                                         uint64_t mask, uint32_t* __restrict__ fail) {
  verify_body<kD>(units, n_units, n_segments, seg_bytes, shift, mask, fail);
}
__global__ __launch_bounds__(256) void verify_kernel(const TsaVerifyUnit* __restrict__ units, uint32_t n_units,
                                                     uint64_t n_segments, uint64_t seg_bytes, uint32_t shift,
                                                     uint64_t mask, uint32_t* __restrict__ fail) {
  verify_body<0>(units, n_units, n_segments, seg_bytes, shift, mask, fail);
}

// Device-gated verify: one quad per segment of a unit, the launch's units (all of the arena's part shape) along the grid's
// y or packed, each from a wave of its own on, so that a wave has one unit: its key and slot are scalar, and no segment
// index is divided. kCopy (the staged units' fused scatter): unit u's bytes are read from
// src + u x unit_bytes, where its parts lie back to back, and written to their arena slot as they are hashed; the last
// segment's lane 0 also moves the unit's tail.
struct DgSeg {
  const uint64_t* state = nullptr;
  uint64_t digest = 0;
  uint32_t stripes = 0;
  bool live = false, last = false;
  const unsigned char* from = nullptr;  // the segment's first byte (where it is read)
  unsigned char* to = nullptr;          // (kCopy) where it is written
  const unsigned char* tail = nullptr;  // (last) the bytes after the last stripe, and where they are written
  unsigned char* tail_to = nullptr;
  uint32_t tail_len = 0;
};

// The wave's unit and its first segment there: kPack, each unit's unit_waves waves right behind the last one's; else a row of
// the grid for each unit.
struct DgWave {
  uint32_t u = 0;
  uint64_t first = 0;
};
template <bool kPack>
__device__ __forceinline__ DgWave dg_wave(uint32_t unit_waves) {
  DgWave w;
  uint32_t k = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  w.u = blockIdx.y;
  if (kPack) {
    w.u = __builtin_amdgcn_readfirstlane(k / unit_waves);
    k -= w.u * unit_waves;
  }
  w.first = uint64_t(k) * 16;
  return w;
}

// (The part's fields are carried along the walk over the parts with constant indices, which keeps every read of the
// launch's arguments a scalar load.)
template <bool kCopy>
__device__ __forceinline__ DgSeg dg_segment(const DgVerifyLaunch& a, const unsigned char* src, uint32_t u, uint64_t local) {
  DgSeg g;
  const uint64_t key = a.keys[u];
  const int32_t slot = a.slots[u];
  g.live = local < a.unit_segs;
  if (!g.live) return g;
  g.state = a.ckpt + (key * a.unit_segs + local) * 4;
  g.digest = a.digests[key];
  uint64_t k = local;
  uint32_t p = 0;
  uint64_t src_off = uint64_t(u) * a.unit_bytes;  // (kCopy) the part's first byte in src
  uint64_t pbytes = a.part_bytes[0], psegs = a.part_segs[0];
  const unsigned char* parena = a.arena[0];
#pragma unroll
  for (uint32_t i = 0; i + 1 < 4; ++i) {
    if (p == i && i + 1 < a.n_parts && k >= a.part_segs[i]) {
      k -= a.part_segs[i];
      src_off += a.part_bytes[i];
      p = i + 1;
      pbytes = a.part_bytes[i + 1];
      psegs = a.part_segs[i + 1];
      parena = a.arena[i + 1];
    }
  }
  const bool last_part = p + 1 == a.n_parts;
  const uint64_t span = last_part ? pbytes / 32 * 32 : pbytes;
  const uint64_t off = k * a.seg_bytes;
  const uint64_t end = off + a.seg_bytes < span ? off + a.seg_bytes : span;
  unsigned char* base = const_cast<unsigned char*>(parena) + uint64_t(slot) * pbytes;
  const unsigned char* from = kCopy ? src + src_off : base;
  g.last = last_part && k + 1 == psegs;
  g.tail = from + span;
  g.tail_to = base + span;
  g.tail_len = uint32_t(pbytes - span);
  g.stripes = end > off ? uint32_t((end - off) / 32) : 0;
  g.from = from + off;
  g.to = base + off;
  return g;
}

// The segment's check (the next checkpoint, or for the unit's last segment the digest) and the gate.
template <bool kCopy>
__device__ __forceinline__ void dg_finish(const DgVerifyLaunch& a, uint32_t u, const DgSeg& g, const Tail& tail, uint64_t v,
                                          uint64_t next, uint32_t q) {
  uint64_t all[4];
  const uint32_t base4 = threadIdx.x & ~3u;
#pragma unroll
  for (int k = 0; k < 4; ++k) all[k] = __shfl(v, int(base4 + k), 64);
  bool bad = false;
  if (g.live) {
    if (!g.last) {
      bad = v != next;
    } else if (q == 0) {
      bad = xfinal(all, a.unit_bytes, tail) != g.digest;
      if (kCopy) store_tail(g.tail_to, tail);
    }
  }
  if (bad) {
    atomicOr(a.fail + u, 1u);
    if (a.abort) {  // the gate: the token fails before the layer's ready word is written
      if (atomicCAS(a.err_code, 0u, a.err) == 0u) atomicExch(a.err_aux, a.aux);
      atomicExch(a.abort, 1u);
    }
  }
}

// Publication after a check, launched behind it on its stream (so it starts once every workgroup of the check has
// ended and its writes, a failing one's abort among them, are visible): the landed units' slot entries, then the
// layer's ready word. Counting the check's workgroups in the check itself instead (an agent-scope atomic per
// workgroup, the last one publishing) cost 8 us per 336 MiB check on this chip: each atomic waits in the memory
// queues behind the check's own reads and holds its workgroup's slot.
__global__ __launch_bounds__(64) void dg_publish_kernel(const DgVerifyLaunch a) {
  if (threadIdx.x != 0) return;
  if (a.slot_of)
    for (uint32_t i = 0; i < a.n; ++i)
      __hip_atomic_store(a.slot_of + a.keys[i], a.slots[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (a.ready) {
    __threadfence_system();
    __hip_atomic_store(a.ready + a.ready_g, a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

template <bool kPack, bool kCopy>
__device__ __forceinline__ void dg_chain_body(const DgVerifyLaunch& a, uint32_t unit_waves, const unsigned char* src) {
  const DgWave w = dg_wave<kPack>(unit_waves);
  if ((kPack && w.u >= a.n) || w.first >= a.unit_segs) return;  // (the whole wave)
  const uint32_t q = threadIdx.x & 3u;
  const DgSeg g = dg_segment<kCopy>(a, src, w.u, w.first + ((threadIdx.x & 63u) >> 2));
  uint64_t v = 0, next = 0;
  if (g.live) {
    next = g.last ? 0 : g.state[4 + q];
    v = chain_t<kCopy>(g.state[q], g.from, g.to, g.stripes, q);
  }
  Tail tail;
  if (g.last && q == 0) tail = load_tail(g.tail, g.tail_len);
  dg_finish<kCopy>(a, w.u, g, tail, v, next, q);
}
template <bool kPack>
__global__ TSA_VERIFY_BOUNDS void dg_verify_kernel(const DgVerifyLaunch a, uint32_t unit_waves) {
  dg_chain_body<kPack, false>(a, unit_waves, nullptr);
}
template <bool kPack>
__global__ TSA_VERIFY_BOUNDS void dg_scatter_verify_kernel(const DgVerifyLaunch a, uint32_t unit_waves,
                                                           const unsigned char* src) {
  dg_chain_body<kPack, true>(a, unit_waves, src);
}

template <uint32_t kD, bool kPack, bool kCopy>
__device__ __forceinline__ void dg_lds_body(const DgVerifyLaunch& a, uint32_t unit_waves, const unsigned char* src) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[4 * wave_lds_bytes<kD>()];
  const DgWave w = dg_wave<kPack>(unit_waves);
  if ((kPack && w.u >= a.n) || w.first >= a.unit_segs) return;  // (the whole wave)
  const uint32_t q = threadIdx.x & 3u;
  const DgSeg g = dg_segment<kCopy>(a, src, w.u, w.first + ((threadIdx.x & 63u) >> 2));
  Tail tail;  // (read ahead of the chains: at the end it would be one more memory latency)
  if (g.last && q == 0) tail = load_tail(g.tail, g.tail_len);
  uint64_t v = 0, next = 0;
  if (__all(!g.live || (reinterpret_cast<uintptr_t>(g.from) | (kCopy ? reinterpret_cast<uintptr_t>(g.to) : 0)) % 16 == 0)) {
    v = lds_check<kD, kCopy>(g.live, g.stripes ? g.from : reinterpret_cast<const unsigned char*>(g.state), g.to, g.stripes,
                                  g.state, g.last, wave_lds<kD>(lds), &next);
  } else if (g.live) {
    next = g.last ? 0 : g.state[4 + q];
    v = chain_t<kCopy>(g.state[q], g.from, g.to, g.stripes, q);
  }
  dg_finish<kCopy>(a, w.u, g, tail, v, next, q);
}
template <uint32_t kD, bool kPack>
__global__ __launch_bounds__(256) void dg_verify_lds_kernel(const DgVerifyLaunch a, uint32_t unit_waves) {
  dg_lds_body<kD, kPack, false>(a, unit_waves, nullptr);
}
template <uint32_t kD, bool kPack>
__global__ __launch_bounds__(256) void dg_scatter_verify_lds_kernel(const DgVerifyLaunch a, uint32_t unit_waves,
                                                                    const unsigned char* src) {
  dg_lds_body<kD, kPack, true>(a, unit_waves, src);
}

}  // namespace dev

// Units per workgroup: with up to 512 one each (two workgroups on every CU), then the power of two that keeps it at 512
// workgroups, so that every chain has a wave's full issue rate; 16 from 4097 units on, where three workgroups fit a CU's
// LDS and 12288 units hash at once. Beyond that the workgroups would queue, and a quad per unit has lanes enough of its
// own. Measured (us, quads / fed): 128 x 9 MiB 15847 / 3658; 512 x 1 MiB 1771 / 433; 4096 x 128 KiB 242 / 102;
// 8192 x 64 KiB 144 / 96; 16384 x 32 KiB 112 / 130; 65536 x 8 KiB 101 / 127.
int launch_digest(const TsaUnit* units_dev, uint32_t n, uint64_t* out_dev, hipStream_t stream) {
  if (n == 0) return 0;
  if (n > 12288) {
    hipLaunchKernelGGL(dev::digest_quads_kernel, dim3((n + 63) / 64), dim3(256), 0, stream, units_dev, n, out_dev);
    return int(hipGetLastError());
  }
  uint32_t g = 1;
  while (g < 16 && n > 512 * g) g *= 2;
  auto* k = g == 1   ? dev::digest_fed_kernel<1>
            : g == 2 ? dev::digest_fed_kernel<2>
            : g == 4 ? dev::digest_fed_kernel<4>
            : g == 8 ? dev::digest_fed_kernel<8>
                     : dev::digest_fed_kernel<16>;
  hipLaunchKernelGGL(k, dim3((n + g - 1) / g), dim3(64 + dev::kFeeders), 0, stream, units_dev, n, out_dev);
  return int(hipGetLastError());
}

// Whether a launch that touches `bytes` (the copy: twice its units') streams its segments: those of 2 KiB; where every part
// lies on whole cache lines, checks above 80 MB those of 1 KiB too, the copy those of 512 bytes to 4 KiB in whole chunk pairs
// (above 80 MB only 1 KiB). Streamed / chain loop, us in a loop on changing buffers:
//  * Checks: 8.6 MB in 1.5 KiB segments 5.4 / 4.5, 8.4 MB in 4 KiB ones 7.9 / 6.4, 62 MB in 512-byte ones 11.9 / 10.9 (a
//    wave's pieces lie far apart, or a wave ends after one pair); 1 KiB: 61 MB 11.5 / 10.9, 182 MB 29.6 / 31.7, but 148 MB
//    that start in the middle of lines 31.0 / 27.0 (every chunk shares its ends' lines with its neighbours).
//  * The copy: 17 MB moved in 4 KiB segments 11.4 / 13.8, in 1.5 KiB ones 7.7 / 8.0, 119 MB in 1 KiB ones 22.3 / 30.7; off
//    the lines 53 MB in 4 KiB ones 20.5 / 16.7, in 1 KiB ones 14.7 / 13.2, in 2 KiB ones 14.1 / 14.6.
//
// Two buffers a wave; four for the copy above 80 MB and for checks above it whose parts lie off the cache lines; all of a
// segment's chunks in flight for checks of units (batches) of up to 96 segments of 2 KiB. Reads go past the caches, stores
// (the copy's) through them. Measured in workgroups of four waves, us (in a loop on changing buffers / one launch after
// other reads):
//  * Four buffers, 70 KB of LDS a workgroup, two on a CU. On whole lines: 85 MB 16.0 / 19.9, two 15.5 / 19.0; 358 MB 56.9 /
//    58.8, two 56.4 / 59.5; 307 MB batch 48.8 / 53.4, two 47.9 / 51.0. Off them: 358 MB 62.6 / 65.0, two 71.4 / 73.9; 178 MB
//    32.1 / 37.7, two 35.0 / 41.8 (a batch's extents are not known here: two). The copy: 150 MB moved 28.8 / 31.6, two 30.0 /
//    32.4; 50 MB moved 11.8 / 15.0, two 12.0 / 15.0.
//  * All chunks in flight, 132 KiB of LDS a workgroup: one unit of 32 KiB 4.77 / 8.1, two buffers 5.17 / 10.0; 192 KiB 5.18 /
//    10.2, two 5.38 / 9.7; eight of them 5.51 / 9.3, two 5.79 / 9.5; a batch of 157 KB 5.44 / 10.9, two 5.71 / 11.4. But one
//    unit of 256 KiB 5.45 / 10.3, two 5.38 / 9.6; 3 MB 6.26 / 12.6, two 5.96 / 10.6: a CU then waits for its four waves'
//    chunks at once.
//  * Cached reads, faster only in the loop (staged 24.8 MB unit 10.2 us against 12.0, 51 MB unit 9.8 / 10.4): after a
//    kernel has left the L2 full of written lines, which they drive out, 19.7 us against 15.4 and 23.8 against 13.4; in
//    decode tokens 14.5 against 14.9 and (48 MiB) 13.7 against 13.1.
//  * Non-temporal stores, likewise: eight staged units (399 MB moved) 71.4 us against 78.5 in the loop, 75.2 against 65.1
//    after other reads.
constexpr uint64_t kNearBytes = 80000000;
constexpr uint64_t kFewSegs = 96;
static bool check_streams(uint64_t seg_bytes, uint64_t bytes) {
  return seg_bytes == 2048 || (seg_bytes == 1024 && bytes > kNearBytes);
}
static bool copy_streams(uint64_t seg_bytes, uint64_t bytes) {
  return bytes <= kNearBytes ? seg_bytes % 512 == 0 && seg_bytes <= 4096 : seg_bytes == 1024 || seg_bytes == 2048;
}
static uint32_t stream_align(uint64_t seg_bytes) { return seg_bytes == 2048 ? 16 : 128; }
// Whether every part of every unit of the launch lies at a multiple of `align`.
static bool aligned(const DgVerifyLaunch& a, uint32_t align) {
  for (uint32_t p = 0; p < a.n_parts; ++p) {
    if (reinterpret_cast<uintptr_t>(a.arena[p]) % align != 0) return false;
    if (a.part_bytes[p] % align == 0) continue;
    for (uint32_t u = 0; u < a.n; ++u)
      if (uint64_t(a.slots[u]) * a.part_bytes[p] % align != 0) return false;
  }
  return true;
}

// A row of whole workgroups for each unit while that is no more of them than the chip has CUs (64 units of one segment 5.8
// us, packed 6.1), else the units' waves one right behind the other: 60 units of 51 waves in rows of 13 workgroups are 780,
// so that some CUs get four, packed 765, three each (100 MB 23.1 us, packed 21.2).
constexpr uint64_t kCus = 256;
static bool dg_grid(const DgVerifyLaunch& a, dim3* grid, uint32_t* unit_waves) {
  const uint64_t own = (a.unit_segs + 15) / 16, rows = (own + 3) / 4, packed = (a.n * own + 3) / 4;
  if (a.n * rows > 0x3fffffffull) return false;
  const bool pack = a.n > 1 && a.n * rows > kCus;
  *unit_waves = pack ? uint32_t(own) : 0;
  *grid = pack ? dim3(uint32_t(packed)) : dim3(uint32_t(rows), a.n);
  return true;
}

static int launch_publish(const DgVerifyLaunch& a, hipStream_t stream) {
  if (!a.publish || (!a.slot_of && !a.ready)) return 0;
  hipLaunchKernelGGL(dev::dg_publish_kernel, dim3(1), dim3(64), 0, stream, a);
  return int(hipGetLastError());
}

// start and stop (both or neither) take the dispatch's own begin and end timestamps.
template <class K, class... A>
static int launch_timed(K* k, dim3 grid, uint32_t threads, hipStream_t stream, hipEvent_t start, hipEvent_t stop,
                        const A&... args) {
  if (start && stop)
    hipExtLaunchKernelGGL(k, grid, dim3(threads), 0, stream, start, stop, 0, args...);
  else
    hipLaunchKernelGGL(k, grid, dim3(threads), 0, stream, args...);
  return int(hipGetLastError());
}

int launch_dg_verify(const DgVerifyLaunch& a, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  if (a.n == 0 || a.unit_segs == 0) return 0;
  if (a.n > kDgVerifyMax || a.n_parts == 0 || a.n_parts > 4) return int(hipErrorInvalidValue);
  dim3 grid;
  uint32_t waves = 0;
  if (!dg_grid(a, &grid, &waves)) return int(hipErrorInvalidValue);
  // An arena that is not aligned streams wave by wave only above 80 MB in 2 KiB segments (102 MB, a third of it unaligned:
  // 16.0 us against 18.9 for the chain loop on the same buffers); else the chain loop's kernel with its 8 waves on a SIMD
  // is the better one (8.5 MB 5.2 us, wave by wave 5.8; 34 MB 7.7 / 7.9).
  const uint64_t bytes = a.n * a.unit_bytes;
  const bool stream_it = check_streams(a.seg_bytes, bytes) &&
                         (aligned(a, stream_align(a.seg_bytes)) || (a.seg_bytes == 2048 && bytes > kNearBytes));
  const bool few = a.seg_bytes == 2048 && a.unit_segs <= kFewSegs;
  static_assert(kDgVerifyMax * ((kFewSegs + 63) / 64) <= kCus, "a launch of few segments a unit is never packed");
  const bool four = stream_it && bytes > kNearBytes && !aligned(a, 128);
  auto* k = !stream_it ? (waves ? dev::dg_verify_kernel<true> : dev::dg_verify_kernel<false>)
            : few      ? dev::dg_verify_lds_kernel<8, false>
            : four     ? (waves ? dev::dg_verify_lds_kernel<4, true> : dev::dg_verify_lds_kernel<4, false>)
                       : (waves ? dev::dg_verify_lds_kernel<2, true> : dev::dg_verify_lds_kernel<2, false>);
  const int e = launch_timed(k, grid, 256, stream, start, stop, a, waves);
  return e ? e : launch_publish(a, stream);
}

int launch_dg_scatter_verify(const DgVerifyLaunch& a, const void* src, hipStream_t stream, hipEvent_t start,
                             hipEvent_t stop) {
  if (a.n == 0 || a.unit_segs == 0) return 0;
  if (a.n > kDgVerifyMax || a.n_parts == 0 || a.n_parts > 4 || !src) return int(hipErrorInvalidValue);
  dim3 grid;
  uint32_t waves = 0;
  if (!dg_grid(a, &grid, &waves)) return int(hipErrorInvalidValue);
  const uint64_t bytes = 2 * a.n * a.unit_bytes;
  bool stream_it = copy_streams(a.seg_bytes, bytes);
  if (stream_it && a.seg_bytes != 2048) {  // (2 KiB: its waves look for themselves)
    const uint32_t align = stream_align(a.seg_bytes);
    stream_it = aligned(a, align) && reinterpret_cast<uintptr_t>(src) % align == 0 && (a.n == 1 || a.unit_bytes % align == 0);
    for (uint32_t p = 0; p + 1 < a.n_parts; ++p) stream_it = stream_it && a.part_bytes[p] % align == 0;
  }
  const bool four = bytes > kNearBytes;
  auto* k = !stream_it ? (waves ? dev::dg_scatter_verify_kernel<true> : dev::dg_scatter_verify_kernel<false>)
            : four     ? (waves ? dev::dg_scatter_verify_lds_kernel<4, true> : dev::dg_scatter_verify_lds_kernel<4, false>)
                       : (waves ? dev::dg_scatter_verify_lds_kernel<2, true> : dev::dg_scatter_verify_lds_kernel<2, false>);
  const int e = launch_timed(k, grid, 256, stream, start, stop, a, waves, static_cast<const unsigned char*>(src));
  return e ? e : launch_publish(a, stream);
}

int launch_verify(const TsaVerifyUnit* units_dev, uint32_t n_units, uint64_t n_segments, uint64_t seg_bytes,
                  uint32_t* fail_dev, hipStream_t stream, hipEvent_t start, hipEvent_t stop) {
  if (n_units == 0 || n_segments == 0) return 0;
  const uint32_t threads = 256;
  const uint64_t blocks = (n_segments * 4 + threads - 1) / threads;
  if (blocks > 0x7fffffffull) return int(hipErrorInvalidValue);
  const uint32_t shift = seg_bytes & (seg_bytes - 1) ? 64 : uint32_t(__builtin_ctzll(seg_bytes));
  auto* k = !check_streams(seg_bytes, n_segments * seg_bytes) ? dev::verify_kernel
            : seg_bytes == 2048 && n_segments <= kFewSegs     ? dev::verify_lds_kernel<8>
                                                              : dev::verify_lds_kernel<2>;
  const uint64_t mask = stream_align(seg_bytes) - 1;
  return launch_timed(k, dim3(uint32_t(blocks)), threads, stream, start, stop, units_dev, n_units, n_segments, seg_bytes,
                      shift, mask, fail_dev);
}

}  // namespace tsa
