// Byte-moving kernels over HBM: the unit scatter (a staged unit's parts into their arena slots) and the synthetic
// byte generator the benchmarks and tests fill sources with.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tsa_device.hpp"
#include "wave_search.hpp"

namespace tsa {
namespace dev {

// ---- scatter ------------------------------------------------------------------------------------------------------
// The launch is a flat list of 16 KiB blocks: job j owns blocks [block_first_j, block_first_j + blocks_j), part by
// part. A workgroup of 256 lanes moves one block: 4 x 16 bytes per lane, each load and store a 128-bit access, lanes
// adjacent in memory (a wavefront covers 1 KiB per instruction). Consecutive workgroups take consecutive blocks, so a
// part streams through HBM in order. The job is found by the wave's lanes together and its entry read at once, with
// scalar loads: block by block, a chain of dependent reads ahead of every 16 KiB cost a tenth of a large launch.
//
// Reads go past the caches (each byte is read once), stores do not (the engine reads the slot next). The other ways were
// faster only in an unbroken run of launches on changing buffers: cached reads 8.9 us against 10.3 for one unit of 24.8
// MB, non-temporal stores 65.6 against 75.0 for eight. On its own, after a kernel has left the L2 full of written lines,
// the first takes 16.9 us against 13.0 (the reads drive those lines out); after other reads the second takes 67.8 against
// 62.5, and a 256 MiB copy 90.4 against 79.4.
constexpr uint32_t kBlock = TSA_SCATTER_BLOCK_BYTES;
constexpr uint32_t kThreads = 256;
constexpr uint32_t kPerLane = kBlock / (16 * kThreads);  // 4

// Held to 8 waves per SIMD: unbounded, the whole entry took the kernel from 54 to 72 registers and 7 waves, so that 2048
// workgroups no longer ran at once (63 MB moved 14.8 us, with 54 registers 13.8, held 12.8).
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(8, 8))) void scatter_kernel(
    const TsaScatterJob* __restrict__ jobs, uint32_t n_jobs, uint64_t n_blocks) {
  const uint64_t blk = blockIdx.x;
  if (blk >= n_blocks) return;
  const uint32_t at = last_at_most(n_jobs, blk, [&](uint32_t i) { return jobs[i].block_first; });
  const TsaScatterJob j = jobs[__builtin_amdgcn_readfirstlane(at)];
  uint64_t b = blk - j.block_first;
  uint64_t src_off = 0, part_bytes = 0;
  char* dst = nullptr;
#pragma unroll
  for (uint32_t p = 0; p < TSA_MAX_EXTENTS; ++p) {
    if (p >= j.n_parts || dst) continue;
    const uint64_t nb = (j.bytes[p] + kBlock - 1) / kBlock;
    if (b < nb) {
      dst = static_cast<char*>(j.dst[p]);
      part_bytes = j.bytes[p];
    } else {
      b -= nb;
      src_off += j.bytes[p];
    }
  }
  if (!dst) return;  // (the host computed block_first from the same bytes: never reached)
  const uint64_t off = b * kBlock;
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  const u32x4* __restrict__ s = reinterpret_cast<const u32x4*>(static_cast<const char*>(j.src) + src_off + off);
  u32x4* __restrict__ d = reinterpret_cast<u32x4*>(dst + off);
  const uint64_t n16 = (part_bytes - off < kBlock ? part_bytes - off : kBlock) / 16;
  u32x4 v[kPerLane];
#pragma unroll
  for (uint32_t k = 0; k < kPerLane; ++k) {
    const uint64_t i = threadIdx.x + uint64_t(k) * kThreads;
    if (i < n16) v[k] = __builtin_nontemporal_load(s + i);
  }
#pragma unroll
  for (uint32_t k = 0; k < kPerLane; ++k) {
    const uint64_t i = threadIdx.x + uint64_t(k) * kThreads;
    if (i < n16) d[i] = v[k];
  }
}

// ---- synthetic bytes ----------------------------------------------------------------------------------------------
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
// Word i of stream `sid` under `seed`: mix64(key + (i + 1) * golden), key = mix64(seed ^ sid * odd).
constexpr uint64_t kGolden = 0x9E3779B97F4A7C15ull;

typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
typedef u64x2 u64x2_a8 __attribute__((aligned(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Two normals of one source word by Box-Muller (below), as bf16 values, the cosine's in the low half.
// The angle is exact up to its last step: lo32 counts 2^-32 turns, so its nearest quarter turn q and the signed rest r
// (lo32 << 2 as a signed number, in 2^-34 turns) are integer work, and only r, within an eighth of a turn, is rounded.
// sin and cos of the rest are polynomials in x^2 fitted here to |x| <= pi / 4 (relative error 6.1e-9 and 7.0e-10, both
// under the 6e-8 of a 32-bit rounding). Logarithm and square root are the hardware's (1 ulp).
__device__ __forceinline__ uint32_t normal_pair(uint64_t w, float sigma) {
  uint32_t hi = uint32_t(w >> 32);
  const uint32_t lo = uint32_t(w);
  asm("" : "+v"(hi));  // (a 32-bit value: the compiler would convert it as a 64-bit one, six instructions more)
  const float u1 = __builtin_fmaf(float(hi), 0x1p-32f, 0x1p-33f);
  const float rad = sigma * __builtin_amdgcn_sqrtf(__builtin_amdgcn_logf(u1) * -1.3862943611198906f);  // -2 ln 2 log2
  const float x = __builtin_fmaf(float(int32_t(lo << 2)), 6.283185307179586f * 0x1p-34f, 6.283185307179586f * 0x1p-33f);
  const uint32_t q = lo + 0x20000000u;  // the quarter turn in the top two bits
  const float z = x * x;
  const float sn = __builtin_fmaf(
      z * x, __builtin_fmaf(z, __builtin_fmaf(z, -1.95172979e-4f, 8.33217800e-3f), -1.66666552e-1f), x);
  const float cs = __builtin_fmaf(
      z, __builtin_fmaf(z, __builtin_fmaf(z, __builtin_fmaf(z, 2.44384512e-5f, -1.38873676e-3f), 4.16666456e-2f), -0.5f),
      1.0f);
  const bool odd = q & 0x40000000u;
  const uint32_t c = __float_as_uint(odd ? sn : cs) ^ ((q + 0x40000000u) & 0x80000000u);
  const uint32_t s = __float_as_uint(odd ? cs : sn) ^ (q & 0x80000000u);
  const bf16x2 v = __builtin_convertvector(f32x2{rad * __uint_as_float(c), rad * __uint_as_float(s)}, bf16x2);
  return __builtin_bit_cast(uint32_t, v);
}

// kind 0: every 8-byte word is word_at(i). kind 1: word i gives two bf16 values (elements 2i, 2i + 1) by Box-Muller:
// u1 = (hi32 + 0.5) / 2^32, u2 = (lo32 + 0.5) / 2^32, r = sigma sqrt(-2 ln u1), (r cos 2 pi u2, r sin 2 pi u2); a
// 64-bit output word then holds elements 4w .. 4w + 3, i.e. source words 2w and 2w + 1. A lane makes two output words
// and stores them at once; the source words' counters step by kGolden, one product per lane. Kind 1 is bound by its
// arithmetic, about 52 vector instructions per source word of which 21 mix it: 112 MiB in 39.8 us (66.2 with the
// library's sinf, cosf, logf and sqrtf), 17 us of it the store; the values nearest to the 64-bit ones in all but 2.3e-5
// of the cases (1.6e-4). Kind 0: 112 MiB in 19.1 us (20.8 with 8-byte stores).
template <uint32_t kKind>
__global__ __launch_bounds__(256) void synth_kernel(uint64_t* __restrict__ dst, uint64_t n_words, uint64_t key,
                                                    uint64_t first_word, float sigma) {
  const uint64_t stride = uint64_t(gridDim.x) * blockDim.x * 2;
  for (uint64_t w = (uint64_t(blockIdx.x) * blockDim.x + threadIdx.x) * 2; w < n_words; w += stride) {
    u64x2 out;
    if constexpr (kKind == 0) {
      const uint64_t z = key + (first_word + w + 1) * kGolden;
      out = u64x2{mix64(z), mix64(z + kGolden)};
    } else {
      const uint64_t z = key + (2 * (first_word + w) + 1) * kGolden;
      uint32_t pair[4];
#pragma unroll
      for (uint32_t h = 0; h < 4; ++h) pair[h] = normal_pair(mix64(z + h * kGolden), sigma);
      out = u64x2{pair[0] | uint64_t(pair[1]) << 32, pair[2] | uint64_t(pair[3]) << 32};
    }
    if (w + 1 < n_words)
      *reinterpret_cast<u64x2_a8*>(dst + w) = out;
    else
      dst[w] = out.x;
  }
}

// kind 2: Q4 blocks of 18 bytes: block b is a little-endian fp16 scale, then 16 bytes of packed 4-bit values. The scale
// is 0x2000 | (low 10 bits of word 3b): exponent field 8, so 2^-7 x (1 + m / 1024), a positive scale in [0.0078,
// 0.0156); the 16 value bytes are words 3b + 1 and 3b + 2, little-endian. The blocks start at the stream's byte 0.
// Four blocks are nine output words, so a lane makes four blocks from their twelve source words, each mixed once (byte
// by byte, every output byte mixes a word again), and the workgroup's 18 KiB leave through LDS as whole lines. 7.9 MiB:
// 20.5 -> 3.9 us; 112 MiB: 245 -> 19.4 us, the rate of the plain store.
constexpr uint32_t kQ4Words = 9;
__global__ __launch_bounds__(256) void synth_q4_kernel(uint64_t* __restrict__ dst, uint64_t n_words, uint64_t key,
                                                       uint64_t first_word) {
  __shared__ __attribute__((aligned(16))) uint64_t lds[256 * kQ4Words];
  const uint64_t group0 = first_word / kQ4Words + uint64_t(blockIdx.x) * 256;  // the workgroup's first four blocks
  const uint64_t z = key + ((group0 + threadIdx.x) * 12 + 1) * kGolden;
  uint64_t s[4], a[4], b[4];
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    s[k] = 0x2000u | (mix64(z + (3 * k) * kGolden) & 0x3FFu);
    a[k] = mix64(z + (3 * k + 1) * kGolden);
    b[k] = mix64(z + (3 * k + 2) * kGolden);
  }
  uint64_t* o = lds + threadIdx.x * kQ4Words;
  o[0] = s[0] | a[0] << 16;
  o[1] = a[0] >> 48 | b[0] << 16;
  o[2] = b[0] >> 48 | s[1] << 16 | a[1] << 32;
  o[3] = a[1] >> 32 | b[1] << 32;
  o[4] = b[1] >> 32 | s[2] << 32 | a[2] << 48;
  o[5] = a[2] >> 16 | b[2] << 48;
  o[6] = b[2] >> 16 | s[3] << 48;
  o[7] = a[3];
  o[8] = b[3];
  __syncthreads();
  const int64_t w0 = int64_t(group0 * kQ4Words - first_word);  // where lds[0] goes (before dst in the first workgroup)
  for (uint32_t i = threadIdx.x * 2; i < 256 * kQ4Words; i += 512) {
    const int64_t w = w0 + i;
    const u64x2 v = *reinterpret_cast<const u64x2*>(lds + i);
    if (w >= 0 && uint64_t(w) + 1 < n_words) {
      *reinterpret_cast<u64x2_a8*>(dst + w) = v;
    } else {
      if (w >= 0 && uint64_t(w) < n_words) dst[w] = v.x;
      if (w + 1 >= 0 && uint64_t(w + 1) < n_words) dst[w + 1] = v.y;
    }
  }
}

}  // namespace dev

int launch_scatter(const TsaScatterJob* jobs_dev, uint32_t n_jobs, uint64_t n_blocks, hipStream_t stream) {
  if (n_jobs == 0 || n_blocks == 0) return 0;
  if (n_blocks > 0x7fffffffull) return int(hipErrorInvalidValue);
  hipLaunchKernelGGL(dev::scatter_kernel, dim3(uint32_t(n_blocks)), dim3(dev::kThreads), 0, stream, jobs_dev, n_jobs,
                     n_blocks);
  return int(hipGetLastError());
}

int launch_synth(void* dst, uint64_t bytes, uint64_t seed, uint64_t stream_id, uint64_t offset, uint32_t kind,
                 float sigma, hipStream_t stream) {
  const uint64_t n_words = bytes / 8;
  if (n_words == 0) return 0;
  const uint64_t key = dev_key(seed, stream_id);
  uint64_t* d = static_cast<uint64_t*>(dst);
  const uint64_t first = offset / 8;
  if (kind == 2) {
    const uint64_t groups = (first + n_words - 1) / dev::kQ4Words - first / dev::kQ4Words + 1;
    const uint64_t blocks = (groups + 255) / 256;
    if (blocks > 0x7fffffffull) return int(hipErrorInvalidValue);
    hipLaunchKernelGGL(dev::synth_q4_kernel, dim3(uint32_t(blocks)), dim3(256), 0, stream, d, n_words, key, first);
    return int(hipGetLastError());
  }
  // One pass per lane: a capped grid of whole rounds left up to an eighth of the chip's time in its last one.
  const uint64_t want = (n_words + 511) / 512;
  const uint32_t blocks = uint32_t(want < (1u << 20) ? want : 1u << 20);
  hipLaunchKernelGGL(kind == 0 ? dev::synth_kernel<0> : dev::synth_kernel<1>, dim3(blocks), dim3(256), 0, stream, d,
                     n_words, key, first, sigma);
  return int(hipGetLastError());
}

}  // namespace tsa
