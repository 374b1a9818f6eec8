// Device top-M of a logits vector: the M largest (index, value) pairs in the sampler's order - value descending, the
// lower index first among equal values (top_m and the sort in Sampler::dist, /root/reference/src/sampler.cpp:12-27 and
// :41-42).  The host then applies its penalties / temperature / top-p to those M candidates, so it receives M pairs
// instead of V floats.
//
// Each pair is one 64-bit key whose ascending order is the sampler's order: the high word is the complement of the
// value's order-preserving unsigned image, the low word the index.  Rounds: every workgroup reduces a chunk of keys to
// its first M; the survivors form the next round's input, until one chunk is left, whose first M keys are the result.
// A wave keeps the first 64 E keys it has seen (64 E >= M) sorted in registers, E per lane.  It sorts the next 64 E the
// other way round (bitonic, lane exchanges by DPP and swizzles), keeps the smaller of each pair - the smallest 64 E of
// both, a bitonic sequence - and sorts that in log2(64 E) stages; keys none of which precedes the list's last are
// skipped.  A workgroup's 16 lists are merged pairwise in the same way through LDS, two barriers for each of the four levels.  It is a chain of
// lane exchanges, so its latency bounds it.  Measured (MI355X, 151936 values, us): M = 40 14 + 5, M = 100 15 + 9, M = 200 17 +
// 18, M = 512 26 + 44 (before: a bitonic sort of 4096 keys per workgroup in LDS, 78 barriers and 28 - 32 us for each of two
// rounds, three at M = 512).
#include <mutex>

#include "launch.hpp"

namespace qph {

// keys per workgroup: 4096 of the logits (with a vocabulary of 32 - 152 thousand the second round then has 8 - 38 M keys),
// up to 32768 survivors, so that two rounds do for every vocabulary of up to 262144
constexpr int kTopkChunk = 4096, kTopkChunkNext = 32768, kTopkThreads = 1024, kTopkWaves = kTopkThreads / 64;

__device__ __forceinline__ uint64_t topk_key(float v, int i) {
  // -0 compares equal to +0 (the index then decides, as in the sampler's comparison), so it takes +0's key
  const uint32_t b = v == 0.f ? 0u : __builtin_bit_cast(uint32_t, v);
  const uint32_t k = (b & 0x80000000u) ? ~b : (b | 0x80000000u);   // ascending with the float value
  return ((uint64_t)(~k) << 32) | (uint32_t)i;
}
__device__ __forceinline__ float topk_val(uint64_t key) {
  const uint32_t k = ~(uint32_t)(key >> 32);
  return __builtin_bit_cast(float, (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

__device__ __forceinline__ uint32_t lane_xor(uint32_t v, int j) {   // lane l reads lane l ^ j
  switch (j) {
    case 1: return (uint32_t)dpp_i<kDppQuadXor1>((int)v);
    case 2: return (uint32_t)dpp_i<kDppQuadXor2>((int)v);
    case 4: return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, 0x101f);
    case 8: return (uint32_t)dpp_i<kDppRowRor8>((int)v);
    case 16: return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, 0x401f);
    default: return (uint32_t)__shfl_xor((int)v, 32);
  }
}
// one compare-exchange stage over elements i = 64 e + lane: pairs (i, i ^ j), ascending where bit k of i is clear
template <int E>
__device__ __forceinline__ void topk_stage(uint64_t (&key)[E], int k, int j, bool desc, int lane) {
  if (j >= 64) {
#pragma unroll
    for (int e = 0; e < E; e++) {
      const int p = e ^ (j >> 6);
      if (p < e) continue;
      const bool up = ((64 * e & k) == 0) != desc;
      const uint64_t a = key[e], b = key[p];
      const bool swap = (a > b) == up;
      key[e] = swap ? b : a; key[p] = swap ? a : b;
    }
    return;
  }
#pragma unroll
  for (int e = 0; e < E; e++) {
    const uint64_t a = key[e];
    const uint64_t b = (uint64_t)lane_xor((uint32_t)(a >> 32), j) << 32 | lane_xor((uint32_t)a, j);
    const bool up = (((64 * e | lane) & k) == 0) != desc, low = (lane & j) == 0;
    key[e] = (a > b) == (low == up) ? b : a;   // the low element of an ascending pair takes the smaller
  }
}
// 64 E keys in any order -> sorted, descending
template <int E>
__device__ __forceinline__ void topk_sort_desc(uint64_t (&key)[E], int lane) {
#pragma unroll
  for (int k = 2; k <= 64 * E; k <<= 1)
#pragma unroll
    for (int j = k >> 1; j > 0; j >>= 1) topk_stage<E>(key, k, j, true, lane);
}
// list (ascending) and other (descending) -> list: the smallest 64 E of both, ascending
template <int E>
__device__ __forceinline__ void topk_merge(uint64_t (&list)[E], const uint64_t (&other)[E], int lane) {
#pragma unroll
  for (int e = 0; e < E; e++) list[e] = other[e] < list[e] ? other[e] : list[e];
#pragma unroll
  for (int j = 32 * E; j > 0; j >>= 1) topk_stage<E>(list, 128 * E, j, false, lane);   // bit k of no element is set
}

// one chunk of n input keys (from x when keys_in is null) -> its M smallest keys at out + chunk * M, or, in the last
// round (idx != null, one chunk), decoded into idx[M] / val[M].  M <= 64 E
template <int E>
__global__ __launch_bounds__(kTopkThreads) void k_topk_chunk(const float *x, const uint64_t *keys_in, int n, int chunk, int M,
                                                             uint64_t *out, int *idx, float *val) {
  __shared__ uint64_t s[kTopkWaves / 2][64 * E];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int base = blockIdx.x * chunk, end = min(n - base, chunk);
  constexpr int L = 64 * E, U = E < 4 ? 4 / E : 1;   // U runs of L keys are loaded at a time
  uint64_t list[E];
#pragma unroll
  for (int e = 0; e < E; e++) list[e] = ~0ull;   // padding sorts last
  for (int g = wave * L; g < end; g += kTopkWaves * L * U) {
    uint64_t key[U][E];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int e = 0; e < E; e++) {
        const int i = g + u * kTopkWaves * L + 64 * e + lane;
        key[u][e] = i < end ? (keys_in ? keys_in[base + i] : topk_key(x[base + i], base + i)) : ~0ull;
      }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint64_t last = __shfl(list[E - 1], 63);
      bool any = false;
#pragma unroll
      for (int e = 0; e < E; e++) any |= key[u][e] < last;
      if (!__any(any)) continue;
      topk_sort_desc<E>(key[u], lane);
      topk_merge<E>(list, key[u], lane);
    }
  }
  for (int h = kTopkWaves / 2; h > 0; h >>= 1) {   // waves h .. 2 h - 1 leave their lists to waves 0 .. h - 1
    if (wave >= h && wave < 2 * h)
#pragma unroll
      for (int e = 0; e < E; e++) s[wave - h][L - 1 - (64 * e + lane)] = list[e];
    __syncthreads();
    if (wave < h) {
      uint64_t other[E];
#pragma unroll
      for (int e = 0; e < E; e++) other[e] = s[wave][64 * e + lane];
      topk_merge<E>(list, other, lane);
    }
    __syncthreads();
  }
  if (wave == 0)
#pragma unroll
    for (int e = 0; e < E; e++) {
      const int i = 64 * e + lane;
      if (i >= M) continue;
      if (idx) { idx[i] = (int)(uint32_t)list[e]; val[i] = topk_val(list[e]); }
      else out[(size_t)blockIdx.x * M + i] = list[e];
    }
}

size_t topk_scratch_keys(int n, int M) { return (size_t)((n + kTopkChunk - 1) / kTopkChunk) * (size_t)M; }

hipError_t launch_topk(const float *x, int n, int M, uint64_t *buf_a, uint64_t *buf_b, int *idx, float *val,
                       hipStream_t st) {
  if (n <= 0 || M < 1 || M > kTopkMax || M > n) return hipErrorInvalidValue;
  const uint64_t *in = nullptr;
  uint64_t *out = buf_a, *spare = buf_b;
  int len = n;
  for (;;) {
    const int chunk = in ? kTopkChunkNext : kTopkChunk, chunks = (len + chunk - 1) / chunk;
    const bool last = chunks == 1;
#define QPH_TOPK(E)                                                                                                 \
  hipLaunchKernelGGL(k_topk_chunk<E>, dim3(chunks), dim3(kTopkThreads), 0, st, in ? nullptr : x, in, len, chunk, M, \
                     out, last ? idx : nullptr, last ? val : nullptr)
    if (M <= 64) QPH_TOPK(1);
    else if (M <= 128) QPH_TOPK(2);
    else if (M <= 256) QPH_TOPK(4);
    else QPH_TOPK(8);
#undef QPH_TOPK
    if (last) break;
    len = chunks * M;   // survivors (M per chunk; M <= chunk / 8, so every round shrinks the input 8 times or more)
    in = out;
    std::swap(out, spare);
  }
  return hipGetLastError();
}

// ---- the top-M without allocation (qph_topk_noalloc): the key buffers live in a file-scope device array, one copy per
// GPU, held until the process ends.  Its address comes from hipGetSymbolAddress once per device, with that device
// current (the array's name in host code is only a stand-in: passed to a kernel it would fault).  Calls that overlap
// on one GPU share the array and race; the array keeps the last call's keys (every round writes what the next reads,
// so nothing needs clearing).
constexpr int kTopkNoAllocMaxN = 262144;
constexpr size_t kTopkNoAllocKeys = (size_t)(kTopkNoAllocMaxN / kTopkChunk) * kTopkMax;   // per buffer: 32768 keys
static __device__ __align__(256) uint64_t scratch[2 * kTopkNoAllocKeys];                  // 512 KiB per GPU

static uint64_t *scratch_ptr(int dev) {
  static std::mutex mu;
  static uint64_t *ptrs[64] = {};
  if (dev < 0 || dev >= 64) return nullptr;
  std::lock_guard<std::mutex> lock(mu);
  if (!ptrs[dev]) {
    void *p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
    ptrs[dev] = (uint64_t *)p;
  }
  return ptrs[dev];
}

hipError_t launch_topk_noalloc(const float *x, int n, int M, int *idx, float *val, hipStream_t st) {
  if (n <= 0 || n > kTopkNoAllocMaxN || M < 1 || M > kTopkMax || M > n) return hipErrorInvalidValue;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  uint64_t *base = scratch_ptr(dev);
  if (!base) return hipErrorInvalidSymbol;
  return launch_topk(x, n, M, base, base + kTopkNoAllocKeys, idx, val, st);
}

}  // namespace qph
