// Reduction of a 4-D decoder attention mask to per-token key validity, for
// sparse_prefill_attention_forward (sparse/attention.py:147-150, 173-176 in the
// reference pass the mask on as it is; here padded batches take the kernel that
// needs only key validity).
//
// A mask is causal key padding when, the same for every head and with only
// 0 / <= finfo.min / 2 values (or bool), every query row r attends exactly the
// keys j <= r that are real -- key j is real when the last row attends it --
// except that a padding row may also attend nothing or everything.
//
// One wavefront per (batch, query row), one read of the mask (the last row
// comes from L2).  Bound: that read and the launch: [4, 1, 2048, 2048] bool in
// 6.5 us, byte by byte 10.5 us; the fourteen tensor operations this replaces
// took 100 us and waited for the GPU three times.
#include "common.h"

namespace spruce {

namespace {

struct MaskParams {
  const void* mask;
  int64_t st[4];     // element strides (batch, head, query, key = 1)
  int B, Hm, T;
  float floor;       // values above it (and below 0) are biases: finfo.min / 2
  uint8_t* valid;    // [B, T]
  int32_t* flags;    // [0]: not causal key padding, [1]: some key is padding
};

struct MBool {
  using raw = uint8_t;
  static __device__ bool attends(raw v) { return v != 0; }
  static __device__ bool biased(raw, float) { return false; }
  static __device__ bool same(raw a, raw b) { return (a != 0) == (b != 0); }
};
template <typename Raw, bool F16>
struct MFloat {
  using raw = Raw;
  static __device__ float value(raw v) {
    if constexpr (sizeof(Raw) == 4)
      return __builtin_bit_cast(float, v);
    else
      return unpack1<F16>(v);
  }
  static __device__ bool attends(raw v) { return value(v) >= 0.f; }
  static __device__ bool biased(raw v, float floor) {
    const float x = value(v);
    return x >= 0.f ? x != 0.f : x > floor;
  }
  static __device__ bool same(raw a, raw b) { return value(a) == value(b); }
};

// VEC: rows are 16-byte aligned, read 16 bytes a lane; the tail of T that
// does not fill 16 bytes, and every element otherwise, is read one by one.
template <typename M, bool VEC>
__global__ __launch_bounds__(256) void mask_key_validity_kernel(const MaskParams p) {
  using Raw = typename M::raw;
  constexpr int N = VEC ? 16 / (int)sizeof(Raw) : 1;
  struct alignas(VEC ? 16 : sizeof(Raw)) Pack { Raw v[N]; };
  const int lane = threadIdx.x & 63;
  const int64_t g = (int64_t)flat_block() * 4 + (threadIdx.x >> 6);
  if (g >= (int64_t)p.B * p.T) return;
  const int b = (int)(g / p.T), r = (int)(g - (int64_t)b * p.T);
  const Raw* base = static_cast<const Raw*>(p.mask) + b * p.st[0];
  const Raw* row = base + r * p.st[2];
  const Raw* last = base + (int64_t)(p.T - 1) * p.st[2];
  bool bad = false, differs = false, any = false, all = true, padded = false;
  auto one = [&](int j, Raw v, Raw l) {
    const bool at = M::attends(v), real = M::attends(l);
    bad |= M::biased(v, p.floor);
    differs |= at != (real && j <= r);
    any |= at;
    all &= at;
    padded |= !real;
    if (r == p.T - 1) p.valid[(int64_t)b * p.T + j] = real ? 1 : 0;
  };
  const int whole = p.T / N * N;
  int j_first = lane * N;
  if constexpr (VEC && sizeof(Raw) == 1) {
    // Bool rows of one head, four keys a word: bit 7 of a byte is its truth.
    if (p.Hm == 1) {
      auto truth = [](uint32_t w) { return (((w & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w) & 0x80808080u; };
      uint32_t diff = 0, seen = 0, unseen = 0, unreal = 0;
      for (int j0 = j_first; j0 < whole; j0 += 64 * N) {
        const uint4 v = *reinterpret_cast<const uint4*>(row + j0), l = *reinterpret_cast<const uint4*>(last + j0);
        const uint32_t vw[4] = {v.x, v.y, v.z, v.w}, lw[4] = {l.x, l.y, l.z, l.w};
        uint32_t rw[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const uint32_t at = truth(vw[w]), real = truth(lw[w]);
          const int n = r - (j0 + 4 * w) + 1;  // causal keys of the word
          const uint32_t cm = n >= 4 ? 0xffffffffu : n <= 0 ? 0u : (1u << (8 * n)) - 1u;
          diff |= at ^ (real & cm);
          seen |= at;
          unseen |= at ^ 0x80808080u;
          unreal |= real ^ 0x80808080u;
          rw[w] = real >> 7;
        }
        if (r == p.T - 1)
          for (int w = 0; w < 16; ++w) p.valid[(int64_t)b * p.T + j0 + w] = (rw[w / 4] >> (8 * (w % 4))) & 1u;
      }
      differs = diff != 0;
      any = seen != 0;
      all = unseen == 0;
      padded = unreal != 0;
      j_first = whole;
    }
  }
  for (int j0 = j_first; j0 < whole; j0 += 64 * N) {
    const Pack v = *reinterpret_cast<const Pack*>(row + j0), l = *reinterpret_cast<const Pack*>(last + j0);
#pragma unroll
    for (int e = 0; e < N; ++e) one(j0 + e, v.v[e], l.v[e]);
    for (int h = 1; h < p.Hm; ++h) {
      const Pack o = *reinterpret_cast<const Pack*>(row + h * p.st[1] + j0);
#pragma unroll
      for (int e = 0; e < N; ++e) bad |= !M::same(o.v[e], v.v[e]);
    }
  }
  for (int j = whole + lane; j < p.T; j += 64) {
    one(j, row[j], last[j]);
    for (int h = 1; h < p.Hm; ++h) bad |= !M::same(row[h * p.st[1] + j], row[j]);
  }
  const bool real_row = M::attends(last[r]);
  const bool opened = __ballot(!all) == 0 || __ballot(any) == 0;
  const bool fail = __ballot(bad) != 0 || (__ballot(differs) != 0 && (real_row || !opened));
  const bool pad = __ballot(padded) != 0;
  if (lane == 0) {
    if (fail) p.flags[0] = 1;
    if (pad && r == p.T - 1) p.flags[1] = 1;
  }
}

// Rows with no listed block (every entry negative) among `rows` contiguous
// rows of K: a thread per row, one read of the lists.
__global__ __launch_bounds__(256) void empty_rows_kernel(const int32_t* __restrict__ ids, int64_t rows, int64_t K,
                                                         int32_t* flag) {
  const int64_t r = (int64_t)flat_block() * 256 + threadIdx.x;
  if (r >= rows) return;
  bool listed = false;
  for (int64_t k = 0; k < K && !listed; ++k) listed = ids[r * K + k] >= 0;
  if (!listed) *flag = 1;
}

}  // namespace
}  // namespace spruce

using namespace spruce;

extern "C" int spruce_empty_rows(const int32_t* ids, int64_t rows, int64_t K, int32_t* flag, void* stream) {
  SPRUCE_REQUIRE(ids && flag, "ids and flag must be non-null");
  SPRUCE_REQUIRE(rows >= 1 && K >= 1 && K < ((int64_t)1 << 31) && rows < ((int64_t)1 << 38), "invalid list shape");
  hipLaunchKernelGGL(empty_rows_kernel, flat_grid((rows + 255) / 256), dim3(256), 0, (hipStream_t)stream, ids,
                     rows, K, flag);
  return check_launch("empty_rows_kernel");
}

extern "C" int spruce_mask_key_validity(const void* mask, const int64_t ms[4], int64_t Hm, int mask_dtype, int64_t B,
                                        int64_t T, uint8_t* valid, int32_t* flags, void* stream) {
  SPRUCE_REQUIRE(mask && ms && valid && flags, "mask, strides, valid and flags must be non-null");
  SPRUCE_REQUIRE(B >= 1 && Hm >= 1 && T >= 1 && T < ((int64_t)1 << 30) && B < ((int64_t)1 << 30) &&
                     Hm < ((int64_t)1 << 30) && B * T < ((int64_t)1 << 31),
                 "invalid mask shape");
  SPRUCE_REQUIRE(ms[3] == 1, "the mask's last dimension must be contiguous");
  SPRUCE_REQUIRE(mask_dtype >= 0 && mask_dtype <= 3, "unsupported mask dtype code %d", mask_dtype);
  const int eb = mask_dtype == 3 ? 1 : (mask_dtype == 2 ? 4 : 2);
  MaskParams p{};
  p.mask = mask;
  for (int i = 0; i < 4; ++i) p.st[i] = ms[i];
  p.B = (int)B;
  p.Hm = (int)Hm;
  p.T = (int)T;
  p.valid = valid;
  p.flags = flags;
  // finfo.min / 2 of the mask's dtype.
  p.floor = mask_dtype == 1 ? -32752.f : mask_dtype == 0 ? -0x1.fep126f : -0x1.fffffep126f;
  bool vec = (uintptr_t)mask % 16 == 0;
  for (int i = 0; i < 3; ++i) vec = vec && (ms[i] * eb) % 16 == 0;
  const dim3 grid = flat_grid((B * T + 3) / 4);
  auto go = [&](auto m) {
    using M = decltype(m);
    if (vec)
      hipLaunchKernelGGL((mask_key_validity_kernel<M, true>), grid, dim3(256), 0, (hipStream_t)stream, p);
    else
      hipLaunchKernelGGL((mask_key_validity_kernel<M, false>), grid, dim3(256), 0, (hipStream_t)stream, p);
  };
  if (mask_dtype == 3) go(MBool{});
  else if (mask_dtype == 2) go(MFloat<uint32_t, false>{});
  else if (mask_dtype == 1) go(MFloat<uint16_t, true>{});
  else go(MFloat<uint16_t, false>{});
  return check_launch("mask_key_validity_kernel");
}
