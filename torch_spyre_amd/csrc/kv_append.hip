// Writes of the paged stick-layout KV cache.
//
// Batched append (spyre_kv_append_f16): the new token of every sequence is written into its
// page slot in one launch, with the positions read from device memory.
//
//   K cache [num_pages, Hkv, D/64, 64 tok, 64]: the token's D values land as
//     D/64 partial-stick writes of 128 contiguous bytes each;
//   V cache [num_pages, Hkv, D, 64 tok]: the token is one column of the
//     page's D sticks (the transposed, relayout-on-write half).
//
// Positions < 0 skip the sequence; positions past the block table's row and
// page ids outside [0, num_pages) are not written (dropped rather than faulting).

#include <hip/hip_runtime.h>

#include "fast_div.h"
#include "spyre_common.h"
#include "transpose8.h"

namespace {

using spyre_hip::fdiv;
using spyre_hip::u32x4_t;

constexpr int kPage = 64;

__global__ void kv_append_kernel(const _Float16* __restrict__ k_new,
                                 const _Float16* __restrict__ v_new, _Float16* __restrict__ kc,
                                 _Float16* __restrict__ vc, const int32_t* __restrict__ bt,
                                 int64_t bt_stride, int64_t pages_per_seq,
                                 const int32_t* __restrict__ pos, int Hkv, int D,
                                 int64_t num_pages) {
  const int h = blockIdx.x, b = blockIdx.y, d = threadIdx.x;
  const int p = pos[b];
  if (p < 0 || p / kPage >= pages_per_seq) return;
  const int64_t page = bt[static_cast<int64_t>(b) * bt_stride + p / kPage];
  if (page < 0 || page >= num_pages) return;
  const int slot = p % kPage;
  const int64_t src = (static_cast<int64_t>(b) * Hkv + h) * D + d;
  const int64_t head = (page * Hkv + h) * static_cast<int64_t>(D) * kPage;
  kc[head + (d / 64) * (kPage * 64) + slot * 64 + (d % 64)] = k_new[src];
  vc[head + static_cast<int64_t>(d) * kPage + slot] = v_new[src];
}

// Dense K / V into whole pages (spyre_dense_to_pages_f16).  A wavefront moves
// one unit: 64 tokens x 64 features of K, a copy whose 8 KiB are contiguous
// in the page, and the same block of V, transposed in registers (8 x 8
// elements per lane) to 8 contiguous KiB.  Bound by memory: every load and
// store instruction covers whole 128-byte lines, the 16 loads of a unit go out
// before its first store, and tokens past S are written as zeros by the same
// stores.  8 x 8 heads x 3000 tokens of D 128 (197 MB moved): 33.9 us, 5.8 TB/s
// (traced); padding the tensors first and moving them as two relayouts took
// 93.7 us a call, 56 of them for the padding.
struct PagesArgs {
  const uint16_t *k, *v;
  int64_t k_sb, k_sh, k_ss, v_sb, v_sh, v_ss;  // elements
  uint16_t *kc, *vc;
  uint32_t Hkv, P, DT, units;  // units: B P Hkv DT, in the pages' own order
  int S;
  spyre_hip::FastDiv by_dt, by_h, by_p;
};
constexpr int kUnitWaves = 4;

template <bool WHOLE>
__device__ __forceinline__ void move_unit(const uint16_t* ks, int64_t k_ss, const uint16_t* vs, int64_t v_ss,
                                          uint16_t* kd, uint16_t* vd, int rows, int lane) {
  const int lr = lane / 8, lc = lane % 8;
  u32x4_t x[8], y[8], z[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {  // K token 8 j + lr, features 8 lc .. + 7
    const int t = 8 * j + lr;
    x[j] = u32x4_t{0, 0, 0, 0};
    if (WHOLE || t < rows) x[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(ks + t * k_ss + 8 * lc));
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {  // V token 8 lr + j, features 8 lc .. + 7
    const int t = 8 * lr + j;
    y[j] = u32x4_t{0, 0, 0, 0};
    if (WHOLE || t < rows) y[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(vs + t * v_ss + 8 * lc));
  }
  __builtin_amdgcn_sched_barrier(0);  // keep every load ahead of the stores
#pragma unroll
  for (int j = 0; j < 8; ++j) __builtin_nontemporal_store(x[j], reinterpret_cast<u32x4_t*>(kd + 512 * j + 8 * lane));
  spyre_hip::transpose8x8_b16(y, z);
#pragma unroll
  for (int e = 0; e < 8; ++e)  // feature 8 lc + e, tokens 8 lr .. + 7
    __builtin_nontemporal_store(z[e], reinterpret_cast<u32x4_t*>(vd + (8 * lc + e) * kPage + 8 * lr));
}

__global__ __launch_bounds__(kUnitWaves * 64) void dense_to_pages_kernel(PagesArgs a) {
  const uint32_t u = blockIdx.x * kUnitWaves + __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  if (u >= a.units) return;
  const int lane = threadIdx.x % 64;
  const uint32_t i1 = fdiv(u, a.by_dt), i2 = fdiv(i1, a.by_h), b = fdiv(i2, a.by_p);
  const uint32_t dt = u - i1 * a.DT, h = i1 - i2 * a.Hkv, p = i2 - b * a.P;
  const int64_t t0 = static_cast<int64_t>(p) * kPage;
  const uint16_t* ks = a.k + b * a.k_sb + h * a.k_sh + t0 * a.k_ss + dt * 64;
  const uint16_t* vs = a.v + b * a.v_sb + h * a.v_sh + t0 * a.v_ss + dt * 64;
  uint16_t* kd = a.kc + static_cast<int64_t>(u) * (kPage * 64);
  uint16_t* vd = a.vc + static_cast<int64_t>(u) * (kPage * 64);
  const int rows = a.S - static_cast<int>(t0);
  if (rows >= kPage)
    move_unit<true>(ks, a.k_ss, vs, a.v_ss, kd, vd, kPage, lane);
  else
    move_unit<false>(ks, a.k_ss, vs, a.v_ss, kd, vd, rows, lane);
}

}  // namespace

extern "C" int spyre_dense_to_pages_f16(const void* k, const int64_t* k_strides, const void* v,
                                        const int64_t* v_strides, void* k_pages, void* v_pages, int B, int Hkv,
                                        int S, int D, void* stream) {
  spyre_hip::clear_error();
  SPYRE_REQUIRE(B >= 0 && Hkv > 0 && S >= 0, SPYRE_EINVAL, "bad sizes B=%d Hkv=%d S=%d", B, Hkv, S);
  SPYRE_REQUIRE(D > 0 && D % 64 == 0, SPYRE_EUNSUPPORTED, "head_dim %d not a multiple of 64", D);
  if (B == 0) return SPYRE_OK;  // no page: empty tensors have no address
  SPYRE_REQUIRE(k_strides && v_strides && k_pages && v_pages && (S == 0 || (k && v)), SPYRE_EINVAL,
                "null pointer argument");
  auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  SPYRE_REQUIRE(aligned(k) && aligned(v) && aligned(k_pages) && aligned(v_pages), SPYRE_EINVAL,
                "k, v and the pages must be 16-byte aligned");
  for (int i = 0; i < 3; ++i)
    SPYRE_REQUIRE(k_strides[i] % 8 == 0 && v_strides[i] % 8 == 0 && k_strides[i] >= 0 && v_strides[i] >= 0,
                  SPYRE_EINVAL, "k/v strides must be non-negative multiples of 8 elements");
  const int64_t P = S > 0 ? (static_cast<int64_t>(S) + kPage - 1) / kPage : 1;
  const int64_t units = B * P * Hkv * (D / 64);
  SPYRE_REQUIRE(units < (int64_t{1} << 31) - kUnitWaves, SPYRE_EUNSUPPORTED, "too many pages");
  PagesArgs a{static_cast<const uint16_t*>(k), static_cast<const uint16_t*>(v), k_strides[0], k_strides[1],
              k_strides[2], v_strides[0], v_strides[1], v_strides[2], static_cast<uint16_t*>(k_pages),
              static_cast<uint16_t*>(v_pages), static_cast<uint32_t>(Hkv), static_cast<uint32_t>(P),
              static_cast<uint32_t>(D / 64), static_cast<uint32_t>(units), S,
              spyre_hip::make_fastdiv(static_cast<uint32_t>(D / 64)),
              spyre_hip::make_fastdiv(static_cast<uint32_t>(Hkv)), spyre_hip::make_fastdiv(static_cast<uint32_t>(P))};
  dense_to_pages_kernel<<<dim3(static_cast<uint32_t>((units + kUnitWaves - 1) / kUnitWaves)), kUnitWaves * 64, 0,
                          static_cast<hipStream_t>(stream)>>>(a);
  const hipError_t e = hipGetLastError();
  SPYRE_REQUIRE(e == hipSuccess, SPYRE_EHIP, "dense to pages launch failed: %s", hipGetErrorString(e));
  return SPYRE_OK;
}

extern "C" int spyre_kv_append_f16(const void* k_new, const void* v_new, void* k_cache,
                                   void* v_cache, const int32_t* block_table, int64_t bt_stride,
                                   int64_t pages_per_seq, const int32_t* positions, int B, int Hkv,
                                   int D, int page_size, int64_t num_pages, void* stream) {
  spyre_hip::clear_error();
  SPYRE_REQUIRE(k_new && v_new && k_cache && v_cache && block_table && positions, SPYRE_EINVAL,
                "null pointer argument");
  SPYRE_REQUIRE(B >= 0 && Hkv > 0 && num_pages > 0 && bt_stride >= 0 && pages_per_seq >= 0,
                SPYRE_EINVAL,
                "bad sizes B=%d Hkv=%d num_pages=%lld", B, Hkv, static_cast<long long>(num_pages));
  SPYRE_REQUIRE(D == 64 || D == 128, SPYRE_EUNSUPPORTED, "head_dim %d not in {64, 128}", D);
  SPYRE_REQUIRE(page_size == kPage, SPYRE_EUNSUPPORTED, "page_size %d != %d", page_size, kPage);
  if (B == 0) return SPYRE_OK;
  kv_append_kernel<<<dim3(Hkv, B), D, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const _Float16*>(k_new), static_cast<const _Float16*>(v_new),
      static_cast<_Float16*>(k_cache), static_cast<_Float16*>(v_cache), block_table, bt_stride,
      pages_per_seq, positions, Hkv, D, num_pages);
  const hipError_t e = hipGetLastError();
  SPYRE_REQUIRE(e == hipSuccess, SPYRE_EHIP, "kv append launch failed: %s", hipGetErrorString(e));
  return SPYRE_OK;
}
