// Scaled dot-product attention forward for gfx950 (spyre_sdpa_fwd_f16):
// prefill and any Sq, with GQA, causal masking or an additive / boolean mask,
// and the natural-log logsumexp.
//
// Semantics (torch_spyre/_inductor/decompositions.py:523-609, with torch's
// CPU SDPA as the numerical reference):
//   out[b,h,i,:] = softmax_j(scale * q[b,h,i,:] . k[b,h/g,j,:] + bias[b,h,i,j]) v[b,h/g,j,:]
// bias = 0, or the mask (boolean masks keep where true), or for causal
// attention -inf where j > i (top-left aligned, triu(diagonal=1)).  A row
// whose keys are all masked gives zeros and LSE -inf (torch's CPU result;
// the reference's torch.softmax would give NaN there).
//
// Kernels, on the caller's stream:
//  * sdpa_fwd_lds_kernel serves calls without a mask (plain or causal),
//    fp16 / boolean masks whose rows are whole 16-byte units (others are
//    copied first) and fp32 biases with contiguous keys.  A workgroup
//    of 4 or 8 wavefronts takes 32 queries of one (sequence, q head) per
//    wavefront or pair of wavefronts (pick_shape).  Per 64-key step the K and
//    V tiles (row-major, swizzled) move from L2 straight into LDS (buffer loads
//    with the LDS flag), once for all its wavefronts:
//       S^T[key, q] = K[key, :] Q^T[:, q]     2 x D/16 MFMA 32x32x16
//       online softmax in fp32 (exp2 domain), lazy rescaling of the max;
//       O^T[d, q] += V^T[d, key] P^T[key, q]  4 x D/32 MFMA 32x32x16
//    with the V^T operands read from the row-major V tile by transposing
//    LDS reads.  The loop is software-pipelined: step t's softmax overlaps
//    S(t+1).  A mask is staged per wavefront beside the tiles, a step ahead;
//    steps it blanks for the whole wavefront skip their softmax and P V.
//  * Decode: sdpa_decode_short_kernel (a row tile's keys all in flight at
//    once) and the split-KV kernels of decode_attn.hip (dense_route), with
//    or without a mask.
//  * Other masks (fp32 biases whose keys are not contiguous, slices of 2 GiB):
//    1. v_token_sticks_kernel: V [B, Hkv, Skv, D] (rows may be strided) ->
//       Vt [B, Hkv, D, S64] in the workspace: V with its sticks along tokens
//       (the transpose-restick of each head), zero-padded to S64 = ceil(Skv
//       / 64) * 64, so the PV product's reduction dim (keys) is contiguous.
//    2. sdpa_fwd_kernel: one wavefront per 32 queries of one (sequence, q
//       head), four per workgroup, streaming 64 keys per step from L2:
//         S^T[key, q] = K[key, :] Q^T[:, q]   4 x D/32 x 2 MFMA 16x16x32
//         O^T[d, q] += Vt[d, key] P^T[key, q]   D/16 x 2 x 2 MFMA 16x16x32
//       reading the mask element by element through its broadcast strides.
// In both, the keys of the S rows are permuted so that each lane's P values
// are the 8 consecutive keys the PV operand needs (no lane exchange), and
// causal attention stops each wavefront at its last query's key.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <type_traits>

#include "decode_dense.h"
#include "fast_div.h"
#include "spyre_common.h"
#include "transpose8.h"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
using spyre_hip::fdiv;
using spyre_hip::u32x4_t;

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kQ = 32;      // queries per wavefront (two MFMA column tiles)
constexpr int kKeys = 64;   // keys per step
constexpr int kStick = 64;  // Vt token padding: whole 64-key steps
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

__device__ __forceinline__ float wave_xor(float x, int m) { return __shfl_xor(x, m, 64); }
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// K and Vt are read with buffer loads: the (sequence, head) base and extent
// in SGPRs, a 32-bit per-lane byte offset in one VGPR, the load-invariant
// part in an SGPR / immediate.  Accesses past the extent read zeros.
typedef __amdgpu_buffer_rsrc_t Rsrc;
constexpr int kRsrcWord3 = 0x00020000;  // raw (untyped) buffer, 32-bit format
// 16 bytes per lane from buffer offset voff into LDS: lane l writes the 16
// bytes at dst + 16 l (dst wave-uniform).  Lanes whose offset lies past the
// buffer's range write zeros.
// ds_read_b64_tr_b16 at LDS element p (see the V operand reads below).
__device__ __forceinline__ short __attribute__((ext_vector_type(4))) tr_read4(const _Float16* p) {
  typedef short v4s __attribute__((ext_vector_type(4)));
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s*)(p));
}

__device__ __forceinline__ void load_lds16(Rsrc r, _Float16* dst, uint32_t voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voff, 0, 0, 0);
}

// The same with 4 bytes per lane (lane l writes dst + 4 l).
__device__ __forceinline__ void load_lds4(Rsrc r, _Float16* dst, uint32_t voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 4, voff, 0, 0, 0);
}

// Range of the buffer descriptors whose bases move with the key step; the
// host keeps every head's K and Vt span within it.
constexpr uint32_t kBufRange = 0x7ffffff0u;

__device__ __forceinline__ Rsrc make_rsrc(const _Float16* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16*>(base), 0, bytes, kRsrcWord3);
}

__device__ __forceinline__ f16x8 bload(Rsrc r, int voff, int soff) {
  return __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// S^T block jh (16 keys of the step): MFMA row i <-> key 32(jh/2) + 8(i/4) + 4(jh%2) + i%4.
__device__ __forceinline__ int key_of(int jh, int i) {
  return 32 * (jh >> 1) + 8 * (i >> 2) + 4 * (jh & 1) + (i & 3);
}

// ---- 1. V -> token sticks -------------------------------------------------

struct VtArgs {
  const _Float16* v;
  int64_t sb, sh, ss;  // V strides (elements); d stride 1
  _Float16* vt;        // [B, Hkv, D, s64]
  int Hkv, Skv, s64, D;
  int64_t tiles;       // 64 x 64 tiles
};

// One wavefront per 64 tokens x 64 features: each lane loads an 8 x 8 block
// as eight 16-byte token rows, transposes it in registers and stores eight
// 16-byte feature rows of Vt.  Tokens past Skv are written as zeros.
__global__ __launch_bounds__(kThreads) void v_token_sticks_kernel(VtArgs a) {
  const int64_t tile = static_cast<int64_t>(blockIdx.x) * kWaves + threadIdx.x / 64;
  if (tile >= a.tiles) return;
  const int lane = threadIdx.x % 64;
  const int ts_n = a.s64 / 64, td_n = a.D / 64;
  const int ts = static_cast<int>(tile % ts_n);
  const int64_t r = tile / ts_n;
  const int td = static_cast<int>(r % td_n);
  const int64_t bh = r / td_n;
  const int64_t b = bh / a.Hkv, kvh = bh % a.Hkv;
  const int s0 = ts * 64 + (lane / 8) * 8, d0 = td * 64 + (lane % 8) * 8;
  const _Float16* src = a.v + b * a.sb + kvh * a.sh + d0;
  u32x4_t x[8], y[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const int s = s0 + t;
    x[t] = s < a.Skv ? *reinterpret_cast<const u32x4_t*>(src + s * a.ss) : u32x4_t{0, 0, 0, 0};
  }
  spyre_hip::transpose8x8_b16(x, y);
  _Float16* dst = a.vt + (bh * a.D + d0) * a.s64 + s0;
#pragma unroll
  for (int e = 0; e < 8; ++e) *reinterpret_cast<u32x4_t*>(dst + e * a.s64) = y[e];
}

// ---- 2. attention -----------------------------------------------------------

enum MaskKind { kNoMask = 0, kMaskF16 = 1, kMaskF32 = 2, kMaskBool = 3 };

struct FwdArgs {
  const _Float16* q;
  const _Float16* k;
  const _Float16* vt;
  int64_t q_sb, q_sh, q_ss;
  int64_t k_sb, k_sh, k_ss;
  int64_t vt_sb, vt_sh;
  uint32_t k_bytes, vt_bytes;  // extent of one (sequence, KV head) of K / Vt
  const void* mask;
  int64_t m_sb, m_sh, m_sq, m_sk;
  _Float16* out;  // [B, Sq, Hq, D]
  float* lse;     // [B, Hq, Sq] or null
  int B, Hq, Hkv, g, Sq, Skv, s64, mask_kind, causal;
  float scale_log2;
};

// Mask element types by kind.
template <int MK> struct MaskElem { using T = uint8_t; };
template <> struct MaskElem<kMaskF16> { using T = _Float16; };
template <> struct MaskElem<kMaskF32> { using T = float; };

// Additive bias (log2 domain) of mask element x.
template <int MK>
__device__ __forceinline__ float bias_of(typename MaskElem<MK>::T x) {
  if constexpr (MK == kMaskBool)
    return x ? 0.f : -INFINITY;
  else
    return static_cast<float>(x) * kLog2e;
}

// MK: mask kind (a separate kernel each, so the unmasked one carries no mask code).
template <int D, int MK>
__global__ __launch_bounds__(kThreads, 2) void sdpa_fwd_kernel(FwdArgs a) {
  constexpr int DS = D / 32;  // QK k-steps
  constexpr int DT = D / 16;  // O row tiles
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  const int b = blockIdx.z, h = blockIdx.y;
  const int q0 = (blockIdx.x * kWaves + wave) * kQ;
  if (q0 >= a.Sq) return;
  const int kvh = h / a.g;
  const int col = lane & 15, grp = lane >> 4;
  const _Float16* qp = a.q + b * a.q_sb + h * a.q_sh;
  const Rsrc kr = make_rsrc(a.k + b * a.k_sb + kvh * a.k_sh, a.k_bytes);
  const Rsrc vr = make_rsrc(a.vt + b * a.vt_sb + kvh * a.vt_sh, a.vt_bytes);

  // Q^T operands: lane (query column col, feature group grp).
  f16x8 qb[2][DS];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const int qi = q0 + 16 * nt + col;
#pragma unroll
    for (int ds = 0; ds < DS; ++ds)
      qb[nt][ds] = qi < a.Sq ? *reinterpret_cast<const f16x8*>(qp + qi * a.q_ss + 32 * ds + 8 * grp)
                             : f16x8{};
  }

  float m_run[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.f, 0.f};
  f32x4 o[2][DT];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[nt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Mask rows of this lane's two query columns (clamped into the mask).
  using MT = typename MaskElem<MK>::T;
  const MT* mrow[2] = {nullptr, nullptr};
  if constexpr (MK != kNoMask) {
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int qc = min(q0 + 16 * nt + col, a.Sq - 1);
      mrow[nt] = static_cast<const MT*>(a.mask) + b * a.m_sb + h * a.m_sh + qc * a.m_sq;
    }
  }
  const int m_sk = static_cast<int>(a.m_sk);

  // Per-lane byte offsets: K row key_of(jh, col) (+ 16-byte feature group),
  // Vt row col (+ 8 keys of group grp).  Keys past Skv are masked below;
  // their K rows are clamped to the last row.
  const int vt_lane = (col * a.s64 + 8 * grp) * 2;
  // Causal: no key past this wavefront's last query is needed.
  const int key_end = a.causal ? min(a.Skv, q0 + kQ) : a.Skv;
  for (int kb = 0; kb < key_end; kb += kKeys) {
    f16x8 ka[4][DS];
#pragma unroll
    for (int jh = 0; jh < 4; ++jh) {
      const int key = min(kb + key_of(jh, col), a.Skv - 1);
      const int voff = static_cast<int>(key * a.k_ss * 2) + 16 * grp;
#pragma unroll
      for (int ds = 0; ds < DS; ++ds) ka[jh][ds] = bload(kr, voff, 64 * ds);
    }
    f32x4 sc[4][2];
#pragma unroll
    for (int jh = 0; jh < 4; ++jh) {
      sc[jh][0] = sc[jh][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ds = 0; ds < DS; ++ds) {
        sc[jh][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka[jh][ds], qb[0][ds], sc[jh][0], 0, 0, 0);
        sc[jh][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka[jh][ds], qb[1][ds], sc[jh][1], 0, 0, 0);
      }
    }
    // The K registers are free: the Vt operands load during the softmax.
    f16x8 va[DT][2];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int j = 0; j < 2; ++j) va[dt][j] = bload(vr, vt_lane + kb * 2, (16 * dt * a.s64 + 32 * j) * 2);
    // Lane (query column, group grp) holds keys kb + 32j + 8grp + 4h + v.
    f16x8 pb[2][2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int qi = q0 + 16 * nt + col;
      float mx = -INFINITY;
#pragma unroll
      for (int jh = 0; jh < 4; ++jh)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int key = kb + 32 * (jh >> 1) + 8 * grp + 4 * (jh & 1) + v;
          bool keep = key < a.Skv && qi < a.Sq;
          if (a.causal) keep = keep && key <= qi;
          float x = sc[jh][nt][v] * a.scale_log2;
          if constexpr (MK != kNoMask) x += bias_of<MK>(mrow[nt][min(key, a.Skv - 1) * m_sk]);
          x = keep ? x : -INFINITY;
          sc[jh][nt][v] = x;
          mx = fmaxf(mx, x);
        }
      mx = fmaxf(mx, wave_xor(mx, 16));
      mx = fmaxf(mx, wave_xor(mx, 32));
      const float m_new = fmaxf(m_run[nt], mx);
      const float m_use = m_new == -INFINITY ? 0.f : m_new;  // all masked so far: p = 0
      const float alpha = fast_exp2(m_run[nt] - m_use);
      float psum = 0.f;
#pragma unroll
      for (int jh = 0; jh < 4; ++jh)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float p = fast_exp2(sc[jh][nt][v] - m_use);
          psum += p;
          pb[nt][jh >> 1][(jh & 1) * 4 + v] = static_cast<_Float16>(p);
        }
      l_run[nt] = l_run[nt] * alpha + psum;
      m_run[nt] = m_new;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[nt][dt] *= alpha;
    }
    // O^T += Vt[d, keys] P^T[keys, q]; Vt is zero past Skv (up to s64).
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        o[0][dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[dt][j], pb[0][j], o[0][dt], 0, 0, 0);
        o[1][dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[dt][j], pb[1][j], o[1][dt], 0, 0, 0);
      }
  }

  // Lane (query column, group grp) holds O^T[d = 16dt + 4grp + v][q].
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    float l = l_run[nt];
    l += wave_xor(l, 16);
    l += wave_xor(l, 32);
    const int qi = q0 + 16 * nt + col;
    if (qi >= a.Sq) continue;
    _Float16* op = a.out + ((static_cast<int64_t>(b) * a.Sq + qi) * a.Hq + h) * D;
    const float inv = l > 0.f ? 1.f / l : 0.f;  // every key masked: zeros
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      f16x4 r;
#pragma unroll
      for (int v = 0; v < 4; ++v) r[v] = static_cast<_Float16>(o[nt][dt][v] * inv);
      *reinterpret_cast<f16x4*>(op + 16 * dt + 4 * grp) = r;
    }
    if (a.lse && grp == 0)
      a.lse[(static_cast<int64_t>(b) * a.Hq + h) * a.Sq + qi] =
          l > 0.f ? (m_run[nt] + log2f(l)) * kLn2 : -INFINITY;
  }
}

// ---- 3. attention with K/V tiles shared through LDS -------------------------
//
// A workgroup of W = 8 or 4 wavefronts takes W x 32 queries of one (sequence,
// q head), wavefront w 32 of them (or, in half steps, W / 2 x 32 queries;
// which of them a call runs: pick_shape).  Per 64-key step t the workgroup
// stages the K tile and the V tile, both [64 keys][D] as K and V lie in
// memory, in LDS, and every wavefront reads its MFMA operands from there:
//   S^T[key, q] = K Q^T   2 x D/16 MFMA 32x32x16 (M = 32 keys, N = 32 queries)
//   O^T[d, q] += V^T P^T  D/32 x 4 MFMA 32x32x16
// The V^T operand (8 consecutive keys of one feature per lane) comes from
// the row-major V tile through the transposing LDS read ds_read_b64_tr_b16,
// so V needs no relayout before the kernel.
// The loop is software-pipelined: K runs one step ahead of V, so while the
// VALU computes step t's softmax the matrix cores already compute step
// t+1's scores and then step t's P V.  Two LDS slots each hold K(t+1) /
// K(t+2) and V(t) / V(t+1); the next tiles travel from L2 straight into
// LDS during a step's math.  The 16-byte units of an LDS row are exchanged so
// that those one operand read touches fall in distinct banks (Lds2).  Workgroups are
// numbered so that those of one (sequence, KV head) run on one XCD (one L2),
// and for causal attention each head's latest (heaviest) query block starts
// first.

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef short v4i16 __attribute__((ext_vector_type(4)));

constexpr int kWaves2 = 8;
constexpr int kThreads2 = kWaves2 * 64;
constexpr int kQW = 32;             // queries per wavefront
constexpr int kQB = kWaves2 * kQW;  // rows of the largest workgroup
constexpr int kKT = 64;             // keys per step
static_assert(kStick % kKT == 0, "the Vt padding must cover whole steps");
constexpr int kPadH = 8;            // LDS row padding, halves (16 bytes)
constexpr int kPrefetch = 4;        // LDS operand reads in flight ahead of the MFMA using them

// K and V tiles in LDS: rows of D halves, unpadded (two workgroups of W = 4
// per compute unit then have 80 KB each, masks included, and a step's tiles
// are 32 loads at D 128 where padded rows took 37), the 16-byte units of a
// row exchanged by an XOR of their index with a function of the row.  Against
// padded rows: 4096 x 4096 249.9 -> 246.5 us, causal 137.9 -> 135.6, D 64 (4 x 16
// heads x 2048) 88.6 -> 86.1, fp16 mask [4096, 4096] 292.9 -> 284.7.
template <int D>
struct Lds2 {
  static constexpr int kTile = kKT * D;    // halves
  static constexpr int kSlot = 2 * kTile;  // one slot: a K tile and a V tile
  static constexpr int kUnits = D / 8;     // 16-byte units per row
  // K: the 16 lanes an operand read serves at once read the same unit of 16
  // rows (key32_of of 16 consecutive rho); the XOR puts them in 16 distinct
  // units of the 256 bytes that LDS's 64 banks hold.
  __device__ static __forceinline__ int swz_k(int row) { return D == 128 ? row & 15 : (row >> 1) & 7; }
  // V: a transposed read serves 32 lanes at once, 4 consecutive rows x 64
  // bytes; the XOR moves whole 64-byte groups, to four distinct ones.
  __device__ static __forceinline__ int swz_v(int row) { return D == 128 ? 4 * (row & 3) : 4 * ((row >> 1) & 1); }
};

// The 16 bytes x without its first n (n < 16), zeros behind.
__device__ __forceinline__ u32x4 drop_bytes(u32x4 x, int n) {
  uint64_t w[2];
  __builtin_memcpy(w, &x, 16);
  if (n >= 8) {
    w[0] = w[1] >> (8 * (n - 8));
    w[1] = 0;
  } else if (n > 0) {
    w[0] = w[0] >> (8 * n) | w[1] << (64 - 8 * n);
    w[1] >>= 8 * n;
  }
  __builtin_memcpy(&x, w, 16);
  return x;
}

// S^T row rho of a 32-key half maps to key key32_of(rho) of that half: MFMA
// row tile i (8 rows) of lane half h holds rows 8i + 4h + v (i, v < 4); they
// are the keys 16(i/2) + 8h + 4(i%2) + v, i.e. the two 8-key runs the PV
// operand of half h needs.
__device__ __forceinline__ int key32_of(int rho) {
  const int i = rho >> 3, h = (rho >> 2) & 1, v = rho & 3;
  return 16 * (i >> 1) + 8 * h + 4 * (i & 1) + v;
}

// max(x of lane l, x of lane l ^ 32), in every lane.
__device__ __forceinline__ float max_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, x),
                                                  false, false);
  return fmaxf(__builtin_bit_cast(float, static_cast<unsigned>(r[0])),
               __builtin_bit_cast(float, static_cast<unsigned>(r[1])));
}

// The same, NaN if either is.
__device__ __forceinline__ float maximum_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, x),
                                                  false, false);
  return __builtin_elementwise_maximum(__builtin_bit_cast(float, static_cast<unsigned>(r[0])),
                                       __builtin_bit_cast(float, static_cast<unsigned>(r[1])));
}

__device__ __forceinline__ float sum_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, x),
                                                  false, false);
  return __builtin_bit_cast(float, static_cast<unsigned>(r[0])) + __builtin_bit_cast(float, static_cast<unsigned>(r[1]));
}

struct Fwd2Args {
  const _Float16* q;
  const _Float16* k;
  const _Float16* v;
  const void* mask;          // fp16 / fp32 bias or uint8 keep-mask, keys contiguous
  int64_t m_sb, m_sh, m_sq;  // elements
  uint32_t m_bytes;          // extent of one block's `pack` q heads of the mask
  int m_wide;                // fp32: rows of whole 16-byte units, loaded as such
  int64_t q_sb, q_sh, q_ss;
  int64_t k_sb, k_sh, k_ss;
  int64_t v_sb, v_sh, v_ss;
  _Float16* out;
  float* lse;
  int B, Hq, Hkv, g, Sq, Skv, causal, qblocks;
  // Rows per query: 1, or (Sq < 256) the g q heads of a KV head, which then
  // share each K / V tile; gp = g / pack.
  int pack, gp;
  // Key split (calls without the causal flag whose blocks would not fill
  // the device): block sp attends keys sp * split_keys .. + split_keys
  // - 1 and writes its fp32 partial (O, row max, row sum) to part; a merge
  // pass combines them.  nsplit == 1: no split.
  int nsplit, split_keys;
  float* part;
  // sdpa_decode_short_kernel's key split: this call's arrival-flag value
  // (nonzero, a new one per call).
  uint32_t ticket;
  uint32_t n_items;
  int xcd_remap;
  float scale_log2;
  // The divisors of the block index and of a row's (query, head), as
  // multiply-high divisions: as integer divisions they cost ~30 instructions
  // each before a block's first load.
  spyre_hip::FastDiv by_split, by_gp, by_qblocks, by_hkv, by_pack;
};

// A wavefront's mask block for one step: its 32 rows x the step's 64 keys
// (HALF: the 32 keys of its half), staged in LDS by buffer loads like the K /
// V tiles, the 16-byte units of a row exchanged like K's.
template <int ESZ, int KEYS> struct MaskRows {
  static constexpr int kEsz = ESZ;
  static constexpr int kU = KEYS * ESZ / 16;  // 16-byte units of a row
  static constexpr int kLoads = 32 * kU / 64, kBytes = 32 * kU * 16;
  __device__ static __forceinline__ int swz(int row) { return (row / (16 / kU)) & (kU - 1); }
};
template <int MK, bool HALF>
struct MaskTile : MaskRows<MK == kMaskF32 ? 4 : MK == kMaskF16 ? 2 : 1, HALF ? 32 : 64> {};
template <bool HALF> struct MaskTile<kNoMask, HALF> {
  static constexpr int kEsz = 1, kU = 1, kLoads = 0, kBytes = 0;
};

// PRESCALED (|scale log2 e| <= 1, so q * that never overflows fp16): Q is
// multiplied by scale log2 e once, and every step's scores leave the MFMA
// already as exponents: the first QK MFMA starts from a tile holding -m
// (the running max), so P = exp2(S) needs no per-score FMA.  Otherwise the
// scale's sign is folded into Q and its magnitude into the exponent's FMA.
// SLOTS: K / V slots in LDS.  Two: each step's tiles are loaded one step
// ahead, a barrier per step.  Four (kHalf8 calls without a mask, e.g. decode, where one wavefront computes and the
// step waits on its loads): loads two steps ahead, a barrier per two steps.
// HALF (blocks of at most 128 rows, e.g. decode): wavefronts 2r and 2r + 1
// share row tile r and take one 32-key half of every step each; the pair's
// partials are folded in LDS at the end.
// ANY (fp16 / boolean masks in half steps): rows of any alignment and length,
// at least 16 bytes, through registers by ordinary loads and stores to the
// mask block at the step's end.  Copied first with 16-byte rows, they cost
// a launch and two passes: 32 heads, D 128, 1001 x 1001, fp16 63.6 -> 36.8 us,
// boolean [1001, 1001] 35.1 -> 32.2; 333 x 333 boolean 16.0 -> 13.1; 4 x 16 heads
// x 150, D 64, boolean 11.3 -> 8.2.  A kernel of its own: behind a flag the loads'
// registers cost the others (2 x 12 heads x 512, D 64, boolean 9.7 -> 11.1).
// fp32 rows this way instead of 4 bytes a lane: 21.7 -> 34.6 (2 x 16 heads x
// 777, D 64).
template <int D, bool PRESCALED, int MK, int SLOTS, bool HALF, int W, bool ANY = false>
__global__ __launch_bounds__(W * 64, 2) void sdpa_fwd_lds_kernel(Fwd2Args a) {
  static_assert(SLOTS == 2 || (SLOTS == 4 && HALF && MK == kNoMask), "four slots: half steps without a mask");
  // fp32 biases: half steps only (the 32-query block of a full step, 8 KB a
  // wavefront, leaves no room beside K and V), scores scaled and biased in
  // fp32 (log2 units), row sums of the fp32 probabilities and a running max
  // that follows every new one (a row's largest probability is then exactly
  // 1 in fp16), as the per-wavefront kernel has them: the same error, 2.6e-4
  // of fp64 at S 777, D 64 (2.9e-4 with the lazy max).
  constexpr bool F32M = MK == kMaskF32;
  constexpr float kLazy = F32M ? 0.f : 8.f;  // half steps: how far a score may pass the running max
  static_assert(!F32M || (HALF && !PRESCALED), "fp32 biases: half steps, q as it is");
  using L = Lds2<D>;
  using MT = MaskTile<MK, HALF>;
  constexpr int DK = D / 16;  // QK k-steps
  constexpr int DM = D / 32;  // O row tiles
  // The K / V slots, then (masked calls) two mask blocks per wavefront, or
  // one where two would not leave room for a second workgroup of W = 4.
  constexpr int kMaskSlots = MK != kNoMask && W == 4 && SLOTS * L::kSlot * 2 + 2 * W * MT::kBytes > 80 * 1024 ? 1 : 2;
  __shared__ __align__(16) _Float16 lds[SLOTS * L::kSlot + kMaskSlots * W * MT::kBytes / 2];

  // item = ((b * Hkv + kvh) * qblocks + (qblocks - 1 - qb)) * gp + gi: the
  // blocks of one (sequence, KV head) are consecutive, latest query block
  // (longest, under causal masking) first across its g q heads.
  // With pack > 1 a block's rows are (query, q head) pairs of one KV head,
  // row = query * pack + head in group.
  uint32_t item = blockIdx.x;
  if (a.xcd_remap) item = (item % 8) * (a.n_items / 8) + item / 8;
  const int pack = a.pack;
  const uint32_t i1 = fdiv(item, a.by_split), i2 = fdiv(i1, a.by_gp), i3 = fdiv(i2, a.by_qblocks);
  const uint32_t bq = fdiv(i3, a.by_hkv);
  const int sp = static_cast<int>(item - i1 * a.nsplit);
  const int gi = static_cast<int>(i1 - i2 * a.gp);
  const int qb = a.qblocks - 1 - static_cast<int>(i2 - i3 * a.qblocks);
  const int kvh = static_cast<int>(i3 - bq * a.Hkv);
  const int b = static_cast<int>(bq);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  __builtin_assume(wave >= 0 && wave < W);  // lets the compiler drop always-true load guards
  const int hw = HALF ? (wave & 1) : 0;  // HALF: the key half of each step
  constexpr int kRows = (HALF ? W / 2 : W) * kQW;
  const int qw0 = qb * kRows, q0 = qw0 + (HALF ? (wave >> 1) : wave) * kQW;  // rows
  const int col = lane & 31, half = lane >> 5;
  const int qrow = q0 + col;
  const int qi = static_cast<int>(fdiv(qrow, a.by_pack));  // this lane's query
  // Block gi of the KV head holds q heads gi * pack .. gi * pack + pack - 1.
  const int h = kvh * a.g + gi * pack + (qrow - qi * pack);
  const bool q_ok = qi < a.Sq;
  // The wavefront's first and last query, and the block's last.
  const int q_lo = static_cast<int>(fdiv(q0, a.by_pack));
  const int q_hi = static_cast<int>(fdiv(q0 + kQW - 1, a.by_pack));
  const int qb_hi = static_cast<int>(fdiv(qw0 + kRows - 1, a.by_pack));

  // Q^T operand: lane (query column, half) holds features 16ks + 8half .. +8.
  f16x8 qv[DK];
  {
    const _Float16* qp = a.q + b * a.q_sb + h * a.q_sh + static_cast<int64_t>(min(qi, a.Sq - 1)) * a.q_ss + 8 * half;
#pragma unroll
    for (int ks = 0; ks < DK; ++ks) {
      qv[ks] = q_ok ? *reinterpret_cast<const f16x8*>(qp + 16 * ks) : f16x8{};
      if constexpr (PRESCALED) {
#pragma unroll
        for (int e = 0; e < 8; ++e) qv[ks][e] = static_cast<_Float16>(static_cast<float>(qv[ks][e]) * a.scale_log2);
      } else if (a.scale_log2 < 0.f) {
        qv[ks] = -qv[ks];  // the scale's sign, exactly
      }
    }
    // Wait for Q here, outside the loop: otherwise the first MFMA of every
    // step also waits for the next tiles' loads, which are then in flight.
#pragma unroll
    for (int ks = 0; ks < DK; ++ks) asm volatile("" : : "v"(qv[ks]));
  }
  const _Float16* kbase = a.k + b * a.k_sb + kvh * a.k_sh;
  const _Float16* vbase = a.v + b * a.v_sb + kvh * a.v_sh;

  // Tiles move from L2 straight into LDS (buffer loads with the LDS flag):
  // lane l of a load writes the 16 bytes at M0 + 16 l, so load i of a tile
  // fills its 16-byte units 64 i .. 64 i + 63.  Lane l of load i fetches the
  // unit's source (the row's unit that the XOR puts there); K / V rows past
  // Skv lie past the buffer's range and are written as zeros.  Per-lane
  // offsets are fixed for the whole loop; the step only moves the base.
  constexpr int kU = L::kUnits, kJ = kU / W;  // loads per tile, and per wavefront
  static_assert(kU % W == 0, "every wavefront loads as much");
  constexpr uint32_t kOob = 0x80000000u;  // past kBufRange
  uint32_t k_off[kJ], v_off[kJ];
#pragma unroll
  for (int j = 0; j < kJ; ++j) {
    const int u = 64 * (wave + W * j) + lane, row = u / kU, ch = u % kU;
    k_off[j] = (static_cast<uint32_t>(row) * static_cast<uint32_t>(a.k_ss) + 8 * (ch ^ L::swz_k(row))) * 2;
    v_off[j] = (static_cast<uint32_t>(row) * static_cast<uint32_t>(a.v_ss) + 8 * (ch ^ L::swz_v(row))) * 2;
  }
  // K / V tiles load in sequence (K(0), K(1), ... and V(0), V(1), ...), so
  // each has a running cursor: the next tile's first row and the bytes from
  // it to the end of row Skv - 1.  Rows past Skv lie past the descriptor's
  // range and arrive as zeros without a per-lane test (no unit straddles
  // the end: a row's units end within its stride); with a key stride of 0
  // every row reads row 0's bytes, finite values the key test masks.
  const _Float16* k_cur = kbase + static_cast<int64_t>(sp) * a.split_keys * a.k_ss;
  const _Float16* v_cur = vbase + static_cast<int64_t>(sp) * a.split_keys * a.v_ss;
  const int64_t k_tile = static_cast<int64_t>(kKT) * a.k_ss, v_tile = static_cast<int64_t>(kKT) * a.v_ss;
  // Bytes left as 32-bit values: the head's whole span fits one descriptor
  // (< 2 GiB, checked by the host), so a count clamped to kBufRange at the
  // start still covers every valid row and no row past Skv.
  auto left0 = [&](int64_t ss) {
    if (ss == 0) return static_cast<int32_t>(kBufRange);
    const int64_t all = static_cast<int64_t>(a.Skv) * ss * 2;
    return static_cast<int32_t>(min(all, static_cast<int64_t>(kBufRange)) - static_cast<int64_t>(sp) * a.split_keys * ss * 2);
  };
  int32_t k_left = left0(a.k_ss), v_left = left0(a.v_ss);
  const int32_t k_step = static_cast<int32_t>(min(2 * k_tile, static_cast<int64_t>(kBufRange)));
  const int32_t v_step = static_cast<int32_t>(min(2 * v_tile, static_cast<int64_t>(kBufRange)));
  auto range_of = [](int32_t left) { return static_cast<uint32_t>(max(left, 0)); };
  // The next K tile into slot `slot`.
  auto dma_k = [&](int slot) {
    const Rsrc r = make_rsrc(k_cur, range_of(k_left));
#pragma unroll
    for (int j = 0; j < kJ; ++j) load_lds16(r, lds + slot * L::kSlot + 512 * (wave + W * j), k_off[j]);
    k_cur += k_tile;
    k_left -= k_step;
  };
  // The next V tile into slot `slot` (rows past Skv as zeros, so that a
  // masked key's P = 0 never meets stale bits).
  auto dma_v = [&](int slot) {
    const Rsrc r = make_rsrc(v_cur, range_of(v_left));
#pragma unroll
    for (int j = 0; j < kJ; ++j) load_lds16(r, lds + slot * L::kSlot + L::kTile + 512 * (wave + W * j), v_off[j]);
    v_cur += v_tile;
    v_left -= v_step;
  };
  // The wavefront's mask block of keys kb .. kb + 63 (HALF: its 32 of them)
  // into its slot `slot`: rows past Sq and bytes past the block's heads
  // arrive as zeros.  Offsets are from the first of the block's `pack` q
  // heads (a row is a (query, head) pair); the descriptor's range ends with
  // the last of them.
  // fp32 rows need not be whole 16-byte units (nor start on one): those are
  // loaded 4 bytes a lane, two rows of 32 keys per load, whose range check
  // is exact to the key.
  constexpr int kNarrow = F32M ? 16 : 0;  // such loads
  uint32_t m_off[kNarrow > 0 ? kNarrow : MT::kLoads > 0 ? MT::kLoads : 1];
  const char* mbase = nullptr;
  if constexpr (MK != kNoMask) {
    mbase = static_cast<const char*>(a.mask) + (b * a.m_sb + (kvh * a.g + gi * pack) * a.m_sh) * MT::kEsz;
    const uint32_t m_sq = static_cast<uint32_t>(a.m_sq), m_sh = static_cast<uint32_t>(a.m_sh);
    // Byte offset of the wavefront's row `row`, key 32 hw; kOob past Sq.  A
    // valid row's offset lies below m_bytes < 2^31, so 32 bits of each product do.
    auto row_off = [&](int row) -> uint32_t {
      uint32_t mq = q0 + row, at = mq * m_sq;
      if (pack > 1) {
        mq = fdiv(q0 + row, a.by_pack);
        at = mq * m_sq + (q0 + row - mq * pack) * m_sh;
      }
      return static_cast<int>(mq) < a.Sq ? (at + 32 * hw) * MT::kEsz : kOob;
    };
    if (F32M && !a.m_wide) {
#pragma unroll
      for (int j = 0; j < kNarrow; ++j) {
        const int row = 2 * j + half;
        m_off[j] = row_off(row) + (((col >> 2) ^ MT::swz(row)) * 4 + (col & 3)) * 4;
      }
    } else {
#pragma unroll
      for (int j = 0; j < MT::kLoads; ++j) {
        const int u = 64 * j + lane, row = u / MT::kU, ch = (u % MT::kU) ^ MT::swz(row);
        m_off[j] = row_off(row) + 16 * ch;
      }
    }
  }
  auto mask_block = [&](int slot) {
    return lds + SLOTS * L::kSlot + ((kMaskSlots == 2 ? slot : 0) * W + wave) * (MT::kBytes / 2);
  };
  auto dma_m = [&](int kb, int slot) {
    if constexpr (MK != kNoMask) {
      const uint32_t done = static_cast<uint32_t>(kb) * MT::kEsz;  // < Skv esz <= m_bytes
      const Rsrc r = make_rsrc(reinterpret_cast<const _Float16*>(mbase + done), a.m_bytes - done);
      if (F32M && !a.m_wide) {
#pragma unroll
        for (int j = 0; j < kNarrow; ++j) load_lds4(r, mask_block(slot) + 128 * j, m_off[j]);
      } else {
#pragma unroll
        for (int j = 0; j < MT::kLoads; ++j) load_lds16(r, mask_block(slot) + 512 * j, m_off[j]);
      }
    }
  };
  // ANY: the block's units of keys kb .. in registers, and from there to
  // its slot.  A unit that crosses the row's end is read as the row's last 16
  // bytes, shifted (rows have at least 16: the host's check).
  u32x4 m_reg[MT::kLoads > 0 ? MT::kLoads : 1];
  auto read_m = [&](int kb) {
    if constexpr (ANY) {
      const char* p = mbase + static_cast<int64_t>(kb) * MT::kEsz;
#pragma unroll
      for (int j = 0; j < MT::kLoads; ++j) {
        m_reg[j] = u32x4{0, 0, 0, 0};
        if (kb + kKT <= a.Skv) {
          if (m_off[j] < kOob) __builtin_memcpy(&m_reg[j], p + m_off[j], 16);
        } else {
          const int u = 64 * j + lane;
          const int at = (kb + 32 * hw) * MT::kEsz + 16 * ((u % MT::kU) ^ MT::swz(u / MT::kU));  // the unit's bytes in its row
          const int past = at + 16 - a.Skv * MT::kEsz;  // of them past the row
          if (m_off[j] < kOob && past < 16) {
            const int back = max(past, 0);
            __builtin_memcpy(&m_reg[j], p + (static_cast<int64_t>(m_off[j]) - back), 16);
            m_reg[j] = drop_bytes(m_reg[j], back);
          }
        }
      }
    }
  };
  auto write_m = [&](int slot) {
    if constexpr (ANY) {
#pragma unroll
      for (int j = 0; j < MT::kLoads; ++j)
        *reinterpret_cast<u32x4*>(mask_block(slot) + 512 * j + 8 * lane) = m_reg[j];
    }
  };
  // The loads must have landed before the barrier that publishes them.
  auto dma_wait = [] { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };

  // This block's keys: kb0 .. key_end - 1 (the whole row unless split).
  const int kb0 = sp * a.split_keys;
  const int key_end = a.causal ? min(a.Skv, qb_hi + 1) : (a.nsplit > 1 ? min(a.Skv, kb0 + a.split_keys) : a.Skv);
  const int n_tiles = (key_end - kb0 + kKT - 1) / kKT;
  // Step t has work for this wavefront unless all its keys are masked
  // (causal: keys past the wavefront's last query).
  auto active = [&](int t) { return t < n_tiles && q_lo < a.Sq && (!a.causal || kb0 + t * kKT <= q_hi); };
  // Only steps crossing Skv or the causal diagonal need the key test.
  auto edge = [&](int t) { return kb0 + t * kKT + kKT > a.Skv || (a.causal && kb0 + t * kKT + kKT - 1 > q_lo); };
  // |scale| (its sign is folded into Q), kept above 0 so that masked scores
  // (-inf) stay -inf; a scale of 0 then gives the uniform weights it should.
  const float scale_abs = fmaxf(fabsf(a.scale_log2), 1e-30f);
  float m_run = -INFINITY, l_run = 0.f;
  // PRESCALED: scores are carried relative to m_use (m_run, or 0 while no
  // finite score has been seen); neg_m_tile holds -m_use in every row.
  // fp16 biases: 0 too while m_run is below kLow, a row's dropped keys at the
  // type's lowest number (about -94500 here, where fp32 steps by 2^-7): the
  // scores of its first kept keys would be accumulated there.  Relative
  // error of 300 keys, the last 40 of them kept: 4.3e-3, with this 3.6e-4.
  constexpr bool kClamp = PRESCALED && MK == kMaskF16;
  constexpr float kLow = -1024.f;
  float m_use = 0.f;
  bool low = false;  // some row's m_run is below kLow
  auto reference = [&](float m) {  // m_use for m_run = m
    if (kClamp) low = __builtin_amdgcn_ballot_w64(m < kLow && m > -INFINITY) != 0;
    return m == -INFINITY || (kClamp && m < kLow) ? 0.f : m;
  };
  f32x16 neg_m_tile = f32x16{};
  f32x16 o[DM];
#pragma unroll
  for (int dm = 0; dm < DM; ++dm) o[dm] = f32x16{};

  auto lds_at = [&](uint32_t byte) { return reinterpret_cast<const char*>(lds) + byte; };
  // This lane's K operands in a K tile: row key32_of(col) of a 32-key half,
  // unit 2 ks + half of k-step ks, at byte k_lane ^ (32 ks) + 64 D mt.
  const uint32_t k_lane = static_cast<uint32_t>(key32_of(col) * D * 2 + ((half ^ L::swz_k(key32_of(col))) * 16));
  auto k_frag = [&](uint32_t kt, int mt, int ks) -> f16x8 {  // kt: the tile's byte + k_lane
    return *reinterpret_cast<const f16x8*>(lds_at((kt ^ (32 * ks)) + mt * 32 * D * 2));
  };
  // S^T half mt (keys 32mt .. 32mt + 31 of the step) from K tile 0 of slot 0.
  auto qk = [&](int mt) {
    f32x16 acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(k_frag(k_lane, mt, 0), qv[0],
                                                        PRESCALED ? neg_m_tile : f32x16{}, 0, 0, 0);
#pragma unroll
    for (int ks = 1; ks < DK; ++ks)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(k_frag(k_lane, mt, ks), qv[ks], acc, 0, 0, 0);
    return acc;
  };
  // Lane (query column, half) holds S^T rows 8i + 4half + v of each 32-key
  // half (register 4i + v).  Masked scores become -inf.
  const int key_last = a.causal ? min(a.Skv - 1, qi) : a.Skv - 1;  // this lane's last visible key
  auto mask_step = [&](int t, f32x16 (&s)[2]) {
    const int kl = key_last - (kb0 + t * kKT) - 8 * half;  // key32_of adds 8 per lane half
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) {
        const int kr = mt * 32 + key32_of(8 * (rr >> 2) + (rr & 3));  // key - t kKT - 8 half
        s[mt][rr] = kr <= kl ? s[mt][rr] : -INFINITY;
      }
  };
  // The step's mask from the wavefront's block in LDS: registers 4i + v of
  // half mt are keys 32 mt + 16 (i / 2) + 8 half + 4 (i % 2) + v of query
  // col, four consecutive keys per read.  A bias is added in the scores'
  // units (PRESCALED: log2 units, else divided by |scale|), a keep-mask
  // sends dropped scores to -inf.
  const float bias_mul = PRESCALED ? kLog2e : kLog2e / scale_abs;
  // This lane's byte of the block: row col, its first key's unit (fp16: unit
  // `half`; fp32: unit 2 half; boolean: byte 8 half of unit 0).
  uint32_t m_lane = 0;
  if constexpr (MK == kMaskF16) m_lane = col * (16 * MT::kU) + ((half ^ MT::swz(col)) * 16);
  if constexpr (F32M) m_lane = col * (16 * MT::kU) + (((2 * half) ^ MT::swz(col)) * 16);
  if constexpr (MK == kMaskBool) m_lane = col * (16 * MT::kU) + MT::swz(col) * 16 + 8 * half;
  // Half mt of the mask block (HALF: its one half, mt 0) onto S half s.
  auto apply_mask_half = [&](int t, int mt, f32x16& s) {
    if constexpr (MK != kNoMask) {
      const char* blk = reinterpret_cast<const char*>(mask_block(t & 1));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // keys 32 mt + 16 (i / 2) + 8 half + 4 (i % 2) .. + 3 of row col
        if constexpr (F32M) {
          const uint32_t at = m_lane ^ (64 * (i >> 1) + 16 * (i & 1));
          const f32x4 m4 = *reinterpret_cast<const f32x4*>(blk + at);
#pragma unroll
          for (int v = 0; v < 4; ++v) s[4 * i + v] = __builtin_fmaf(s[4 * i + v], scale_abs, m4[v] * kLog2e);
        } else if constexpr (MK == kMaskF16) {
          const uint32_t at = (m_lane ^ (64 * mt + 32 * (i >> 1))) + 8 * (i & 1);
          const f16x4 m4 = *reinterpret_cast<const f16x4*>(blk + at);
#pragma unroll
          for (int v = 0; v < 4; ++v) s[4 * i + v] = __builtin_fmaf(static_cast<float>(m4[v]), bias_mul, s[4 * i + v]);
        } else {
          const uint32_t at = (m_lane ^ (32 * mt + 16 * (i >> 1))) + 4 * (i & 1);
          const uint32_t m4 = *reinterpret_cast<const uint32_t*>(blk + at);
#pragma unroll
          for (int v = 0; v < 4; ++v) s[4 * i + v] = ((m4 >> (8 * v)) & 0xffu) != 0 ? s[4 * i + v] : -INFINITY;
        }
      }
    }
  };
  // One mask block per wavefront: the next step's loads go out once this
  // step's reads have returned.
  auto next_mask = [&](int t) {
    if constexpr (MK != kNoMask && kMaskSlots == 1) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (t + 1 < n_tiles && !ANY) dma_m(kb0 + (t + 1) * kKT, 0);
    }
  };
  auto apply_mask = [&](int t, f32x16 (&s)[2]) {
    apply_mask_half(t, 0, s[0]);
    apply_mask_half(t, 1, s[1]);
    next_mask(t);
  };
  // The running max (log2 domain) moves only when a score of the step
  // exceeds it by more than 2^8, so P <= 256 (fine in fp16) and most steps
  // skip the rescale of O; O / l is exact whatever max is used.
  // PRESCALED: s holds exponents relative to m_use, and so does `ahead`
  // (the next step's scores, computed before this update); a move of m_use
  // shifts both, and the tile.
  // The step's row max in the units of m_run.
  // Masked: NaN if a score is, so that a NaN does not leave its step blank.
  auto max_of = [](float x, float y) {
    if constexpr (MK != kNoMask)
      return __builtin_elementwise_maximum(x, y);
    else
      return fmaxf(x, y);
  };
  auto max_halves = [](float x) {
    if constexpr (MK != kNoMask)
      return maximum_xor32(x);
    else
      return max_xor32(x);
  };
  auto row_max = [&](const f32x16 (&s)[2]) {
    float mx = -INFINITY;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) mx = max_of(mx, s[mt][rr]);
    return PRESCALED ? max_halves(mx) + m_use : max_halves(mx) * scale_abs;
  };
  // Whether a masked step adds anything to a real row: mx is this lane's row
  // max (of both lane halves).  A NaN does.  Boolean masks leave none on a
  // dropped key; an fp16 bias may (a cache's unused keys), so in a step where
  // no row has a number that adds something, a NaN row counts only if it
  // keeps a key, i.e. has a bias other than one that alone makes the weight 0
  // (-inf, the type's lowest number).  Read from memory, since the block in
  // LDS may be the next step's by now.
  auto adds = [&](int t, float mx) {
    const float least = fmaxf(m_run - 32.f, -__FLT_MAX__);  // (-inf is below it)
    if constexpr (MK != kMaskF16) return __builtin_amdgcn_ballot_w64(q_ok && !(mx < least)) != 0;
    bool any = __builtin_amdgcn_ballot_w64(q_ok && mx >= least) != 0;
    if (__builtin_expect(!any && __builtin_amdgcn_ballot_w64(q_ok && mx != mx) != 0, 0)) {
      constexpr float kDropped = -1024.f;
      const int at = kb0 + t * kKT + (HALF ? 32 * hw : 0) + 8 * half, n = HALF ? 2 : 4;
      bool keeps = false;
      if (q_ok) {
        const _Float16* row = static_cast<const _Float16*>(a.mask) + b * a.m_sb + h * a.m_sh + qi * a.m_sq + at;
#pragma unroll 1
        for (int k = 0; k < 16 * n; ++k)  // this lane's: 8 of every 16 keys
          keeps = keeps || ((k & 8) == 0 && at + k <= key_last && !(static_cast<float>(row[k]) <= kDropped));
      }
      any = __builtin_amdgcn_ballot_w64(q_ok && mx != mx && keeps) != 0;
    }
    return any;
  };
  // Masked full steps: s is S(t), ahead S(t+1), both complete.
  auto update_max = [&](f32x16 (&s)[2], f32x16 (&ahead)[2], float mx) {
    if (__builtin_amdgcn_ballot_w64(mx > m_run + 8.f) != 0) {
      const float m_new = fmaxf(m_run, mx);
      const float alpha = m_new == -INFINITY ? 1.f : fast_exp2(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int dm = 0; dm < DM; ++dm) o[dm] *= alpha;
      m_run = m_new;
      if constexpr (PRESCALED) {
        const float m_use_new = reference(m_new);
        const float d = m_use_new - m_use;
        m_use = m_use_new;
#pragma unroll
        for (int rr = 0; rr < 16; ++rr) {
          s[0][rr] -= d;
          s[1][rr] -= d;
          ahead[0][rr] -= d;
          ahead[1][rr] -= d;
          neg_m_tile[rr] = -m_use;
        }
      }
    }
  };
  // kClamp: the scores of rows below kLow made relative to m_run, which they
  // are not carried against.
  auto rebase = [&](f32x16& s) {
    if (kClamp && __builtin_expect(low, 0)) {
      const float d = m_use - (m_run == -INFINITY ? m_use : m_run);  // 0 in the other rows
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) s[rr] += d;
    }
  };
  // P (fp16) of half mt; the row sum adds the same fp16 values the PV
  // product uses (fp32 biases: the fp32 values).
  auto softmax_half = [&](const f32x16& s, float neg_m, f16x8 (&pb)[2]) {
    float psum = 0.f;
#pragma unroll
    for (int rr = 0; rr < 16; ++rr) {
      const float p = fast_exp2(PRESCALED ? s[rr] : F32M ? s[rr] + neg_m : __builtin_fmaf(s[rr], scale_abs, neg_m));
      const int i = rr >> 2;  // masked: 0
      pb[i >> 1][(i & 1) * 4 + (rr & 3)] = static_cast<_Float16>(p);
      if constexpr (F32M) psum += p;
    }
#pragma unroll
    for (int j = 0; j < 2 && !F32M; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        psum = __builtin_amdgcn_fdot2(f16x2{pb[j][2 * e], pb[j][2 * e + 1]}, f16x2{1, 1}, psum, false);
    l_run += psum;
  };
  // P (fp16) of S^T registers 8j .. 8j + 7 of a half: the B operand of the
  // half's PV k-step j.  Returns the sum of the same fp16 values.
  auto softmax_q = [&](const f32x16& s, int j, float neg_m, f16x8& pb) -> float {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int rr = 8 * j + e;
      pb[e] = static_cast<_Float16>(fast_exp2(PRESCALED ? s[rr] : __builtin_fmaf(s[rr], scale_abs, neg_m)));
    }
    float psum = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      psum = __builtin_amdgcn_fdot2(f16x2{pb[2 * e], pb[2 * e + 1]}, f16x2{1, 1}, psum, false);
    return psum;
  };
  // A move of the running max to m_new = max(m_run, mx): O and l rescaled;
  // PRESCALED: S(t) and S(t+1) shifted with m_use, and the -m tile.
  auto rescale = [&](f32x16 (&s)[2], f32x16 (&ahead)[2], float mx) {
    const float m_new = fmaxf(m_run, mx);
    const float alpha = m_new == -INFINITY ? 1.f : fast_exp2(m_run - m_new);
    l_run *= alpha;
#pragma unroll
    for (int dm = 0; dm < DM; ++dm) o[dm] *= alpha;
    m_run = m_new;
    if constexpr (PRESCALED) {
      const float m_use_new = m_new == -INFINITY ? m_use : m_new;  // lanes still without a score keep 0
      const float d = m_use_new - m_use;
      m_use = m_use_new;
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) {
        s[0][rr] -= d;
        s[1][rr] -= d;
        ahead[0][rr] -= d;
        ahead[1][rr] -= d;
        neg_m_tile[rr] = -m_use;
      }
    }
  };
  // The 2 DK + 4 DM MFMAs of a step in issue order, each with its LDS operand
  // fragment: 0 .. 2DK-1 the K operands of S(t+1) (half i / DK, k-step
  // i % DK), then the V^T operands of O^T += V^T P^T (two transposed reads
  // each), k-steps (half, j) = c / 2, c % 2 for c = (i - 2DK) / DM, O row tile
  // dm = (i - 2DK) % DM.
  // Each fragment is read kPrefetch MFMAs before its use: with reads issued
  // only just ahead, every MFMA waited out an LDS read.
  constexpr int kNF = 2 * DK + 4 * DM;
  // Within each 16 lanes, lane s reads V[key 8 half + s / 4][d 16 (lane / 16 % 2) + 4 (s % 4)
  // .. + 3]; ds_read_b64_tr_b16 hands lane j of the 16 the four keys of column d + j.
  const int v_row = 8 * half + ((lane & 15) >> 2);
  const uint32_t v_lane = static_cast<uint32_t>(L::kTile * 2 + v_row * D * 2 + L::swz_v(v_row) * 16 +
                                                32 * ((lane >> 4) & 1) + 8 * (lane & 3));
  // Half steps: the step's LDS bytes of this lane's K and V operands, the XOR
  // of a k-step or O row tile applied at each read (their registers have
  // room for two workgroups anyway, their time is latency).  Full steps: every
  // such byte in a register of its own for the whole loop, the slot (the
  // step's parity) in the reads' immediate offset -- the XORs in an
  // issue-bound loop cost 2-9 % (4096 causal 136.1 -> 145.1 us).  Hidden
  // from the compiler either way: it would pair reads whose addresses are 32
  // bytes apart and issue the earlier one late, beside the later one.
  uint32_t k_cur_lds, v_cur_lds, k_at[DK], v_at[DM];
  if constexpr (!HALF) {
#pragma unroll
    for (int ks = 0; ks < DK; ++ks) {
      k_at[ks] = k_lane ^ (32 * ks);
      asm volatile("" : "+v"(k_at[ks]));
    }
#pragma unroll
    for (int dm = 0; dm < DM; ++dm) {
      v_at[dm] = v_lane ^ (64 * dm);
      asm volatile("" : "+v"(v_at[dm]));
    }
  }
  auto step_lds = [&](int t) {
    k_cur_lds = static_cast<uint32_t>(((t + 1) % SLOTS) * L::kSlot * 2) + k_lane;
    v_cur_lds = static_cast<uint32_t>((t % SLOTS) * L::kSlot * 2) + v_lane;
    asm volatile("" : "+v"(k_cur_lds), "+v"(v_cur_lds));
  };
  // V^T operand at LDS byte `at` (of c = 0): keys 16 c + 8 half .. + 7 of one
  // feature per lane (rows + 4 have the XOR of rows + 0).
  auto v_frag = [&](uint32_t at, int c) -> f16x8 {
    const char* p = lds_at(at + 16 * c * D * 2);
    const v4i16 lo = tr_read4(reinterpret_cast<const _Float16*>(p)),
                hi = tr_read4(reinterpret_cast<const _Float16*>(p + 4 * D * 2));
    return __builtin_bit_cast(f16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  // Fragment i of a full step of parity par (K(t+1) in slot 1 - par, V(t) in
  // slot par).
  auto frag = [&](int par, int i) -> f16x8 {
    if (i < 2 * DK)  // the two halves' chains alternate
      return *reinterpret_cast<const f16x8*>(
          lds_at(k_at[i / 2] + (1 - par) * L::kSlot * 2 + (i % 2) * 32 * D * 2));
    return v_frag(v_at[(i - 2 * DK) % DM] + par * L::kSlot * 2, (i - 2 * DK) / DM);
  };
  // Keeps a region's operand reads interleaved one per MFMA (n of each).
  // Keeps a region's operand reads interleaved with its MFMAs i0 .. i1 - 1:
  // each MFMA, then the reads of the fragment kPrefetch ahead (two for a V
  // fragment).
  auto interleave_reads = [](int i0, int i1) {
    for (int i = i0; i < i1; ++i) {
      const int f = i + kPrefetch;
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
      if (f < 2 * DK)
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read (K)
      else if (f < kNF)
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // two (V, transposed)
    }
  };

  // Interleaves MFMAs i0 .. i1 - 1 with the rest of their region: after
  // each MFMA the reads of the fragment kPrefetch ahead, then te (after the
  // region's even MFMAs) or to (odd) transcendental and nv other VALU
  // instructions.
  auto interleave_mix = [](int i0, int i1, int te, int to, int nv) {
    for (int i = i0; i < i1; ++i) {
      const int f = i + kPrefetch;
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
      if (f < 2 * DK)
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read (K)
      else if (f < kNF)
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // two (V, transposed)
      const int nt = (i - i0) % 2 == 0 ? te : to;
      if (nt == 1) __builtin_amdgcn_sched_group_barrier(0x400, 1, 0);  // transcendental
      if (nt == 2) __builtin_amdgcn_sched_group_barrier(0x400, 2, 0);
      if (nv == 1) __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);  // other VALU
      if (nv == 2) __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
      if (nv == 3) __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
      if (nv == 4) __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
    }
  };

  // HALF: the wavefront's S tile (keys 32 hw .. 32 hw + 31 of the step)
  // lives in slot 0 of cur / nxt; its fragments are K half hw (vi < DK) and
  // the V^T operands of keys 32 hw .. + 31 (vi - DK = j DM + dm).
  constexpr int kNFH = DK + 2 * DM;
  auto frag_h = [&](int vi) -> f16x8 {
    if (vi < DK) return *reinterpret_cast<const f16x8*>(lds_at((k_cur_lds ^ (32 * vi)) + hw * 32 * D * 2));
    return v_frag(v_cur_lds ^ (64 * ((vi - DK) % DM)), 2 * hw + (vi - DK) / DM);
  };
  auto interleave_h = [](int i0, int i1) {
    for (int i = i0; i < i1; ++i) {
      const int f = i + kPrefetch;
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if (f < DK)
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      else if (f < kNFH)
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
  };
  auto step_h = [&](int t, f32x16& cur, f32x16& nxt) {
    if constexpr (SLOTS == 2) {
      if (t + 2 < n_tiles) dma_k(t & 1);
      if (t + 1 < n_tiles) dma_v((t + 1) & 1);
      if (kMaskSlots == 2 && t + 1 < n_tiles && !ANY) dma_m(kb0 + (t + 1) * kKT, (t + 1) & 1);
      if (ANY && t + 1 < n_tiles) read_m(kb0 + (t + 1) * kKT);
    } else if ((t & 1) == 0) {
      // Steps t, t + 1 read K(t+1), K(t+2), V(t), V(t+1) (slot = tile % 4);
      // K(t+3), K(t+4), V(t+2), V(t+3) fill the other four slot halves,
      // whose last readers were steps t - 2 and t - 1, and land by the
      // barrier after step t + 1.
      if (t + 3 < n_tiles) dma_k((t + 3) % 4);
      if (t + 4 < n_tiles) dma_k(t % 4);
      if (t + 2 < n_tiles) dma_v((t + 2) % 4);
      if (t + 3 < n_tiles) dma_v((t + 3) % 4);
    }
    if (active(t)) {
      step_lds(t);
      f16x8 fr[kNFH];
#pragma unroll
      for (int i = 0; i < kPrefetch; ++i) fr[i] = frag_h(i);
      auto mfma = [&](int i, const f16x8& b, f32x16& acc) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[i], b, acc, 0, 0, 0);
        if (i + kPrefetch < kNFH) fr[i + kPrefetch] = frag_h(i + kPrefetch);
      };
      if constexpr (MK != kNoMask) {
        apply_mask_half(t, 0, cur);
        next_mask(t);
      }
      if (edge(t)) {  // the key test on this half
        const int kl = key_last - (kb0 + t * kKT) - 32 * hw - 8 * half;
#pragma unroll
        for (int rr = 0; rr < 16; ++rr)
          cur[rr] = key32_of(8 * (rr >> 2) + (rr & 3)) <= kl ? cur[rr] : -INFINITY;
      }
      nxt = PRESCALED ? neg_m_tile : f32x16{};
#pragma unroll
      for (int ks = 0; ks < DK; ++ks) mfma(ks, qv[ks], nxt);
      interleave_h(0, DK);
      float mx = -INFINITY;
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) mx = max_of(mx, cur[rr]);
      mx = PRESCALED ? max_halves(mx) + m_use : max_halves(mx) * (F32M ? 1.f : scale_abs);
      // A step the mask blanks for every real row adds nothing (see step).
      const bool live = MK == kNoMask || adds(t, mx);
      if (live && __builtin_amdgcn_ballot_w64(mx > m_run + kLazy) != 0) {
        const float m_new = fmaxf(m_run, mx);
        const float alpha = m_new == -INFINITY ? 1.f : fast_exp2(m_run - m_new);
        l_run *= alpha;
#pragma unroll
        for (int dm = 0; dm < DM; ++dm) o[dm] *= alpha;
        m_run = m_new;
        if constexpr (PRESCALED) {
          const float m_use_new = reference(m_new);
          const float d = m_use_new - m_use;
          m_use = m_use_new;
#pragma unroll
          for (int rr = 0; rr < 16; ++rr) {
            cur[rr] -= d;
            nxt[rr] -= d;
            neg_m_tile[rr] = -m_use;
          }
        }
      }
      if (live) {
        rebase(cur);
        const float neg_m = m_run == -INFINITY ? 0.f : -m_run;
        f16x8 p[2];
        softmax_half(cur, neg_m, p);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int dm = 0; dm < DM; ++dm) mfma(DK + j * DM + dm, p[j], o[dm]);
        interleave_h(DK, kNFH);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (SLOTS == 2 || (t & 1)) {
      dma_wait();
      if (ANY && t + 1 < n_tiles) write_m((t + 1) & 1);
      __syncthreads();
    }
  };

  // Step t: LDS holds K(t+1) in slot (t+1)&1 and V(t) in slot t&1, cur
  // holds S(t); the step loads K(t+2) and V(t+1) and leaves S(t+1) in nxt.
  // The MFMAs of S(t+1) and of step t's P V overlap step t's softmax: each
  // scheduling region pairs one MFMA group with one VALU group.  At a
  // wavefront's last active step S(t+1) reads a stale K slot and is never
  // used.
  auto step = [&](int t, int par, f32x16 (&cur)[2], f32x16 (&nxt)[2]) {
    // K(t+2) replaces K(t) (read during step t-1), V(t+1) replaces
    // V(t-1); both land during this step's math.
    if (t + 2 < n_tiles) dma_k(t & 1);
    if (t + 1 < n_tiles) dma_v((t + 1) & 1);
    if (kMaskSlots == 2 && t + 1 < n_tiles) dma_m(kb0 + (t + 1) * kKT, (t + 1) & 1);
    if (active(t)) {
      f16x8 fr[kNF];
#pragma unroll
      for (int i = 0; i < kPrefetch; ++i) fr[i] = frag(par, i);
      // MFMA i, then the read of fragment i + kPrefetch.
      auto mfma = [&](int i, const f16x8& b, f32x16& acc) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[i], b, acc, 0, 0, 0);
        if (i + kPrefetch < kNF) fr[i + kPrefetch] = frag(par, i + kPrefetch);
      };
      if constexpr (MK == kNoMask) {
        if (edge(t)) mask_step(t, cur);
        // Region A: the 2 DK MFMAs of S(t+1) beside P(t) of half 0, computed
        // against the running max as it stands.  The max matters only as a
        // bound: while every lane's sum of a half's P stays <= 2^8, so does
        // every P, and nothing moves.  Otherwise (and at a wavefront's first
        // scores) the branch below takes the row max, rescales and redoes
        // P -- so the common step computes no max at all.
        nxt[0] = PRESCALED ? neg_m_tile : f32x16{};
        nxt[1] = PRESCALED ? neg_m_tile : f32x16{};
#pragma unroll
        for (int ks = 0; ks < DK; ++ks) {
          mfma(2 * ks, qv[ks], nxt[0]);
          mfma(2 * ks + 1, qv[ks], nxt[1]);
        }
        // P(t) of half 0 goes beside region A and P(t) of half 1 beside
        // the PV MFMAs of half 0 (region B1), so both regions carry VALU
        // work; each half has its own bound check.
        f16x8 p0[2], p1[2];
        float neg_m = m_run == -INFINITY ? 0.f : -m_run;
        float ps = softmax_q(cur[0], 0, neg_m, p0[0]) + softmax_q(cur[0], 1, neg_m, p0[1]);
        asm volatile("" : "+v"(p0[0]), "+v"(p0[1]), "+v"(ps));
        interleave_mix(0, 2 * DK, 1, 1, 1);
        if (__builtin_amdgcn_ballot_w64(!(ps <= 256.f) || m_run == -INFINITY) != 0) {
          rescale(cur, nxt, row_max(cur));
          neg_m = m_run == -INFINITY ? 0.f : -m_run;
          ps = softmax_q(cur[0], 0, neg_m, p0[0]) + softmax_q(cur[0], 1, neg_m, p0[1]);
        }
        l_run += ps;
        // Region B1: the PV MFMAs of half 0 beside P(t) of half 1.
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int dm = 0; dm < DM; ++dm) mfma(2 * DK + j * DM + dm, p0[j], o[dm]);
        ps = softmax_q(cur[1], 0, neg_m, p1[0]) + softmax_q(cur[1], 1, neg_m, p1[1]);
        asm volatile("" : "+v"(p1[0]), "+v"(p1[1]), "+v"(ps));
        interleave_mix(2 * DK, 2 * DK + 2 * DM, 2, 2, 2);
        if (__builtin_amdgcn_ballot_w64(!(ps <= 256.f)) != 0) {
          // Half 1 holds a score above the bound: move the max to half 1's
          // row max.  O (half 0's product included) and l are relative to
          // the old max and scale with it.
          float mx = -INFINITY;
#pragma unroll
          for (int rr = 0; rr < 16; ++rr) mx = fmaxf(mx, cur[1][rr]);
          rescale(cur, nxt, PRESCALED ? max_xor32(mx) + m_use : max_xor32(mx) * scale_abs);
          neg_m = m_run == -INFINITY ? 0.f : -m_run;
          ps = softmax_q(cur[1], 0, neg_m, p1[0]) + softmax_q(cur[1], 1, neg_m, p1[1]);
        }
        l_run += ps;
        // Region B2: the PV MFMAs of half 1.
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int dm = 0; dm < DM; ++dm) mfma(2 * DK + 2 * DM + j * DM + dm, p1[j], o[dm]);
        interleave_reads(2 * DK + 2 * DM, kNF);
      } else {
        // A mask can leave a step nothing to add: every score of the
        // wavefront's real rows -inf or more than 32 below its row's running
        // max, so every P rounds to 0 in fp16.  Such a step computes only
        // S(t+1); S(t+1) is therefore computed whole before the softmax.
        apply_mask(t, cur);
        if (edge(t)) mask_step(t, cur);
        const float mx = row_max(cur);
        const bool live = adds(t, mx);
        nxt[0] = PRESCALED ? neg_m_tile : f32x16{};
        nxt[1] = PRESCALED ? neg_m_tile : f32x16{};
#pragma unroll
        for (int ks = 0; ks < DK; ++ks) {
          mfma(2 * ks, qv[ks], nxt[0]);
          mfma(2 * ks + 1, qv[ks], nxt[1]);
        }
        interleave_reads(0, 2 * DK);
        if (live) {
          update_max(cur, nxt, mx);
          rebase(cur[0]);
          rebase(cur[1]);
          const float neg_m = m_run == -INFINITY ? 0.f : -m_run;
          f16x8 p0[2], p1[2];
          softmax_half(cur[0], neg_m, p0);
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int dm = 0; dm < DM; ++dm) mfma(2 * DK + j * DM + dm, p0[j], o[dm]);
          softmax_half(cur[1], neg_m, p1);
          interleave_reads(2 * DK, 2 * DK + 2 * DM);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int dm = 0; dm < DM; ++dm) mfma(2 * DK + 2 * DM + j * DM + dm, p1[j], o[dm]);
        }
      }
    }
    dma_wait();
    __syncthreads();
  };

  // Prologue: K(0), V(0) in slot 0 and K(1) in slot 1 (four slots: also
  // V(1) and K(2)), then S(0).  A step
  // writes nxt only when it is active, and a step is active only if the one
  // before it is, so S is never read unwritten.
  f32x16 sa[2], sb[2];
  if (n_tiles > 0) {
    dma_k(0);
    dma_v(0);
    if (!ANY) dma_m(kb0, 0);
  }
  if (n_tiles > 1) dma_k(1);
  if constexpr (SLOTS == 4) {
    if (n_tiles > 1) dma_v(1);
    if (n_tiles > 2) dma_k(2);
  }
  if (ANY && n_tiles > 0) read_m(kb0);
  dma_wait();
  if (ANY && n_tiles > 0) write_m(0);
  __syncthreads();
  if (active(0)) {
    if constexpr (HALF) {
      sa[0] = qk(hw);
    } else {
      sa[0] = qk(0);
      sa[1] = qk(1);
    }
  }
  __syncthreads();  // step 0 overwrites K(0)
  // Two steps per iteration, S(t) alternating between sa and sb.
  for (int t = 0; t < n_tiles; t += 2) {
    if constexpr (HALF) {
      step_h(t, sa[0], sb[0]);
      if (t + 1 < n_tiles) step_h(t + 1, sb[0], sa[0]);
    } else {
      step(t, 0, sa, sb);
      if (t + 1 < n_tiles) step(t + 1, 1, sb, sa);
    }
  }
  if constexpr (HALF) {
    // Fold each pair: wavefront 2r + 1 leaves O, m, l (per lane) in LDS,
    // 2r weights both by exp2(m - max) (a half that saw no key weighs 0).
    dma_wait();
    __syncthreads();  // every wavefront is done with the tiles
    constexpr int kRec = DM * 16 + 2;
    static_assert(W / 2 * 64 * kRec * 4 <= sizeof(lds), "the records fit where the tiles were");
    float* rec = reinterpret_cast<float*>(lds) + ((wave >> 1) * 64 + lane) * kRec;
    if (hw == 1) {
#pragma unroll
      for (int dm = 0; dm < DM; ++dm)
#pragma unroll
        for (int k = 0; k < 16; ++k) rec[dm * 16 + k] = o[dm][k];
      rec[DM * 16] = m_run;
      rec[DM * 16 + 1] = l_run;
    }
    __syncthreads();
    if (hw == 1) return;
    const float m1 = rec[DM * 16], l1 = rec[DM * 16 + 1];
    const float M = fmaxf(m_run, m1);
    const float w0 = m_run == -INFINITY ? 0.f : fast_exp2(m_run - M);
    const float w1 = m1 == -INFINITY ? 0.f : fast_exp2(m1 - M);
#pragma unroll
    for (int dm = 0; dm < DM; ++dm)
#pragma unroll
      for (int k = 0; k < 16; ++k) o[dm][k] = o[dm][k] * w0 + rec[dm * 16 + k] * w1;
    l_run = l_run * w0 + l1 * w1;
    m_run = M;
  }

  const float l = sum_xor32(l_run);
  if (!q_ok) return;
  if (a.nsplit > 1) {
    // The partial: O unnormalised (relative to m_run), then m_run and l.
    const int64_t prow = ((static_cast<int64_t>(b) * a.Hq + h) * a.Sq + qi) * a.nsplit + sp;
    float* po = a.part + prow * D;
#pragma unroll
    for (int dm = 0; dm < DM; ++dm)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<f32x4*>(po + 32 * dm + 8 * i + 4 * half) =
            f32x4{o[dm][4 * i], o[dm][4 * i + 1], o[dm][4 * i + 2], o[dm][4 * i + 3]};
    if (half == 0) {
      float* pml = a.part + static_cast<int64_t>(a.B) * a.Hq * a.Sq * a.nsplit * D + 2 * prow;
      pml[0] = m_run;
      pml[1] = l;
    }
    return;
  }
  _Float16* op = a.out + ((static_cast<int64_t>(b) * a.Sq + qi) * a.Hq + h) * D;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  // Lane (query column, half) holds O^T rows d = 32dm + 8i + 4half + v.
#pragma unroll
  for (int dm = 0; dm < DM; ++dm)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f16x4 rv;
#pragma unroll
      for (int v = 0; v < 4; ++v) rv[v] = static_cast<_Float16>(o[dm][4 * i + v] * inv);
      *reinterpret_cast<f16x4*>(op + 32 * dm + 8 * i + 4 * half) = rv;
    }
  if (a.lse && half == 0)
    a.lse[(static_cast<int64_t>(b) * a.Hq + h) * a.Sq + qi] = l > 0.f ? (m_run + log2f(l)) * kLn2 : -INFINITY;
}

// ---- 4. short decode: a block's keys all in flight at once ----------------
//
// Calls without the causal flag whose block holds one row tile (the g
// q heads of a KV head times Sq <= 32 rows) and at most kWaves2 * KW keys
// (KW = 64 keys at D = 64, 32 at D = 128): wavefront w loads keys
// kb + w KW .. + KW - 1 of K and V into its own LDS slice, all loads issued
// at kernel start, and computes its partial of the rows over them (S^T =
// K Q^T, softmax, O^T = V^T P^T as in sdpa_fwd_lds_kernel, the V^T operands
// through transposing LDS reads).  The W partials are then folded in LDS:
// the call is one round of loads and one kernel.  Longer key runs are split
// across blocks, which merge inside the kernel (below).  W = 8 wavefronts,
// or 4 when a split needs at most half the device's compute units at 8: the
// blocks then use every unit, each loading half the keys.
template <int D>
struct ShortLds {
  static constexpr int kKW = D == 64 ? 64 : 32;          // keys per wavefront
  static constexpr int kRowK = D + kPadH;                // K row, halves (padded)
  static constexpr int kUK = kRowK / 8;                  // 16-byte units per K row
  static constexpr int kNK = (kKW * kUK + 63) / 64;      // loads per K slice
  static constexpr int kNV = kKW * D / 8 / 64;           // loads per V slice (rows of D halves)
  static constexpr int kSliceB = (kNK + kNV) * 1024;     // bytes per wavefront
  static constexpr int kFoldF = D / 2 + 4;               // per-lane record of a partial: O^T, m, l (16-byte aligned)
  static_assert(kKW * D / 8 % 64 == 0, "V slices must be whole loads");
  static_assert(64 * kFoldF * 4 <= kSliceB, "a wavefront's fold records fit its own slice");
};

// A mask with contiguous keys is read as it lies, 4 elements of the lane's
// row at a time, while the slices load (masked calls keep q unscaled and sum
// the fp32 probabilities).
template <int D, bool PRESCALED, int W, int MK = kNoMask>
__global__ __launch_bounds__(W * 64) void sdpa_decode_short_kernel(Fwd2Args a) {
  static_assert(MK == kNoMask || !PRESCALED, "masked: scores scaled in fp32");
  using L = ShortLds<D>;
  constexpr int DK = D / 16, DM = D / 32;
  constexpr int KW = L::kKW, MT = KW / 32;  // 32-key S^T tiles per wavefront
  constexpr int NT = W * 64;                // threads
  // W slices; a four-wavefront block asks for more than half a compute
  // unit's 160 KiB, so that no unit runs two blocks while another idles.
  constexpr int kLdsB = W * L::kSliceB > 82 * 1024 ? W * L::kSliceB : 82 * 1024;
  __shared__ __align__(16) _Float16 lds[kLdsB / 2];

  // item = ((b * Hkv + kvh) * gp + gi) * nsplit + sp (one query block).
  uint32_t item = blockIdx.x;
  if (a.xcd_remap) item = (item % 8) * (a.n_items / 8) + item / 8;
  const uint32_t i1 = fdiv(item, a.by_split), i2 = fdiv(i1, a.by_gp), bq = fdiv(i2, a.by_hkv);
  const int sp = static_cast<int>(item - i1 * a.nsplit);
  item = i1;
  const int gi = static_cast<int>(i1 - i2 * a.gp);
  const int kvh = static_cast<int>(i2 - bq * a.Hkv);
  const int b = static_cast<int>(bq);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  __builtin_assume(wave >= 0 && wave < W);
  const int col = lane & 31, half = lane >> 5;
  const int pack = a.pack;
  const int qi = static_cast<int>(fdiv(col, a.by_pack));  // this lane's row: query qi, q head h
  const int h = kvh * a.g + gi * pack + (col - qi * pack);
  const bool q_ok = qi < a.Sq;

  // This wavefront's keys: kw .. kw + KW - 1, those below key_end visible.
  const int kb0 = sp * a.split_keys;
  const int key_end = a.nsplit > 1 ? min(a.Skv, kb0 + a.split_keys) : a.Skv;
  const int kw = kb0 + wave * KW;
  const int rows_here = min(key_end - kw, KW);  // <= 0: no key for this wavefront
  // Q^T operand: lane (row, half) holds features 16ks + 8half .. +8; loaded
  // first, so that scaling it waits for Q alone.
  f16x8 qv[DK];
  {
    const _Float16* qp = a.q + b * a.q_sb + h * a.q_sh + static_cast<int64_t>(min(qi, a.Sq - 1)) * a.q_ss + 8 * half;
#pragma unroll
    for (int ks = 0; ks < DK; ++ks) qv[ks] = q_ok ? *reinterpret_cast<const f16x8*>(qp + 16 * ks) : f16x8{};
  }
  _Float16* slice = lds + wave * (L::kSliceB / 2);
  constexpr uint32_t kOob = 0x80000000u;
  if (rows_here > 0) {
    const Rsrc rk = make_rsrc(a.k + b * a.k_sb + kvh * a.k_sh + static_cast<int64_t>(kw) * a.k_ss, kBufRange);
    const Rsrc rv = make_rsrc(a.v + b * a.v_sb + kvh * a.v_sh + static_cast<int64_t>(kw) * a.v_ss, kBufRange);
#pragma unroll
    for (int j = 0; j < L::kNK; ++j) {
      const int u = 64 * j + lane, row = u / L::kUK, ch = u % L::kUK;
      const bool ok = row < rows_here && ch < D / 8;  // pads, rows past the keys or the slice: zeros
      load_lds16(rk, slice + 512 * j,
                 ok ? (static_cast<uint32_t>(row) * static_cast<uint32_t>(a.k_ss) + 8 * ch) * 2 : kOob);
    }
#pragma unroll
    for (int j = 0; j < L::kNV; ++j) {
      const int u = 64 * j + lane, row = u / (D / 8), ch = u % (D / 8);
      load_lds16(rv, slice + 512 * (L::kNK + j),
                 row < rows_here ? (static_cast<uint32_t>(row) * static_cast<uint32_t>(a.v_ss) + 8 * ch) * 2 : kOob);
    }
  }
  // Mask elements of this lane's row, keys kw + 32 mt + 16 (i / 2) + 8 half +
  // 4 (i % 2) .. + 3 in mw[mt][i]; a ragged slice's keys past its last one
  // repeat that one (the key test below drops them).
  using ME = typename MaskElem<MK>::T;
  constexpr int kMW = sizeof(ME);  // 32-bit words of 4 elements
  uint32_t mw[MT][4][kMW];
  if constexpr (MK != kNoMask) {
    if (rows_here > 0) {
      const ME* mrow = static_cast<const ME*>(a.mask) + b * a.m_sb + (q_ok ? h * a.m_sh + qi * a.m_sq : kvh * a.g * a.m_sh) + kw;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int k4 = 32 * mt + 16 * (i >> 1) + 8 * half + 4 * (i & 1);
          if (rows_here >= KW) {
            __builtin_memcpy(mw[mt][i], mrow + k4, sizeof(mw[mt][i]));
          } else {
            ME x[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = mrow[min(k4 + e, rows_here - 1)];
            __builtin_memcpy(mw[mt][i], x, sizeof(x));
          }
        }
    }
  }
#pragma unroll
  for (int ks = 0; ks < DK; ++ks) {
    if constexpr (PRESCALED) {
#pragma unroll
      for (int e = 0; e < 8; ++e) qv[ks][e] = static_cast<_Float16>(static_cast<float>(qv[ks][e]) * a.scale_log2);
    } else if (a.scale_log2 < 0.f) {
      qv[ks] = -qv[ks];
    }
  }
  const float scale_abs = fmaxf(fabsf(a.scale_log2), 1e-30f);
  // The wavefront's own slice: its loads landing is all it waits for.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  float m = -INFINITY, l = 0.f;  // m: the rows' max over the slice (log2 units)
  f32x16 o[DM];
#pragma unroll
  for (int dm = 0; dm < DM; ++dm) o[dm] = f32x16{};
  // A slice whose mask drops every key for every row is left out (m -inf, l
  // 0): what K and V hold there, an unused cache's NaN, does not count.
  bool live = rows_here > 0;
  if constexpr (MK != kNoMask) {
    constexpr uint32_t kNone = MK == kMaskBool ? 0u : MK == kMaskF16 ? 0xfc00fc00u : 0xff800000u;  // a word of dropped keys
    bool kept = false;
    if (live) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int w = 0; w < kMW; ++w) kept = kept || mw[mt][i][w] != kNone;
    }
    live = __builtin_amdgcn_ballot_w64(q_ok && kept) != 0;
  }
  if (live) {
    // S^T tile mt: keys 32mt .. 32mt + 31 of the slice; lane (row, half)
    // holds keys key32_of(8i + 4half + v) in register 4i + v.
    f32x16 s[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const _Float16* krow = slice + (mt * 32 + key32_of(col)) * L::kRowK + 8 * half;
      s[mt] = f32x16{};
#pragma unroll
      for (int ks = 0; ks < DK; ++ks)
        s[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const f16x8*>(krow + 16 * ks), qv[ks], s[mt],
                                                       0, 0, 0);
    }
    // Keys past the run (and past Skv) are masked; scores in log2 units.
    const int kl = key_end - 1 - kw - 8 * half;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) {
        const int kr = mt * 32 + key32_of(8 * (rr >> 2) + (rr & 3));
        float x = PRESCALED ? s[mt][rr] : s[mt][rr] * scale_abs;
        if constexpr (MK == kMaskBool) x = ((mw[mt][rr >> 2][0] >> (8 * (rr & 3))) & 0xffu) != 0 ? x : -INFINITY;
        if constexpr (MK == kMaskF16)
          x = __builtin_fmaf(static_cast<float>(__builtin_bit_cast(f16x2, mw[mt][rr >> 2][(rr & 3) / 2])[rr & 1]), kLog2e, x);
        if constexpr (MK == kMaskF32)
          x = __builtin_fmaf(__builtin_bit_cast(float, mw[mt][rr >> 2][rr & 3]), kLog2e, x);
        s[mt][rr] = kr <= kl ? x : -INFINITY;
      }
    float mx = -INFINITY;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) mx = fmaxf(mx, s[mt][rr]);
    m = max_xor32(mx);  // the row's max over both lane halves (finite without a mask: key kw is visible)
    const float mu = MK != kNoMask && m == -INFINITY ? 0.f : m;  // a row with every key masked: weights 0
    // P (fp16) and its row sum over the same fp16 values; pb[mt][j] is the
    // PV operand of keys 32mt + 16j + 8half .. + 7.
    f16x8 pb[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float p = fast_exp2(s[mt][8 * j + e] - mu);
          pb[mt][j][e] = static_cast<_Float16>(p);
          if constexpr (MK != kNoMask) l += p;
        }
#pragma unroll
        for (int e = 0; e < 4 && MK == kNoMask; ++e)
          l = __builtin_amdgcn_fdot2(f16x2{pb[mt][j][2 * e], pb[mt][j][2 * e + 1]}, f16x2{1, 1}, l, false);
      }
    // O^T += V^T P^T: V^T operands by transposing reads of the V slice (rows
    // of D halves).
    const uint32_t vtr = static_cast<uint32_t>(wave * (L::kSliceB / 2) + L::kNK * 512) +
                         static_cast<uint32_t>((8 * half + ((lane & 15) >> 2)) * D + 16 * ((lane >> 4) & 1) +
                                               4 * (lane & 3));
#pragma unroll
    for (int c = 0; c < KW / 16; ++c)
#pragma unroll
      for (int dm = 0; dm < DM; ++dm) {
        const uint32_t e = vtr + 16 * c * D + 32 * dm;
        const v4i16 lo = tr_read4(lds + e), hi = tr_read4(lds + e + 4 * D);
        const f16x8 va = __builtin_bit_cast(f16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        o[dm] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va, pb[c >> 1][c & 1], o[dm], 0, 0, 0);
      }
  }

  // Fold: every wavefront's partial (O^T relative to m, then m and l) to
  // LDS, one 16-byte aligned record per lane, over its own slice -- free once
  // its P.V operands are read, so no barrier comes before the records.
  // Lanes of padding rows (qi >= Sq: a decode tile holds g of its 32 rows)
  // write nothing.
  constexpr int kF = L::kFoldF;
  auto rec_of = [&](int w, int ln) { return reinterpret_cast<float*>(lds + w * (L::kSliceB / 2)) + ln * kF; };
  if (q_ok) {
    float* mine = rec_of(wave, lane);
#pragma unroll
    for (int dm = 0; dm < DM; ++dm)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<f32x4*>(mine + dm * 16 + 4 * i) =
            f32x4{o[dm][4 * i], o[dm][4 * i + 1], o[dm][4 * i + 2], o[dm][4 * i + 3]};
    *reinterpret_cast<f32x2*>(mine + D / 2) = f32x2{m, l};
  }
  __syncthreads();
  // Thread t folds units u = t, t + 512, ... of the valid rows: row j (tile
  // column j) = u / (D / 4), features d = 4 (u % (D / 4)) .. d + 3, over the
  // W partials in wavefront order -- only units of real rows get a thread
  // (a decode tile of g rows: g D / 4 threads), each read 16 bytes or a
  // broadcast.  Lane (column j, half) holds value k = 16 (d / 32) + 4 (d %
  // 32 / 8) + d % 4 of feature d, half = d / 4 % 2.
  constexpr int D4 = D / 4;
  const int nv = pack * a.Sq;  // valid rows: tile columns 0 .. nv - 1
  // Key split: the block's partial of every valid row (O unnormalised
  // relative to M, then M and the row sum) goes to the workspace, then an
  // arrival flag; the block that sees every split's flag merges the rows
  // itself -- one kernel per call.  Partials and flags move with
  // device-scope (sc1) accesses: stores write through to memory and count as
  // done only once there, loads read memory, never a stale line of another
  // XCD's L2 -- no cache-wide write-back or invalidate (as a release /
  // acquire fence would issue, at ~20 us a call here) is needed.
  typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
  constexpr int kAuxDevice = 16;  // sc1: device scope
  const int64_t rows = static_cast<int64_t>(a.B) * a.Hq * a.Sq;
  const Rsrc pr = __builtin_amdgcn_make_buffer_rsrc(a.part, 0, kBufRange, kRsrcWord3);
  const uint32_t ml_off = static_cast<uint32_t>(rows * a.nsplit * D * 4);  // bytes: (M, l) pairs
  for (int u = static_cast<int>(threadIdx.x); u < nv * D4; u += NT) {
    const int j = u / D4, d = 4 * (u - j * D4);
    const int ln = j + 32 * ((d >> 2) & 1), k = 16 * (d >> 5) + 4 * ((d >> 3) & 3);
    f32x2 mlw[W];  // m and half 0's l of row j
    float l1[W];   // half 1's l
    f32x4 val[W];
#pragma unroll
    for (int w = 0; w < W; ++w) {
      mlw[w] = *reinterpret_cast<const f32x2*>(rec_of(w, j) + D / 2);
      l1[w] = rec_of(w, j + 32)[D / 2 + 1];
      val[w] = *reinterpret_cast<const f32x4*>(rec_of(w, ln) + k);
    }
    float M = -INFINITY, lsum = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) M = fmaxf(M, mlw[w][0]);
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float wt = mlw[w][0] == -INFINITY ? 0.f : fast_exp2(mlw[w][0] - M);  // a slice without keys weighs 0
      lsum += (mlw[w][1] + l1[w]) * wt;
      acc += val[w] * wt;
    }
    const int jq = static_cast<int>(fdiv(j, a.by_pack)), jh = kvh * a.g + gi * pack + (j - jq * pack);
    const int64_t r = (static_cast<int64_t>(b) * a.Hq + jh) * a.Sq + jq;
    if (a.nsplit == 1) {
      const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
      f16x4 rv;
#pragma unroll
      for (int e = 0; e < 4; ++e) rv[e] = static_cast<_Float16>(acc[e] * inv);
      *reinterpret_cast<f16x4*>(a.out + ((static_cast<int64_t>(b) * a.Sq + jq) * a.Hq + jh) * D + d) = rv;
      if (a.lse && d == 0) a.lse[r] = lsum > 0.f ? (M + log2f(lsum)) * kLn2 : -INFINITY;
    } else {
      const uint32_t prow = static_cast<uint32_t>(r * a.nsplit + sp);
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, acc), pr, (prow * D + d) * 4, 0, kAuxDevice);
      if (d == 0)
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2_t, f32x2{M, lsum}), pr, ml_off + prow * 8, 0,
                                              kAuxDevice);
    }
  }
  if (a.nsplit == 1) return;

  // Arrival: every wavefront's partial stores done, then wavefront 0 stores
  // the flag (this call's ticket), waits for it, and reads every split's
  // flag of the group.  Of any two blocks, the one whose flag store finished
  // later reads the other's flag after it, so at least one block sees all of
  // them.  Every block that does merges the rows, to the same bits (splits
  // in a fixed order).  Mergers clear the flags, so replays of a captured
  // call (one ticket) start clear; a new call's ticket matches no older
  // call's flags.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  __shared__ int s_merge;
  // The group's flags (item: its (sequence, KV head, head group) index).
  const uint32_t fl_off = ml_off + static_cast<uint32_t>(rows * a.nsplit * 8) + item * a.nsplit * 4;
  if (wave == 0) {
    if (lane == 0) __builtin_amdgcn_raw_buffer_store_b32(a.ticket, pr, fl_off + sp * 4, 0, kAuxDevice);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    bool seen = true;
    for (int s2 = lane; s2 < a.nsplit; s2 += 64)
      seen = seen && __builtin_amdgcn_raw_buffer_load_b32(pr, fl_off + s2 * 4, 0, kAuxDevice) == a.ticket;
    const bool all = __all(seen);
    if (lane == 0) s_merge = all ? 1 : 0;
  }
  __syncthreads();
  if (!s_merge) return;

  // Merge: thread (row j, features 4 d4 .. + 3) over every split in order,
  // G splits' loads in flight at once, without a branch: past the last
  // split the loads repeat it (a valid address) and, like splits with l = 0
  // (no visible key), carry no weight.
  constexpr int RP = NT / D4, G = 16;
  const int d4 = static_cast<int>(threadIdx.x) % D4;
  const uint32_t last = static_cast<uint32_t>(a.nsplit - 1);
  for (int j = static_cast<int>(threadIdx.x) / D4; j < nv; j += RP) {
    const int jq = static_cast<int>(fdiv(j, a.by_pack)), jh = kvh * a.g + gi * pack + (j - jq * pack);
    const int64_t r = (static_cast<int64_t>(b) * a.Hq + jh) * a.Sq + jq;
    const uint32_t r0 = static_cast<uint32_t>(r * a.nsplit);
    float Mr = -INFINITY, Lr = 0.f;
    f32x4 ac = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < a.nsplit; s0 += G) {
      f32x2 ml[G];
      f32x4 ov[G];
#pragma unroll
      for (int jj = 0; jj < G; ++jj) {
        const uint32_t s2 = min(static_cast<uint32_t>(s0 + jj), last);
        ml[jj] = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(pr, ml_off + (r0 + s2) * 8, 0, kAuxDevice));
        ov[jj] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(pr, ((r0 + s2) * D + 4 * d4) * 4, 0,
                                                                                 kAuxDevice));
      }
      // The split's max, or -inf when it carries no weight.  A NaN sum counts
      // (and reaches the row whatever its weight: NaN times 0).
      float mv[G];
#pragma unroll
      for (int jj = 0; jj < G; ++jj) mv[jj] = s0 + jj < a.nsplit && ml[jj][1] != 0.f ? ml[jj][0] : -INFINITY;
      float Mn = Mr;
#pragma unroll
      for (int jj = 0; jj < G; ++jj) Mn = fmaxf(Mn, mv[jj]);
      const float Mu = Mn == -INFINITY ? 0.f : Mn;  // nothing visible yet: weights 0
      const float c = fast_exp2(Mr - Mu);  // Mr = -inf: c = 0
      Lr *= c;
      ac *= c;
#pragma unroll
      for (int jj = 0; jj < G; ++jj) {
        const float w = fast_exp2(mv[jj] - Mu);  // -inf: 0
        Lr += ml[jj][1] * w;
        ac += ov[jj] * w;
      }
      Mr = Mn;
    }
    const float inv = Lr > 0.f ? 1.f / Lr : 0.f;
    f16x4 rv;
#pragma unroll
    for (int e = 0; e < 4; ++e) rv[e] = static_cast<_Float16>(ac[e] * inv);
    *reinterpret_cast<f16x4*>(a.out + ((static_cast<int64_t>(b) * a.Sq + jq) * a.Hq + jh) * D + 4 * d4) = rv;
    if (a.lse && d4 == 0) a.lse[r] = Lr > 0.f ? (Mr + log2f(Lr)) * kLn2 : -INFINITY;
  }
  for (int s2 = static_cast<int>(threadIdx.x); s2 < a.nsplit; s2 += NT)
    __builtin_amdgcn_raw_buffer_store_b32(0u, pr, fl_off + s2 * 4, 0, kAuxDevice);
}

// Combines a key split's partials per (sequence, q head, query): one
// workgroup per row.  Thread (sl, d4) folds splits sl, sl + SL, ... of
// features 4 d4 .. 4 d4 + 3, G of them loaded at once (every load issued
// before the first is used); the SL folds of a feature are then combined
// through LDS.  Splits with l = 0 (no visible key) carry no weight; a row
// with none gives zeros and LSE -inf.  (One work-item per 4 features of a
// row, looping over the splits, took 5-7 us for 32 splits of 32 rows: the
// whole merge ran on 4 compute units.)
struct MergeArgs {
  const float* part;
  _Float16* out;
  float* lse;
  int Hq, Sq, D, nsplit;
  int64_t rows;  // B * Hq * Sq
};

template <int D>
__global__ __launch_bounds__(256) void sdpa_split_merge_kernel(MergeArgs a) {
  constexpr int D4 = D / 4, SL = 256 / D4, G = 4;
  __shared__ float s_m[SL], s_l[SL];
  __shared__ f32x4 s_acc[SL][D4];
  const int64_t r = blockIdx.x;
  const int d4 = static_cast<int>(threadIdx.x) % D4, sl = static_cast<int>(threadIdx.x) / D4;
  const float* pml = a.part + a.rows * a.nsplit * D + 2 * r * a.nsplit;
  const float* po = a.part + r * a.nsplit * D + 4 * d4;
  float M = -INFINITY, L = 0.f;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s0 = sl; s0 < a.nsplit; s0 += SL * G) {
    f32x2 ml[G];
    f32x4 ov[G];
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const int sp = s0 + j * SL;
      const bool in = sp < a.nsplit;
      ml[j] = in ? *reinterpret_cast<const f32x2*>(pml + 2 * sp) : f32x2{-INFINITY, 0.f};
      ov[j] = in ? *reinterpret_cast<const f32x4*>(po + static_cast<int64_t>(sp) * D) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    float Mn = M;
#pragma unroll
    for (int j = 0; j < G; ++j)
      if (ml[j][1] != 0.f) Mn = fmaxf(Mn, ml[j][0]);  // (a NaN sum counts: it reaches the row's result)
    const float Mu = Mn == -INFINITY ? 0.f : Mn;  // nothing visible yet: weights 0
    const float c = exp2f(M - Mu);  // M = -inf: c = 0
    L *= c;
    acc *= c;
#pragma unroll
    for (int j = 0; j < G; ++j) {
      if (ml[j][1] == 0.f) continue;
      const float w = exp2f(ml[j][0] - Mu);
      L += ml[j][1] * w;
      acc += ov[j] * w;
    }
    M = Mn;
  }
  if (d4 == 0) {
    s_m[sl] = M;
    s_l[sl] = L;
  }
  s_acc[sl][d4] = acc;
  __syncthreads();
  if (sl != 0) return;
  M = -INFINITY;
#pragma unroll
  for (int t = 0; t < SL; ++t)
    if (s_l[t] != 0.f) M = fmaxf(M, s_m[t]);
  L = 0.f;
  acc = f32x4{0.f, 0.f, 0.f, 0.f};
  const float Mu = M == -INFINITY ? 0.f : M;
#pragma unroll
  for (int t = 0; t < SL; ++t) {
    if (s_l[t] == 0.f) continue;
    const float w = exp2f(s_m[t] - Mu);
    L += s_l[t] * w;
    acc += s_acc[t][d4] * w;
  }
  const int d = 4 * d4;
  const int64_t qi = r % a.Sq, bh = r / a.Sq;
  const int64_t h = bh % a.Hq, b = bh / a.Hq;
  const float inv = L > 0.f ? 1.f / L : 0.f;
  f16x4 rv;
#pragma unroll
  for (int v = 0; v < 4; ++v) rv[v] = static_cast<_Float16>(acc[v] * inv);
  *reinterpret_cast<f16x4*>(a.out + ((b * a.Sq + qi) * a.Hq + h) * D + d) = rv;
  if (a.lse && d == 0) a.lse[r] = L > 0.f ? (M + log2f(L)) * kLn2 : -INFINITY;
}

// The same merge for many rows and few splits (chunked prefill: thousands
// of rows, 2-16 splits): D / 4 threads per row, each merging its 4 features
// over every split with the loads of 8 splits in flight at once, 256 / (D /
// 4) rows per block.  (The kernel above gives each row a block and spreads
// its splits over the block: right for decode's few rows and many splits;
// with one block per row of 8 splits its blocks take 9.9 us for 8192 rows,
// whose partials are 34 MB.)
template <int D>
__global__ __launch_bounds__(256) void sdpa_split_merge_rows_kernel(MergeArgs a) {
  constexpr int D4 = D / 4, RPB = 256 / D4, G = 8;
  const int d4 = static_cast<int>(threadIdx.x) % D4;
  const int64_t r = static_cast<int64_t>(blockIdx.x) * RPB + static_cast<int>(threadIdx.x) / D4;
  if (r >= a.rows) return;
  const float* pml = a.part + a.rows * a.nsplit * D + 2 * r * a.nsplit;
  const float* po = a.part + r * a.nsplit * D + 4 * d4;
  float M = -INFINITY, L = 0.f;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < a.nsplit; s0 += G) {
    f32x2 ml[G];
    f32x4 ov[G];
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const int sp = s0 + j;
      const bool in = sp < a.nsplit;
      ml[j] = in ? *reinterpret_cast<const f32x2*>(pml + 2 * sp) : f32x2{-INFINITY, 0.f};
      // Non-temporal: each partial is read once (chunked prefill, B 4 x 128
      // queries x 4096 keys, 56.2 -> 55.3 us a call; B 8 x 64 x 4096 56.7 ->
      // 52.9 us; one box, two alternations).
      ov[j] = in ? __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(po + static_cast<int64_t>(sp) * D))
                 : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    float Mn = M;
#pragma unroll
    for (int j = 0; j < G; ++j)
      if (ml[j][1] != 0.f) Mn = fmaxf(Mn, ml[j][0]);  // (a NaN sum counts: it reaches the row's result)
    const float Mu = Mn == -INFINITY ? 0.f : Mn;  // nothing visible yet: weights 0
    const float c = exp2f(M - Mu);  // M = -inf: c = 0
    L *= c;
    acc *= c;
#pragma unroll
    for (int j = 0; j < G; ++j) {
      if (ml[j][1] == 0.f) continue;
      const float w = exp2f(ml[j][0] - Mu);
      L += ml[j][1] * w;
      acc += ov[j] * w;
    }
    M = Mn;
  }
  const int d = 4 * d4;
  const int64_t qi = r % a.Sq, bh = r / a.Sq;
  const int64_t h = bh % a.Hq, b = bh / a.Hq;
  const float inv = L > 0.f ? 1.f / L : 0.f;
  f16x4 rv;
#pragma unroll
  for (int v = 0; v < 4; ++v) rv[v] = static_cast<_Float16>(acc[v] * inv);
  *reinterpret_cast<f16x4*>(a.out + ((b * a.Sq + qi) * a.Hq + h) * D + d) = rv;
  if (a.lse && d == 0) a.lse[r] = L > 0.f ? (M + log2f(L)) * kLn2 : -INFINITY;
}

int device_cus();

// Key split of a call without the causal flag, given its grid of 256-row
// blocks: splits enough that the grid gives every compute unit a block, each
// of at least `least` keys, once the keys are worth the partials' round trip
// through memory and the merge pass -- more keys, the nearer the unsplit grid
// of 64- or 128-row blocks comes to filling the device.  Measured (32 / 8
// heads, D 128, batch 1, us; the boundary's two sides):
//  * blocks of at most 64 rows (decode, short runs of queries), which half
//    steps cover whatever the grid: while the grid leaves units idle, past
//    512 keys in runs of 256 up to 1/8 of the units (2 x 16 heads of D 64 x 40
//    queries x 1100 keys: 11.9, runs of 512 13.3), beyond from 1024 in runs of
//    512 (16 x 32 / 8 heads x 8 x 2100: unsplit 40.3, split 34.4);
//  * up to 1/32 of the units (40 queries): past 512 keys, runs of 256 (512
//    keys unsplit 10.6, split 12.2; 800: 13.6 and 12.9; 1600 in runs of 256
//    14.6, of 512 17.0);
//  * up to 1/8 (256 queries): from 1024, runs of 512 (800 keys unsplit 16.5,
//    split 20.8; 1100: 21.0 and 21.2; 3200 in runs of 256 33.5, of 512 32.6);
//  * up to 1/3 (512 queries): from 2048, runs of 768 (1600 keys unsplit 28.2,
//    split 33.5; 2200: 37.0 and 36.7); D 64 from 1536 (2 x 16 heads x 300 x
//    2000: 26.1 and 22.6);
//  * up to 1/2 (900 queries): from 3072 (2000 keys unsplit 39.6, split 48.9;
//    8000: 136.2 and 126.6; D 64, 2 x 16 heads x 900 x 4000: 49.7 and 44.8);
//  * above, never (1280 x 1280 unsplit 38.9, split 51.0).
// Returns nsplit; split_keys is a multiple of 64.
int plan_split(int64_t blocks, int64_t rows, int Skv, int D, int* split_keys) {
  *split_keys = Skv;
  const int64_t cus = device_cus() > 0 ? device_cus() : 256;
  const bool few = rows <= 64;
  const bool eighth = 8 * blocks <= cus;
  const int from = 32 * blocks <= cus || (few && eighth) ? 513
                   : few || eighth                      ? 1024
                   : 3 * blocks <= cus                  ? (D == 64 ? 1536 : 2048)
                                                        : 3072;
  const int least = 32 * blocks <= cus || (few && eighth) ? 4 * kKT : few || eighth ? 512 : 768;
  if ((few ? blocks >= cus : 2 * blocks > cus) || Skv < from) return 1;
  const int64_t ns = std::min<int64_t>((cus + blocks - 1) / blocks, Skv / least);
  if (ns <= 1) return 1;
  const int64_t keys = ((Skv + ns - 1) / ns + kKT - 1) / kKT * kKT;
  *split_keys = static_cast<int>(keys);
  return static_cast<int>((Skv + keys - 1) / keys);
}

size_t split_bytes(int64_t rows, int nsplit, int D) {
  return nsplit > 1 ? static_cast<size_t>(rows) * nsplit * (D + 2) * sizeof(float) : 0;
}

int pack_heads(int B, int Hkv, int g, int Sq);

int64_t blocks_for(int B, int Hkv, int g, int Sq, int pack, int rows = kQB) {
  return static_cast<int64_t>(B) * Hkv * (g / pack) * ((static_cast<int64_t>(pack) * Sq + rows - 1) / rows);
}

// The workgroup an LDS-kernel call runs: W wavefronts, each a row tile of
// its own (W x 32 rows), or two to a tile in half steps (W / 2 x 32 rows).
//  k256   8 wavefronts, 256 rows, one workgroup per compute unit;
//  k128   4 wavefronts, 128 rows, two per unit: half the rows of k256 waste
//         less of a last round and of causal attention's uneven blocks, and
//         the two of a unit do not wait for each other at barriers;
//  kHalf8 8 wavefronts, 128 rows in half steps, without a mask K / V two
//         steps ahead;
//  kHalf4 4 wavefronts, 64 rows in half steps, two per unit (D 64: three):
//         the shortest chain per block, for grids that leave units idle
//         otherwise.
enum Shape { k256, k128, kHalf8, kHalf4 };
int shape_rows(Shape s) { return s == k256 ? 256 : s == kHalf4 ? 64 : 128; }

// Which of them, for `pairs` (sequence, q heads sharing rows) pairs of `rows`
// rows over nsplit runs of `keys` keys (g: q heads per KV head).  Measured, prepared calls, one box,
// 32 / 8 heads of D 128 at batch 1 unless said (k256 / k128 / kHalf8 /
// kHalf4, us):
//  * one step of keys: k128 (64 x 64: 6.5 / 6.5 / 7.1 / 6.9), the fold of
//    half steps is not paid back;
//  * else at most 64 rows: kHalf8 (16 queries x 2000 keys, boolean mask, B 4:
//    17.8 / 18.4 / 16.4 / 17.7);
//  * a 64-row grid within one round of the device (causal and masked blocks,
//    of uneven cost, two rounds; three at D 64): kHalf4 (512 x 512: 20.5 /
//    15.0 / 16.3 / 13.6; causal 1000: 30.3 / 23.3 / 24.0 / 21.4; causal boolean
//    mask 1000: 43.8 / 34.8 / 32.1 / 31.2; D 64, 8 x 16 heads x 384, padding
//    mask: 16.1 / 16.1 / 21.1 / 14.7).  Past it k128 (1000 x 1000: 32.0 / 25.6
//    / 27.1 / 25.5; B 4 x 640, padding mask: 56.4 / 47.8 / 58.3 / 49.9; causal
//    4096: 142.9 / 141.7 / 190.7 / 188.1; 3072: 170.2 / 151.7 / 184.8 / 183.9),
//    but k256 at D 128 where its grid is whole rounds of even blocks (4096 x
//    4096: 251.8 / 253.7; 8192: 942 / 960; 5000, 2.5 rounds: 408.0 / 383.6),
//    or causal of two rounds, where each long block is followed by its
//    complement, heads that share K and V, and more than 8 blocks a head.
//    With q, k, v in the 256 MB cache, as the projections before leave them,
//    k256 / k128: 3841 rows 130.4 / 132.4, 4096 136.0 / 141.5, 16 / 8 heads x
//    8192 250.4 / 261.8; from HBM the two are within 1 % (128.8 / 129.8, 140.5
//    / 139.2, 259.3 / 257.4).  At 8 blocks a head (B 2 x 2048) 78.0 / 79.0, from
//    HBM 82.9 / 81.5; below, k128 (B 4 x 1024 56.8 / 50.6, B 8 x 512 41.6 / 37.6).
//    32 heads of their own K and V: 187.7 / 172.2; just past two rounds (4097)
//    149.4 / 143.7; B 2, four rounds: 274.1 / 267.8;
//  * key splits, whose blocks are even and end in a store of their partials:
//    kHalf4 within one round (64 queries x 2000 keys: 25.4 / 20.1 / 20.4 /
//    17.3; beyond it, B 4: 30.3 / 29.9 / 37.8 / 35.6); at D 128 k256 when its
//    grid is whole rounds (B 4 x 128 x 8000: 95.6 / 100.2 / 122 / 120; 15
//    sixteenths of a round, B 1: 39.7 / 37.4 / 48.0 / 46.9) or a block has at
//    most 128 rows (B 4 x 32 x 8000: 41.4 / 45.0 / 44.3 / 43.3; D 64: kHalf8,
//    4 x 16 heads x 64 x 8000: 47.0 / 48.1 / 42.3 / 43.8); else k128.
Shape pick_shape(int64_t pairs, int64_t rows, int g, int keys, int nsplit, int D, bool causal, int mask_kind) {
  const int64_t cus = device_cus() > 0 ? device_cus() : 256;
  auto blocks = [&](int64_t r) { return pairs * nsplit * ((rows + r - 1) / r); };
  if (mask_kind == kMaskF32) return rows <= 64 ? kHalf8 : kHalf4;  // the kernel's two
  if (keys <= kKT) return k128;
  if (rows <= 64) return kHalf8;
  if (blocks(64) <= (nsplit > 1 ? 1 : D == 64 ? 3 : causal || mask_kind != kNoMask ? 2 : 1) * cus) return kHalf4;
  const bool whole = D == 128 && blocks(256) % cus == 0;
  const bool paired = g > 1 && blocks(256) == 2 * cus && rows > 8 * 256;
  if (nsplit == 1) return whole && (!causal || paired) ? k256 : k128;
  if (rows <= 128) return D == 128 ? k256 : kHalf8;
  return whole ? k256 : k128;
}

// The grid of a call: short query runs pack all g q heads of a KV head into
// one block's rows and split the keys until the grid fills the device, if
// the workspace (ws_bytes) holds the split's partials; otherwise the heads
// are packed only as far as the unsplit grid still fills the device
// (pack_heads).  Masked calls take the same grid; one block per q head and 256 queries, unsplit, left most units or
// wavefronts idle for short query runs: 128 queries x 4096 keys with the
// chunk's causal boolean mask (B 4, 32 / 8 heads) 94.0 us, packed and split
// 54.3.
struct GridPlan {
  int pack = 1, nsplit = 1, split_keys = 0;
  size_t part_bytes = 0;
  bool short_decode = false;  // sdpa_decode_short_kernel
  int waves = kWaves2;         // its wavefronts per block
  Shape shape = k256;
};

// Short decode: one row tile (the g q heads of a KV head times Sq <= 32
// rows) whose keys fit one block (kWaves2 slices), or a split of them
// over blocks that all run in one round of the device.  Masks are read as they
// lie (contiguous keys: the caller's check).
bool short_grid(int B, int Hq, int Hkv, int Sq, int Skv, int D, size_t ws_bytes, GridPlan& gp) {
  const int g = Hq / Hkv;
  if (Sq <= 0 || static_cast<int64_t>(g) * Sq > 32) return false;
  const int kw = D == 64 ? ShortLds<64>::kKW : ShortLds<128>::kKW;
  const int64_t cus = device_cus() > 0 ? device_cus() : 256;
  int waves = kWaves2;
  int ns = std::max(1, (Skv + waves * kw - 1) / (waves * kw));
  // A split over at most half the units at eight wavefronts: four-wavefront
  // blocks of half the keys, twice as many, one per unit (batch-1 GQA, 4096
  // keys at D 128: 256 blocks of 128 keys instead of 128 of 256).
  if (ns > 1 && static_cast<int64_t>(B) * Hkv * 2 * ns <= cus) {
    waves = 4;
    ns = (Skv + waves * kw - 1) / (waves * kw);
  }
  // the partials, then one arrival flag per (sequence, KV head, split)
  const size_t pb = ns > 1 ? split_bytes(static_cast<int64_t>(B) * Hq * Sq, ns, D) +
                                 static_cast<size_t>(B) * Hkv * ns * sizeof(uint32_t)
                           : 0;
  if (static_cast<int64_t>(B) * Hkv * ns <= cus && (ns == 1 || ws_bytes >= pb)) {
    gp.pack = g;
    gp.nsplit = ns;
    gp.split_keys = ns > 1 ? waves * kw : Skv;
    gp.part_bytes = pb;
    gp.short_decode = true;
    gp.waves = waves;
    return true;
  }
  return false;
}

// mask_kind: a staged or copied mask's; can_pack: its rows of a KV head's q heads
// fit one buffer descriptor (else heads stay apart).
GridPlan plan_grid(int B, int Hq, int Hkv, int Sq, int Skv, int D, bool causal, size_t ws_bytes,
                   int mask_kind = kNoMask, bool can_pack = true) {
  const bool masked = mask_kind != kNoMask;
  GridPlan gp;
  const int g = can_pack ? Hq / Hkv : 1;
  const int Hb = Hq / g;  // the (KV head, pack group) pairs of a sequence
  gp.split_keys = Skv;
  if (!causal && !masked && short_grid(B, Hq, Hkv, Sq, Skv, D, ws_bytes, gp)) return gp;
  if (!causal && Sq > 0) {
    const int p0 = Sq < kQB ? g : 1;
    int keys = Skv;
    const int ns = plan_split(blocks_for(B, Hb, g, Sq, p0), static_cast<int64_t>(p0) * Sq, Skv, D, &keys);
    const size_t pb = split_bytes(static_cast<int64_t>(B) * Hq * Sq, ns, D);
    if (ns > 1 && ws_bytes >= pb) {
      gp.pack = p0;
      gp.nsplit = ns;
      gp.split_keys = keys;
      gp.part_bytes = pb;
      gp.shape = pick_shape(static_cast<int64_t>(B) * Hb * (g / p0), static_cast<int64_t>(p0) * Sq, g, keys, ns, D,
                            causal, mask_kind);
      return gp;
    }
  }
  gp.pack = pack_heads(B, Hb, g, Sq);
  gp.shape = pick_shape(static_cast<int64_t>(B) * Hb * (g / gp.pack), static_cast<int64_t>(gp.pack) * Sq, g, Skv, 1, D,
                        causal, mask_kind);
  return gp;
}

// Decode calls (one query per sequence, no mask, no causal flag) too large
// for the short-decode kernel whose grid of (sequence, KV head, chunk) items
// fills at least half the device: they stream K / V through the split-KV
// decode kernels (decode_attn.hip), whose operands come straight from
// memory into registers -- no LDS tiles, no barrier per step.
// Masks with contiguous keys are read as they lie (16 sequences of up to
// 2048 padded keys, 32 / 8 heads of D 128: 32.4 us in half steps of the LDS
// kernel, 23.2 here, the padding's K and V not read); a mask row shorter than
// the run its loads cover (64 keys) stays with the LDS kernel.
spyre_hip::DenseDecodePlan dense_route(int B, int Hq, int Hkv, int Sq, int Skv, int D, bool causal, int mask_kind,
                                       const int64_t* mask_strides) {
  if (causal || Sq != 1) return {};
  if (mask_kind != kNoMask && (mask_strides[3] != 1 || Skv < kKT)) return {};
  GridPlan gp;
  if (short_grid(B, Hq, Hkv, Sq, Skv, D, SIZE_MAX, gp)) return {};
  return spyre_hip::dense_decode_plan(B, Hq, Hkv, Skv, D);
}

template <int W, int MK>
void launch_short_masked(const Fwd2Args& f2, int D, hipStream_t st) {
  const dim3 grid(f2.n_items);
  if (D == 128)
    sdpa_decode_short_kernel<128, false, W, MK><<<grid, W * 64, 0, st>>>(f2);
  else
    sdpa_decode_short_kernel<64, false, W, MK><<<grid, W * 64, 0, st>>>(f2);
}

template <int W>
void launch_short_w(const Fwd2Args& f2, int D, bool prescaled, int mask_kind, hipStream_t st) {
  const dim3 grid(f2.n_items);
  if (mask_kind == kMaskF16)
    launch_short_masked<W, kMaskF16>(f2, D, st);
  else if (mask_kind == kMaskF32)
    launch_short_masked<W, kMaskF32>(f2, D, st);
  else if (mask_kind == kMaskBool)
    launch_short_masked<W, kMaskBool>(f2, D, st);
  else if (D == 128 && prescaled)
    sdpa_decode_short_kernel<128, true, W><<<grid, W * 64, 0, st>>>(f2);
  else if (D == 128)
    sdpa_decode_short_kernel<128, false, W><<<grid, W * 64, 0, st>>>(f2);
  else if (prescaled)
    sdpa_decode_short_kernel<64, true, W><<<grid, W * 64, 0, st>>>(f2);
  else
    sdpa_decode_short_kernel<64, false, W><<<grid, W * 64, 0, st>>>(f2);
}

void launch_short(const Fwd2Args& f2, int D, bool prescaled, int waves, int mask_kind, hipStream_t st) {
  if (waves == 4)
    launch_short_w<4>(f2, D, prescaled, mask_kind, st);
  else
    launch_short_w<kWaves2>(f2, D, prescaled, mask_kind, st);
}

template <int MK, int SLOTS, bool HALF, int W, bool ANY = false>
void launch_lds(const Fwd2Args& f2, int D, bool prescaled, hipStream_t st) {
  const dim3 grid(f2.n_items);
  if (D == 128 && prescaled)
    sdpa_fwd_lds_kernel<128, true, MK, SLOTS, HALF, W, ANY><<<grid, W * 64, 0, st>>>(f2);
  else if (D == 128)
    sdpa_fwd_lds_kernel<128, false, MK, SLOTS, HALF, W, ANY><<<grid, W * 64, 0, st>>>(f2);
  else if (prescaled)
    sdpa_fwd_lds_kernel<64, true, MK, SLOTS, HALF, W, ANY><<<grid, W * 64, 0, st>>>(f2);
  else
    sdpa_fwd_lds_kernel<64, false, MK, SLOTS, HALF, W, ANY><<<grid, W * 64, 0, st>>>(f2);
}

template <int W>
void launch_f32(const Fwd2Args& f2, int D, hipStream_t st) {
  const dim3 grid(f2.n_items);
  if (D == 128)
    sdpa_fwd_lds_kernel<128, false, kMaskF32, 2, true, W><<<grid, W * 64, 0, st>>>(f2);
  else
    sdpa_fwd_lds_kernel<64, false, kMaskF32, 2, true, W><<<grid, W * 64, 0, st>>>(f2);
}

// A copy of a mask with 16-byte rows: [bm][hm][qm][pitch bytes], keys past
// Skv zero.
struct MaskPadArgs {
  const char* src;
  char* dst;
  int64_t sb, sh, sq, sk;  // source strides, elements
  uint32_t n_units;        // bm * hm * qm * units
  int hm, qm, units, Skv;
  spyre_hip::FastDiv by_units, by_q, by_h;
};

// Bound by memory: a lane takes 4 units (ROWS: contiguous keys, rows of at
// least 16 bytes), each one load at any alignment, loads before stores; the
// unit that crosses a row's end is the row's last 16 bytes, shifted.  Else a
// unit's elements one by one, through their stride, consecutive lanes on
// consecutive rows.  With three 64-bit divisions and element loads for every
// unit, calls with 32 heads of D 128, 4095 x 4095: fp16 bias per head (1.07 GB
// copied) 947 -> 698 us, causal boolean 275 -> 265, its transposed view 326 ->
// 268; 2001 x 2001, fp16 per head 249 -> 191.
template <int ESZ, bool ROWS>
__global__ __launch_bounds__(256) void mask_pad_kernel(MaskPadArgs a) {
  constexpr int U = ROWS ? 4 : 1, E = 16 / ESZ;
  const uint32_t u0 = blockIdx.x * (256 * U) + threadIdx.x;
  u32x4 x[U];
  int64_t at[U];  // units of the copy
#pragma unroll
  for (int it = 0; it < U; ++it) {
    const uint32_t u = u0 + 256 * it;
    if (u >= a.n_units) continue;
    uint32_t bh, q, cu;
    if constexpr (ROWS) {  // consecutive lanes: a row's units
      const uint32_t row = fdiv(u, a.by_units);
      bh = fdiv(row, a.by_q), cu = u - row * a.units, q = row - bh * a.qm;
    } else {  // consecutive lanes: rows (a transposed mask's are contiguous)
      const uint32_t r = fdiv(u, a.by_q);
      bh = fdiv(r, a.by_units), q = u - r * a.qm, cu = r - bh * a.units;
    }
    const uint32_t b = fdiv(bh, a.by_h);
    const int64_t h = bh - b * a.hm;
    at[it] = (static_cast<int64_t>(bh) * a.qm + q) * a.units + cu;
    const char* src = a.src + (static_cast<int64_t>(b) * a.sb + h * a.sh + q * a.sq) * ESZ;
    if constexpr (ROWS) {
      const int back = max(16 * (static_cast<int>(cu) + 1) - a.Skv * ESZ, 0);  // the unit's bytes past the row
      __builtin_memcpy(&x[it], src + (16 * static_cast<int>(cu) - back), 16);
      if (back > 0) x[it] = drop_bytes(x[it], back);
    } else {
      x[it] = u32x4{0, 0, 0, 0};
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int key = static_cast<int>(cu) * E + e;
        uint32_t v = 0;
        __builtin_memcpy(&v, src + min(key, a.Skv - 1) * a.sk * ESZ, ESZ);
        x[it][e * ESZ / 4] |= (key < a.Skv ? v : 0u) << (8 * ESZ * (e % (4 / ESZ)));
      }
    }
  }
#pragma unroll
  for (int it = 0; it < U; ++it)
    if (u0 + 256 * it < a.n_units) *reinterpret_cast<u32x4*>(a.dst + at[it] * 16) = x[it];
}

// The copy of a mask, hm x qm rows for each of bm sequences; past 2^31 units
// (32 GiB) one (sequence, head) a launch, whose slice is below 2 GiB.
template <int ESZ>
int launch_mask_pad(MaskPadArgs a, int64_t bm, hipStream_t st) {
  if (bm * a.hm * a.qm * a.units >= (int64_t{1} << 31) - 1024) {
    for (int64_t b = 0; b < bm; ++b)
      for (int64_t h = 0; h < a.hm; ++h) {
        MaskPadArgs one = a;
        one.src += (b * a.sb + h * a.sh) * ESZ;
        one.dst += (b * a.hm + h) * a.qm * a.units * 16;
        one.hm = 1;
        const int rc = launch_mask_pad<ESZ>(one, 1, st);
        if (rc != SPYRE_OK) return rc;
      }
    return SPYRE_OK;
  }
  a.n_units = static_cast<uint32_t>(bm * a.hm * a.qm * a.units);
  a.by_units = spyre_hip::make_fastdiv(static_cast<uint32_t>(a.units));
  a.by_q = spyre_hip::make_fastdiv(static_cast<uint32_t>(a.qm));
  a.by_h = spyre_hip::make_fastdiv(static_cast<uint32_t>(a.hm));
  if (a.sk == 1 && a.Skv * ESZ >= 16)
    mask_pad_kernel<ESZ, true><<<dim3((a.n_units + 1023) / 1024), 256, 0, st>>>(a);
  else
    mask_pad_kernel<ESZ, false><<<dim3((a.n_units + 255) / 256), 256, 0, st>>>(a);
  const hipError_t e = hipGetLastError();
  SPYRE_REQUIRE(e == hipSuccess, SPYRE_EHIP, "mask copy launch failed: %s", hipGetErrorString(e));
  return SPYRE_OK;
}

bool aligned16(const void* p);
int64_t s64_of(int Skv);

// How a call's mask reaches the kernels:
//  kRouteNone    no mask;
//  kRouteStaged  fp16 / bool, rows of whole 16-byte units: the main kernel
//                stages it as it lies;
//  kRouteCopied  other fp16 / bool masks: copied with 16-byte rows into the
//                workspace first (mask_pad_kernel), then staged;
//  kRouteF32     fp32 with key stride 1: the main kernel in half steps
//                (position bias [1, 16, 777, 777], B 2, D 64: 59.3 us by
//                kRouteVt, 22.9 here; [1, 32, 2048, 2048], 32 / 8 heads, D 128:
//                489 and 192);
//  kRouteVt      other fp32 masks (or a slice, or a copy's, past 2 GiB): the
//                per-wavefront kernel, V through the workspace.
enum MaskRoute { kRouteNone, kRouteStaged, kRouteCopied, kRouteF32, kRouteVt };

struct MaskPlan {
  MaskRoute route = kRouteNone;
  int64_t esz = 1;
  int64_t sb = 0, sh = 0, sq = 0;        // strides as staged, elements
  int64_t span = 0;                      // bytes of one (sequence, head) slice as staged
  int64_t bm = 1, hm = 1, qm = 1, pitch = 0;  // kRouteCopied: extents kept, row pitch (bytes)
  size_t copy_bytes = 0;
  bool wide = false;                     // kRouteF32: slices of whole 16-byte units
};

MaskPlan plan_mask(const void* mask, int kind, const int64_t* ms, int B, int Hq, int Sq, int Skv) {
  MaskPlan p;
  if (kind == kNoMask) return p;
  if (kind == kMaskF32) {
    p.esz = 4;
    p.sb = ms[0];
    p.sh = ms[1];
    p.sq = ms[2];
    p.span = Sq > 0 && Skv > 0 ? ((static_cast<int64_t>(Sq) - 1) * ms[2] + Skv) * 4 : 0;
    p.route = ms[3] == 1 && p.span <= kBufRange ? kRouteF32 : kRouteVt;
    p.wide = aligned16(mask) && ms[0] % 4 == 0 && ms[1] % 4 == 0 && ms[2] % 4 == 0 && Skv % 4 == 0;
    return p;
  }
  const int64_t esz = p.esz = kind == kMaskF16 ? 2 : 1;
  if (Sq == 0 || Skv == 0) {  // nothing of the mask is read
    p.route = kRouteStaged;
    return p;
  }
  // Staged as it lies only if every slice ends on a whole 16-byte unit: the
  // kernel loads whole units and the descriptor's range ends with the slice,
  // so a unit straddling the end would arrive as zeros, valid keys included.
  const int64_t span = ((static_cast<int64_t>(Sq) - 1) * ms[2] + Skv) * esz;
  if (ms[3] == 1 && aligned16(mask) && (ms[0] * esz) % 16 == 0 && (ms[1] * esz) % 16 == 0 &&
      (ms[2] * esz) % 16 == 0 && (Skv * esz) % 16 == 0 && span <= kBufRange) {
    p.route = kRouteStaged;
    p.span = span;
    p.sb = ms[0];
    p.sh = ms[1];
    p.sq = ms[2];
    return p;
  }
  p.bm = ms[0] != 0 ? B : 1;
  p.hm = ms[1] != 0 ? Hq : 1;
  p.qm = ms[2] != 0 ? Sq : 1;
  p.pitch = (static_cast<int64_t>(Skv) * esz + 15) / 16 * 16;
  p.span = p.qm * p.pitch;  // whole rows: the copy holds the last row's padding
  if (p.span > kBufRange) {
    p.route = kRouteVt;
    return p;
  }
  p.route = kRouteCopied;
  p.copy_bytes = static_cast<size_t>(p.bm * p.hm * p.qm * p.pitch);
  const int64_t pe = p.pitch / esz;  // row pitch, elements
  p.sq = p.qm > 1 ? pe : 0;
  p.sh = p.hm > 1 ? p.qm * pe : 0;
  p.sb = p.bm > 1 ? p.hm * p.qm * pe : 0;
  return p;
}

// Bytes of a mask's rows of `pack` consecutive q heads as staged.
int64_t mask_extent(const MaskPlan& mp, int pack) { return mp.span + (pack - 1) * mp.sh * mp.esz; }

// The workspace of a copied mask: the copy, then (256-byte aligned) a key
// split's partials.
size_t copy_room(const MaskPlan& mp) {
  return mp.route == kRouteCopied ? (mp.copy_bytes + 255) / 256 * 256 : 0;
}

// The least workspace a masked call accepts (spyre_sdpa_fwd_min_workspace_bytes)
// or, for a copied mask, its copy.
size_t min_room(const MaskPlan& mp, int B, int Hkv, int Skv, int D) {
  return mp.route == kRouteCopied ? mp.copy_bytes
         : mp.route >= kRouteF32  ? static_cast<size_t>(B) * Hkv * D * s64_of(Skv) * sizeof(_Float16)
                                  : 0;
}

// The grid of a staged or copied mask's call given ws_bytes beyond the copy.
GridPlan masked_grid(const MaskPlan& mp, int kind, int B, int Hq, int Hkv, int Sq, int Skv, int D, size_t ws_bytes) {
  return plan_grid(B, Hq, Hkv, Sq, Skv, D, false, ws_bytes, kind, mask_extent(mp, Hq / Hkv) <= kBufRange);
}

// Compute units of the current device, cached per device; 0 if the runtime
// cannot say.
int device_cus() {
  static std::atomic<int> cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  int v = cache[dev].load(std::memory_order_relaxed);
  if (v > 0) return v;
  if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) return 0;
  cache[dev].store(v, std::memory_order_relaxed);
  return v;
}

// Rows per query for a call without a mask: the largest divisor p of g whose
// packed grid (B Hkv (g / p) ceil(p Sq / 256) blocks) still gives every
// compute unit a block, so packing never idles units.
int pack_heads(int B, int Hkv, int g, int Sq) {
  if (Sq >= kQB || g == 1) return 1;
  const int64_t cus = device_cus() > 0 ? device_cus() : 256;
  for (int p = g; p > 1; --p) {
    if (g % p) continue;
    const int64_t blocks = static_cast<int64_t>(B) * Hkv * (g / p) * ((static_cast<int64_t>(p) * Sq + kQB - 1) / kQB);
    if (blocks >= cus) return p;
  }
  return 1;
}

int64_t s64_of(int Skv) { return (static_cast<int64_t>(Skv) + kStick - 1) / kStick * kStick; }

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace

extern "C" size_t spyre_sdpa_fwd_workspace_bytes(int B, int Hkv, int Skv, int D) {
  if (B <= 0 || Hkv <= 0 || Skv < 0 || D <= 0) return 0;
  return static_cast<size_t>(B) * Hkv * D * s64_of(Skv) * sizeof(_Float16);
}

// The workspace of a call; own: of spyre_sdpa_fwd_own_f16, which asks for
// nothing that the kernels the call runs leave alone.
static size_t call_workspace(bool own, const void* attn_mask, int mask_kind, const int64_t* mask_strides, int B, int Hq,
                             int Hkv, int Sq, int Skv, int D) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv || Sq < 0 || Skv < 0 || (D != 64 && D != 128)) return 0;
  if (mask_kind == kNoMask) {  // a key split's partials (calls without the causal flag)
    const size_t split = plan_grid(B, Hq, Hkv, Sq, Skv, D, false, SIZE_MAX).part_bytes;
    const spyre_hip::DenseDecodePlan dp = dense_route(B, Hq, Hkv, Sq, Skv, D, false, mask_kind, nullptr);
    return dp.ok ? std::max(split, dp.ws_bytes) : split;  // the split for calls the decode route refuses
  }
  if (!mask_strides || mask_kind < kNoMask || mask_kind > kMaskBool) return 0;
  const MaskPlan mp = plan_mask(attn_mask, mask_kind, mask_strides, B, Hq, Sq, Skv);
  // Decode that reads the mask as it lies takes its partials alone; the
  // shared entry also asks for what the kernels that stage or copy the mask
  // would need.
  GridPlan gs;
  if (mask_strides[3] == 1 && short_grid(B, Hq, Hkv, Sq, Skv, D, SIZE_MAX, gs))
    return own ? gs.part_bytes : std::max(gs.part_bytes, min_room(mp, B, Hkv, Skv, D));
  const spyre_hip::DenseDecodePlan dp = dense_route(B, Hq, Hkv, Sq, Skv, D, false, mask_kind, mask_strides);
  const size_t decode = dp.ok ? dp.ws_bytes : 0;
  const size_t vt = spyre_sdpa_fwd_workspace_bytes(B, Hkv, Skv, D);
  if (mp.route == kRouteVt) return std::max(decode, vt);
  const size_t part = masked_grid(mp, mask_kind, B, Hq, Hkv, Sq, Skv, D, SIZE_MAX).part_bytes;
  if (mp.route == kRouteF32) return std::max({decode, part, own ? 0 : vt});
  return std::max(decode, part ? copy_room(mp) + part : mp.copy_bytes);
}

extern "C" size_t spyre_sdpa_fwd_call_workspace_bytes(const void* attn_mask, int mask_kind,
                                                      const int64_t* mask_strides, int B, int Hq, int Hkv,
                                                      int Sq, int Skv, int D) {
  return call_workspace(false, attn_mask, mask_kind, mask_strides, B, Hq, Hkv, Sq, Skv, D);
}

extern "C" size_t spyre_sdpa_fwd_own_workspace_bytes(const void* attn_mask, int mask_kind,
                                                     const int64_t* mask_strides, int B, int Hq, int Hkv,
                                                     int Sq, int Skv, int D) {
  return call_workspace(true, attn_mask, mask_kind, mask_strides, B, Hq, Hkv, Sq, Skv, D);
}

extern "C" size_t spyre_sdpa_fwd_min_workspace_bytes(const void* attn_mask, int mask_kind,
                                                     const int64_t* mask_strides, int B, int Hq, int Hkv,
                                                     int Sq, int Skv, int D) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv || Sq < 0 || Skv < 0 || (D != 64 && D != 128)) return 0;
  if (!mask_strides || mask_kind <= kNoMask || mask_kind > kMaskBool) return 0;
  const MaskPlan mp = plan_mask(attn_mask, mask_kind, mask_strides, B, Hq, Sq, Skv);
  if (mp.route == kRouteStaged) return 0;
  const size_t vt = spyre_sdpa_fwd_workspace_bytes(B, Hkv, Skv, D);
  return mp.route == kRouteCopied ? std::min(mp.copy_bytes, vt) : vt;
}

// own: no other call in flight uses the workspace.
static int sdpa_fwd(bool own, const void* q, const int64_t* q_strides, const void* k, const int64_t* k_strides,
                    const void* v, const int64_t* v_strides, const void* attn_mask, int mask_kind,
                    const int64_t* mask_strides, int is_causal, float scale, void* out, float* lse, void* workspace,
                    size_t workspace_bytes, int B, int Hq, int Hkv, int Sq, int Skv, int D, void* stream) {
  spyre_hip::clear_error();
  SPYRE_REQUIRE(q_strides && k_strides && v_strides, SPYRE_EINVAL, "null stride argument");
  SPYRE_REQUIRE((Sq == 0 || (q && out)) && (Skv == 0 || (k && v)), SPYRE_EINVAL,
                "null pointer argument");
  SPYRE_REQUIRE(B > 0 && Hq > 0 && Hkv > 0 && Hq % Hkv == 0 && Sq >= 0 && Skv >= 0, SPYRE_EINVAL,
                "bad shape B=%d Hq=%d Hkv=%d Sq=%d Skv=%d", B, Hq, Hkv, Sq, Skv);
  SPYRE_REQUIRE(D == 64 || D == 128, SPYRE_EUNSUPPORTED, "head_dim %d not in {64, 128}", D);
  SPYRE_REQUIRE(mask_kind >= kNoMask && mask_kind <= kMaskBool, SPYRE_EINVAL, "bad mask kind %d",
                mask_kind);
  SPYRE_REQUIRE(mask_kind == kNoMask || (attn_mask && mask_strides), SPYRE_EINVAL,
                "mask pointer / strides missing");
  SPYRE_REQUIRE(!(is_causal && mask_kind != kNoMask), SPYRE_EINVAL,
                "is_causal and an attention mask are exclusive");
  SPYRE_REQUIRE(B <= 65535 && Hq <= 65535, SPYRE_EUNSUPPORTED, "B or Hq above 65535");
  // 16-byte rows: every operand row is read as whole 16-byte vectors.
  SPYRE_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out), SPYRE_EINVAL,
                "q, k, v, out must be 16-byte aligned");
  for (int i = 0; i < 3; ++i)
    SPYRE_REQUIRE(q_strides[i] % 8 == 0 && k_strides[i] % 8 == 0 && v_strides[i] % 8 == 0 &&
                      q_strides[i] >= 0 && k_strides[i] >= 0 && v_strides[i] >= 0,
                  SPYRE_EINVAL, "q/k/v strides must be non-negative multiples of 8 elements");
  if (mask_kind != kNoMask) {
    for (int i = 0; i < 4; ++i)
      SPYRE_REQUIRE(mask_strides[i] >= 0, SPYRE_EINVAL, "negative mask stride");
    SPYRE_REQUIRE(static_cast<int64_t>(Skv) * mask_strides[3] < (int64_t{1} << 31), SPYRE_EUNSUPPORTED,
                  "mask row spans 2^31 elements or more");
    const uintptr_t esz = mask_kind == kMaskF32 ? 4 : mask_kind == kMaskF16 ? 2 : 1;
    SPYRE_REQUIRE(reinterpret_cast<uintptr_t>(attn_mask) % esz == 0, SPYRE_EINVAL,
                  "mask pointer not aligned to its element");
  }
  // The mask's route (plan_mask); a masked call whose workspace holds V's
  // relayout but not the mask's copy takes the per-wavefront kernel.
  MaskPlan mp = plan_mask(attn_mask, mask_kind, mask_strides, B, Hq, Sq, Skv);
  if (mp.route == kRouteCopied && (!workspace || workspace_bytes < mp.copy_bytes || !aligned16(workspace)))
    mp.route = kRouteVt;
  // A shared workspace stays untouched by calls whose mask is staged as it
  // lies, so these may overlap; such a call has no key split.
  const bool staged = mask_kind != kNoMask && mp.route == kRouteStaged;
  const size_t ws_room = workspace && aligned16(workspace) && (own || !staged) ? workspace_bytes : 0;
  // Decode that reads its mask as it lies: no copy, no relayout of V.
  const bool direct = mask_kind == kNoMask || mask_strides[3] == 1;
  const spyre_hip::DenseDecodePlan dp =
      direct ? dense_route(B, Hq, Hkv, Sq, Skv, D, is_causal != 0, mask_kind, mask_strides) : spyre_hip::DenseDecodePlan{};
  const bool dense = dp.ok && k_strides[2] < (int64_t{1} << 23) && v_strides[2] < (int64_t{1} << 23) &&
                     (k_strides[2] == 0 || k_strides[2] >= D) && (v_strides[2] == 0 || v_strides[2] >= D) &&
                     (dp.ws_bytes == 0 || ws_room >= dp.ws_bytes);
  GridPlan gs;
  const bool as_it_lies = mask_kind != kNoMask && direct && (dense || short_grid(B, Hq, Hkv, Sq, Skv, D, ws_room, gs));
  // (The shared entry asks for V's relayout for every fp32 mask and for a
  // copied mask's copy whichever kernel runs.)
  const size_t vt_bytes = spyre_sdpa_fwd_workspace_bytes(B, Hkv, Skv, D);
  const size_t need = own && as_it_lies                             ? 0
                      : mp.route == kRouteCopied                    ? mp.copy_bytes
                      : mp.route >= (own ? kRouteVt : kRouteF32) ? vt_bytes
                                                                    : 0;
  SPYRE_REQUIRE(need == 0 || (workspace && workspace_bytes >= need && aligned16(workspace)),
                SPYRE_ENOSPC, "workspace %zu < %zu bytes (or misaligned)", workspace_bytes, need);
  if (Sq == 0) return SPYRE_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (as_it_lies) mp.route = kRouteNone;
  const bool lds_path = mp.route != kRouteVt;
  // Short query runs pack q heads of a KV head into one block's rows, so
  // they share each K / V tile (decode: one block per (sequence, KV head)
  // instead of g mostly idle ones).
  // And (plan_grid) a key split when the blocks would not fill the device
  // and the workspace holds its partials (after a mask's copy).
  const size_t part_at = copy_room(mp);
  const size_t part_room = ws_room > part_at ? ws_room - part_at : 0;
  GridPlan gpl;
  if (lds_path && !dense)
    gpl = as_it_lies               ? gs
          : mask_kind == kNoMask ? plan_grid(B, Hq, Hkv, Sq, Skv, D, is_causal != 0, part_room)
                                 : masked_grid(mp, mask_kind, B, Hq, Hkv, Sq, Skv, D, part_room);
  // Grids of half steps need no copy: they read rows of any alignment and
  // of at least 16 bytes.
  bool any_rows = false;
  if (mp.route == kRouteCopied && (gpl.shape == kHalf8 || gpl.shape == kHalf4) && mask_strides[3] == 1 && Skv * mp.esz >= 16 &&
      ((Sq - 1) * mask_strides[2] + (gpl.pack - 1) * mask_strides[1] + Skv) * mp.esz <= kBufRange) {
    any_rows = true;
    mp.route = kRouteStaged;
    mp.sb = mask_strides[0];
    mp.sh = mask_strides[1];
    mp.sq = mask_strides[2];
  }
  const int s64 = static_cast<int>(s64_of(Skv));
  const void* mask_ptr = attn_mask;
  if (mp.route == kRouteCopied) {
    const MaskPadArgs pa{static_cast<const char*>(attn_mask), static_cast<char*>(workspace), mask_strides[0],
                         mask_strides[1], mask_strides[2], mask_strides[3], 0, static_cast<int>(mp.hm),
                         static_cast<int>(mp.qm), static_cast<int>(mp.pitch / 16), Skv, {}, {}, {}};
    const int rc = mask_kind == kMaskF16 ? launch_mask_pad<2>(pa, mp.bm, st) : launch_mask_pad<1>(pa, mp.bm, st);
    if (rc != SPYRE_OK) return rc;
    mask_ptr = workspace;
  }
  if (Skv > 0 && !lds_path) {
    VtArgs va{static_cast<const _Float16*>(v), v_strides[0], v_strides[1], v_strides[2],
              static_cast<_Float16*>(workspace), Hkv, Skv, s64, D,
              static_cast<int64_t>(B) * Hkv * (s64 / 64) * (D / 64)};
    const int64_t blocks = (va.tiles + kWaves - 1) / kWaves;
    SPYRE_REQUIRE(blocks < (int64_t{1} << 31), SPYRE_EUNSUPPORTED, "V too large");
    v_token_sticks_kernel<<<dim3(static_cast<unsigned>(blocks)), kThreads, 0, st>>>(va);
    const hipError_t e = hipGetLastError();
    SPYRE_REQUIRE(e == hipSuccess, SPYRE_EHIP, "V restick launch failed: %s", hipGetErrorString(e));
  }
  FwdArgs fa{};
  fa.q = static_cast<const _Float16*>(q);
  fa.k = static_cast<const _Float16*>(k);
  fa.vt = static_cast<const _Float16*>(workspace);
  fa.q_sb = q_strides[0];
  fa.q_sh = q_strides[1];
  fa.q_ss = q_strides[2];
  fa.k_sb = k_strides[0];
  fa.k_sh = k_strides[1];
  fa.k_ss = k_strides[2];
  fa.vt_sb = static_cast<int64_t>(Hkv) * D * s64;
  fa.vt_sh = static_cast<int64_t>(D) * s64;
  // Buffer extents (bytes) of one head: K and V rows 0..Skv-1, Vt [D, s64].
  const int64_t k_span = Skv > 0 ? ((static_cast<int64_t>(Skv) - 1) * k_strides[2] + D) * 2 : 0;
  const int64_t v_span = Skv > 0 ? ((static_cast<int64_t>(Skv) - 1) * v_strides[2] + D) * 2 : 0;
  const int64_t vt_span = static_cast<int64_t>(D) * s64 * 2;
  SPYRE_REQUIRE(k_span <= kBufRange && v_span <= kBufRange && vt_span <= kBufRange, SPYRE_EUNSUPPORTED,
                "one head of K or V spans 2 GiB or more");
  fa.k_bytes = static_cast<uint32_t>(k_span);
  fa.vt_bytes = static_cast<uint32_t>(vt_span);
  fa.mask = attn_mask;
  fa.mask_kind = mask_kind;
  if (mask_kind != kNoMask) {
    fa.m_sb = mask_strides[0];
    fa.m_sh = mask_strides[1];
    fa.m_sq = mask_strides[2];
    fa.m_sk = mask_strides[3];
  }
  fa.out = static_cast<_Float16*>(out);
  fa.lse = lse;
  fa.B = B;
  fa.Hq = Hq;
  fa.Hkv = Hkv;
  fa.g = Hq / Hkv;
  fa.Sq = Sq;
  fa.Skv = Skv;
  fa.s64 = s64;
  fa.causal = is_causal ? 1 : 0;
  fa.scale_log2 = scale * kLog2e;
  if (lds_path) {
    if (dense)
      return spyre_hip::dense_decode_launch(dp, q, q_strides, k, k_strides, v, v_strides, attn_mask, mask_kind,
                                            mask_strides, out, lse, workspace, B, Hq, Hkv, Skv, D, scale, stream);
    // K/V tiles (and mask blocks) shared through LDS.
    Fwd2Args f2{};
    f2.q = fa.q;
    f2.k = fa.k;
    f2.v = static_cast<const _Float16*>(v);
    f2.q_sb = fa.q_sb;
    f2.q_sh = fa.q_sh;
    f2.q_ss = fa.q_ss;
    f2.k_sb = fa.k_sb;
    f2.k_sh = fa.k_sh;
    f2.k_ss = fa.k_ss;
    f2.v_sb = v_strides[0];
    f2.v_sh = v_strides[1];
    f2.v_ss = v_strides[2];
    f2.out = fa.out;
    f2.lse = fa.lse;
    f2.B = B;
    f2.Hq = Hq;
    f2.Hkv = Hkv;
    f2.g = fa.g;
    f2.Sq = Sq;
    f2.Skv = Skv;
    f2.causal = fa.causal;
    f2.pack = gpl.pack;
    f2.gp = fa.g / f2.pack;
    const int rows = shape_rows(gpl.shape);
    f2.qblocks = static_cast<int>((static_cast<int64_t>(f2.pack) * Sq + rows - 1) / rows);
    f2.nsplit = gpl.nsplit;
    f2.split_keys = gpl.nsplit > 1 ? gpl.split_keys : Skv;
    f2.part = gpl.nsplit > 1 ? reinterpret_cast<float*>(static_cast<char*>(workspace) + part_at) : nullptr;
    const int64_t items = blocks_for(B, Hkv, fa.g, Sq, f2.pack, rows) * f2.nsplit;
    SPYRE_REQUIRE(items < (int64_t{1} << 31), SPYRE_EUNSUPPORTED, "too many query blocks");
    f2.n_items = static_cast<uint32_t>(items);
    f2.by_split = spyre_hip::make_fastdiv(static_cast<uint32_t>(f2.nsplit));
    f2.by_gp = spyre_hip::make_fastdiv(static_cast<uint32_t>(f2.gp));
    f2.by_qblocks = spyre_hip::make_fastdiv(static_cast<uint32_t>(f2.qblocks));
    f2.by_hkv = spyre_hip::make_fastdiv(static_cast<uint32_t>(Hkv));
    f2.by_pack = spyre_hip::make_fastdiv(static_cast<uint32_t>(f2.pack));
    f2.xcd_remap = items % 8 == 0;
    f2.scale_log2 = fa.scale_log2;
    // |scale log2 e| <= 1: q times it stays within fp16, so Q is prescaled.
    const bool prescaled = fabsf(f2.scale_log2) <= 1.f;
    f2.mask = mask_ptr;
    f2.m_sb = as_it_lies ? mask_strides[0] : mp.sb;
    f2.m_sh = as_it_lies ? mask_strides[1] : mp.sh;
    f2.m_sq = as_it_lies ? mask_strides[2] : mp.sq;
    f2.m_bytes = static_cast<uint32_t>(mask_extent(mp, f2.pack));
    f2.m_wide = mp.wide ? 1 : 0;
    if (gpl.short_decode) {
      // One row tile, its keys all in flight at once; a key split merges in
      // the same kernel.
      f2.ticket = spyre_hip::next_call_ticket();
      launch_short(f2, D, prescaled, gpl.waves, mask_kind, st);
    } else {
      auto go = [&](auto mk) {
        constexpr int MK = decltype(mk)::value;
        if constexpr (MK != kNoMask)
          if (any_rows) {
            gpl.shape == kHalf8 ? launch_lds<MK, 2, true, 8, true>(f2, D, prescaled, st)
                                : launch_lds<MK, 2, true, 4, true>(f2, D, prescaled, st);
            return;
          }
        switch (gpl.shape) {
          case k256: launch_lds<MK, 2, false, 8>(f2, D, prescaled, st); break;
          case kHalf8: launch_lds<MK, MK == kNoMask ? 4 : 2, true, 8>(f2, D, prescaled, st); break;
          case k128: launch_lds<MK, 2, false, 4>(f2, D, prescaled, st); break;
          default: launch_lds<MK, 2, true, 4>(f2, D, prescaled, st); break;
        }
      };
      if (mask_kind == kMaskF32) {
        gpl.shape == kHalf8 ? launch_f32<8>(f2, D, st) : launch_f32<4>(f2, D, st);
      } else if (mask_kind == kMaskF16) go(std::integral_constant<int, kMaskF16>{});
      else if (mask_kind == kMaskBool) go(std::integral_constant<int, kMaskBool>{});
      else go(std::integral_constant<int, kNoMask>{});
    }
    if (f2.nsplit > 1 && !gpl.short_decode) {
      const hipError_t e0 = hipGetLastError();
      SPYRE_REQUIRE(e0 == hipSuccess, SPYRE_EHIP, "sdpa launch failed: %s", hipGetErrorString(e0));
      MergeArgs ma{f2.part, f2.out, f2.lse, Hq, Sq, D, f2.nsplit, static_cast<int64_t>(B) * Hq * Sq};
      SPYRE_REQUIRE(ma.rows < (int64_t{1} << 31), SPYRE_EUNSUPPORTED, "too many rows");
      // Rows of their own threads once they fill 256 blocks and the splits
      // are few; otherwise a block per row over its splits.
      const int64_t rpb = 256 / (D / 4);
      if (f2.nsplit <= 16 && ma.rows >= 256 * rpb) {
        const dim3 mgrid(static_cast<unsigned>((ma.rows + rpb - 1) / rpb));
        if (D == 128)
          sdpa_split_merge_rows_kernel<128><<<mgrid, 256, 0, st>>>(ma);
        else
          sdpa_split_merge_rows_kernel<64><<<mgrid, 256, 0, st>>>(ma);
      } else {
        const dim3 mgrid(static_cast<unsigned>(ma.rows));
        if (D == 128)
          sdpa_split_merge_kernel<128><<<mgrid, 256, 0, st>>>(ma);
        else
          sdpa_split_merge_kernel<64><<<mgrid, 256, 0, st>>>(ma);
      }
    }
  } else {
    const dim3 grid((Sq + kWaves * kQ - 1) / (kWaves * kQ), Hq, B);
    auto launch = [&](auto mk) {
      constexpr int MK = decltype(mk)::value;
      if (D == 128)
        sdpa_fwd_kernel<128, MK><<<grid, kThreads, 0, st>>>(fa);
      else
        sdpa_fwd_kernel<64, MK><<<grid, kThreads, 0, st>>>(fa);
    };
    switch (mask_kind) {
      case kMaskF16: launch(std::integral_constant<int, kMaskF16>{}); break;
      case kMaskF32: launch(std::integral_constant<int, kMaskF32>{}); break;
      default: launch(std::integral_constant<int, kMaskBool>{}); break;
    }
  }
  const hipError_t e = hipGetLastError();
  SPYRE_REQUIRE(e == hipSuccess, SPYRE_EHIP, "sdpa launch failed: %s", hipGetErrorString(e));
  return SPYRE_OK;
}

#define SPYRE_SDPA_ARGS                                                                                            \
  q, q_strides, k, k_strides, v, v_strides, attn_mask, mask_kind, mask_strides, is_causal, scale, out, lse, workspace, \
      workspace_bytes, B, Hq, Hkv, Sq, Skv, D, stream

extern "C" int spyre_sdpa_fwd_f16(const void* q, const int64_t* q_strides, const void* k,
                                  const int64_t* k_strides, const void* v, const int64_t* v_strides,
                                  const void* attn_mask, int mask_kind, const int64_t* mask_strides,
                                  int is_causal, float scale, void* out, float* lse,
                                  void* workspace, size_t workspace_bytes, int B, int Hq, int Hkv,
                                  int Sq, int Skv, int D, void* stream) {
  return sdpa_fwd(false, SPYRE_SDPA_ARGS);
}

extern "C" int spyre_sdpa_fwd_own_f16(const void* q, const int64_t* q_strides, const void* k,
                                      const int64_t* k_strides, const void* v, const int64_t* v_strides,
                                      const void* attn_mask, int mask_kind, const int64_t* mask_strides,
                                      int is_causal, float scale, void* out, float* lse,
                                      void* workspace, size_t workspace_bytes, int B, int Hq, int Hkv,
                                      int Sq, int Skv, int D, void* stream) {
  return sdpa_fwd(true, SPYRE_SDPA_ARGS);
}
#undef SPYRE_SDPA_ARGS
