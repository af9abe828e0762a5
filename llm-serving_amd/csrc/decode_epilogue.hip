// Decode-step attention epilogue of one layer, fused: per-head RMSNorm of q and k, NeoX
// RoPE at each row's position, q out contiguous for the paged decode, k and v scattered into
// the paged pool at each row's write slot.
//
// The reference runs these as separate tensor ops between the projections and the paged
// decode: q_norm / k_norm (RMSNorm, reference model/layers.py:342-350, applied at :193-194),
// apply_rotary_emb (:59-89, applied at :210-211), then PagedKV.write, whose slot scatter is
// mi_kv_slot_write (model/paged.py:503-520). At the decode shape (B = 32 rows, 16 + 8 + 8
// heads of 128) every one of those ops is a few microseconds of launch for kilobytes of
// data; here the whole epilogue is one launch.
//
// Arithmetic follows the reference's tensor ops step by step in the activation dtype: each
// elementwise result is rounded to the dtype as the op it restates would store it (x^2, the
// mean, mean + eps, its square root, x / rms, (x / rms) * w, and each product and sum of the
// rotation), with the mean's sum accumulated in fp32 as the reduction kernel does. The
// result equals the tensor-op chain's except where the fp32 sum's order moves a rounding
// boundary.
//
// With k_out / v_out the roped k and the v of each row are also written packed, (B, H_kv, D)
// contiguous, for a packed prefill's attention (the decode reads them from the pool).
//
// Two q/k norms: norm_mode 0 is the Qwen3 RMSNorm above (x / rms * w, op by op in T);
// norm_mode 1 is Qwen3.5's zero-centred norm (reference model/qwen35.py:67-89): x * (1 /
// sqrt(mean(x^2) + eps)) * (1 + w), all in fp32 and rounded to T once. RoPE rotates the first
// rotary_dim elements of each head (pairs (e, e + rotary_dim/2), NeoX halves of the rotated
// slice, reference model/layers.py:91-117) and passes the rest through; rotary_dim == D is
// the whole-head rotation of Qwen3, 64 of 256 is Qwen3.5's partial RoPE.
//
// Layout: one wave per (row, head) over q, k and v heads of a packed projection row
// [q (H x D) | k (H_kv x D) | v (H_kv x D)] (a longer row stride leaves room for further
// columns, such as Qwen3.5's output gate); lane l holds elements l, l + 64, ... (coalesced
// loads and stores); a rotation partner is in the same lane when rotary_dim/2 is a multiple
// of 64 and in lane l ^ 32 when it is 32. The projection rows are T, or fp32 split-K partial
// sums [parts][B][row_stride] of mi_rows_gemm, summed in split order and rounded once to T
// (the value the projection's own output would hold).
#include <initializer_list>
#include <type_traits>

#include "common.h"

namespace miattn {
namespace {

// Which q/k norm the epilogue applies (see the file comment).
enum NormMode { kNormQwen3 = 0, kNormZeroCentred = 1 };

template <typename T, int D, typename IdxT, int kU>
__global__ __launch_bounds__(256) void qk_norm_rope_write_kernel(
    const void* __restrict__ qkv, int64_t row_stride, int parts, int64_t plane, const T* __restrict__ q_w,
    const T* __restrict__ k_w, const T* __restrict__ cos_tab, const T* __restrict__ sin_tab, int64_t n_pos,
    int rotary, const int64_t* __restrict__ pos, const IdxT* __restrict__ slots, T* __restrict__ q_out,
    T* __restrict__ k_pool, T* __restrict__ v_pool, T* __restrict__ k_out, T* __restrict__ v_out, int B, int H,
    int H_kv, int64_t n_slots, float eps, int norm_mode, int32_t* __restrict__ err) {
  constexpr int NE = D / 64;  // elements per lane: lane l holds e = l + 64 j, j < NE
  const int lane = threadIdx.x & 63;
  const int head = blockIdx.y * (blockDim.x / 64) + (threadIdx.x >> 6);  // over q, k, v heads
  const int b = blockIdx.x;
  const int n_heads = H + 2 * H_kv;
  if (head >= n_heads || b >= B) return;  // wave-uniform
  // slot -1 marks a row with nothing to write this step (an idle or refused seat of a decode
  // step): skipped silently. Any other row whose position is outside the RoPE table or whose
  // slot is outside the pool is not written to the pool and is reported (row + 1) through
  // the error word. Either way the row's packed outputs (q_out, and k_out / v_out when given)
  // are zero-filled, so a consumer that reads every row reads defined values.
  const int64_t pb = pos[b];
  const IdxT slot = slots[b];
  const bool idle = slot == IdxT(-1);
  if (idle || pb < 0 || pb >= n_pos || !(slot >= 0 && int64_t(slot) < n_slots)) {
    if (!idle && lane == 0 && head == 0 && err != nullptr) atomicCAS(err, 0, b + 1);
    T* row = nullptr;
    if (head < H) {
      row = q_out + (int64_t(b) * H + head) * D;
    } else if (head < H + H_kv) {
      if (k_out != nullptr) row = k_out + (int64_t(b) * H_kv + (head - H)) * D;
    } else if (v_out != nullptr) {
      row = v_out + (int64_t(b) * H_kv + (head - H - H_kv)) * D;
    }
    if (row != nullptr) {
#pragma unroll
      for (int j = 0; j < NE; ++j) row[lane + 64 * j] = from_f32<T>(0.0f);
    }
    return;
  }
  const int64_t src = int64_t(b) * row_stride + int64_t(head) * D;
  // every load of this wave's inputs first, then the arithmetic (the rounding helper's empty
  // asm is a scheduling barrier)
  constexpr int kP = kU < 0 ? 1 : kU;
  PartSum<kP> raw[NE];
#pragma unroll
  for (int j = 0; j < NE; ++j) {
    const int e = lane + 64 * j;
    if constexpr (kU < 0) {
      raw[j].v[0] = to_f32(static_cast<const T*>(qkv)[src + e]);
    } else {
      raw[j].load(static_cast<const float*>(qkv) + src + e, parts, plane);
    }
  }
  // norm weights and this row's RoPE table entries (read here, used after the reduction);
  // the tables hold rotary/2 angles per position: element e < rotary uses angle e mod half
  const bool is_q = head < H;
  const int half = rotary >> 1;
  const T* w = is_q ? q_w : k_w;
  float wt[NE], cs[NE], sn[NE];
#pragma unroll
  for (int j = 0; j < NE; ++j) {
    const int e = lane + 64 * j;
    const int a = e < half ? e : (e < rotary ? e - half : 0);
    wt[j] = to_f32(w[e]);
    cs[j] = to_f32(cos_tab[pb * half + a]);
    sn[j] = to_f32(sin_tab[pb * half + a]);
  }
  float x[NE];
#pragma unroll
  for (int j = 0; j < NE; ++j) {
    if constexpr (kU < 0) x[j] = raw[j].v[0];
    else x[j] = rt<T>(raw[j].sum(parts));
  }

  if (head >= H + H_kv) {  // v head: copied as is (exact: x holds T values)
    const int vh = head - H - H_kv;
    T* dst = v_pool + (int64_t(slot) * H_kv + vh) * D;
    T* dst2 = v_out != nullptr ? v_out + (int64_t(b) * H_kv + vh) * D : nullptr;
#pragma unroll
    for (int j = 0; j < NE; ++j) {
      dst[lane + 64 * j] = from_f32<T>(x[j]);
      if (dst2 != nullptr) dst2[lane + 64 * j] = from_f32<T>(x[j]);
    }
    return;
  }

  float y[NE];  // normed head, T values
  if (norm_mode == kNormQwen3) {
    // x / sqrt(mean(x^2) + eps) * w, each op rounded to T, the squares summed in fp32
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < NE; ++j) ss += rt<T>(x[j] * x[j]);
    ss = group_allreduce<64, SumOp>(ss);
    const float ms = rt<T>(ss * (1.0f / D));
    const float rms = rt<T>(sqrtf(rt<T>(ms + eps)));
#pragma unroll
    for (int j = 0; j < NE; ++j) y[j] = rt<T>(rt<T>(x[j] / rms) * wt[j]);
  } else {
    // zero-centred weight, all in fp32, rounded once: x * (1 / sqrt(mean(x^2) + eps)) * (1 + w)
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < NE; ++j) ss += x[j] * x[j];
    ss = group_allreduce<64, SumOp>(ss);
    const float r = 1.0f / sqrtf(ss * (1.0f / D) + eps);
#pragma unroll
    for (int j = 0; j < NE; ++j) y[j] = rt<T>((x[j] * r) * (1.0f + wt[j]));
  }
  // NeoX RoPE over the first `rotary` elements: pairs (e, e + half); the partner is in this
  // lane at j ^ (half / 64) when half >= 64, else in lane ^ 32 (half = 32)
  float o[NE];
#pragma unroll
  for (int j = 0; j < NE; ++j) {
    const float across = swap32(y[j]);
    float partner = across;
    if constexpr (NE > 1) if (half == 64) partner = y[j ^ 1];
    if constexpr (NE > 2) if (half == 128) partner = y[j ^ 2];
    const int e = lane + 64 * j;
    if (e < half) {
      o[j] = rt<T>(rt<T>(y[j] * cs[j]) - rt<T>(partner * sn[j]));
    } else if (e < rotary) {
      o[j] = rt<T>(rt<T>(partner * sn[j]) + rt<T>(y[j] * cs[j]));
    } else {
      o[j] = y[j];
    }
  }

  T* dst;
  T* dst2 = nullptr;  // the packed k copy, when asked for
  if (is_q) {
    dst = q_out + (int64_t(b) * H + head) * D;
  } else {
    dst = k_pool + (int64_t(slot) * H_kv + (head - H)) * D;
    if (k_out != nullptr) dst2 = k_out + (int64_t(b) * H_kv + (head - H)) * D;
  }
#pragma unroll
  for (int j = 0; j < NE; ++j) {
    dst[lane + 64 * j] = from_f32<T>(o[j]);
    if (dst2 != nullptr) dst2[lane + 64 * j] = from_f32<T>(o[j]);
  }
}

// The same epilogue over a T projection (no partial sums) with 16-byte accesses, for 16-bit
// types: a head is D / 8 consecutive lanes, lane c holding elements 8c .. 8c + 7, and a
// workgroup walks one row's heads, so position, slot, RoPE entries and norm weights are
// loaded once per row instead of once per (row, head). Bound by memory: a packed group of T
// tokens moves T x (2 H + 6 H_kv) x D values. Measured (bf16, graph replay, with the packed k/v
// copies) against the kernel above, which moves one 2-byte element per lane per access and
// divides for each: 8192 tokens at H 16 / H_kv 8 / D 128 82.7 -> 37.2 us (168 MB, 4.5 TB/s; a
// large copy reaches 5.1), at 8 / 2 / 256 47.7 -> 33.3, 4311 tokens 44.0 -> 22.8. The
// projection is read and the pool written with the nontemporal hint (39.2 -> 37.2 us at 8192
// tokens): the next reader of either is far away; q_out, k_out and v_out are the attention's
// next input and stay cached.
//
// Bit-equal to the kernel above: its lane l sums the squares of elements l, l + 64, ... in that
// order and then runs the 64-lane butterfly l ^ 1, ^ 2, ... ^ 32. Here the elements l + 64 j of
// one l are in lanes c, c + 8, .. (c = l / 8), added in the same order by head_squares(); the
// butterfly's first three levels are the in-lane tree over the 8 elements and the last three
// an 8-lane butterfly over c.
template <int D>
__device__ __forceinline__ float head_squares(const float (&sq)[8], int c) {
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    if constexpr (D == 64) {
      v[j] = sq[j];
    } else if constexpr (D == 128) {
      v[j] = sq[j] + dpp<kDppRowRor8>(sq[j]);
    } else {
      // ((a0 + a1) + a2) + a3 of lanes c, c + 8, c + 16, c + 24 (c < 8), in every one of them
      const float far = swap16(sq[j]);
      const float low = (c & 16) ? far : sq[j], high = (c & 16) ? sq[j] : far;
      const float high8 = dpp<kDppRowRor8>(high);
      v[j] = ((low + dpp<kDppRowRor8>(low)) + ((c & 8) ? high8 : high)) + ((c & 8) ? high : high8);
    }
  }
  return group_allreduce<8, SumOp>(((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])));
}

template <typename T, int D, typename IdxT>
__global__ __launch_bounds__(256) void qk_norm_rope_write_vec_kernel(
    const T* __restrict__ qkv, int64_t row_stride, const T* __restrict__ q_w, const T* __restrict__ k_w,
    const T* __restrict__ cos_tab, const T* __restrict__ sin_tab, int64_t n_pos, int rotary,
    const int64_t* __restrict__ pos, const IdxT* __restrict__ slots, T* __restrict__ q_out, T* __restrict__ k_pool,
    T* __restrict__ v_pool, T* __restrict__ k_out, T* __restrict__ v_out, int H, int H_kv, int64_t n_slots, float eps,
    int norm_mode, int32_t* __restrict__ err) {
  constexpr int E = 8, LPH = D / E, HPW = 256 / LPH;  // lanes per head, heads per workgroup pass
  const int c = threadIdx.x % LPH;
  const int b = blockIdx.x;
  const int n_heads = H + 2 * H_kv;
  const int step = HPW * gridDim.y;
  const int head0 = blockIdx.y * HPW + threadIdx.x / LPH;
  const int64_t pb = pos[b];
  const IdxT slot = slots[b];
  const T* src = qkv + int64_t(b) * row_stride + c * E;
  // the row of each output a head goes to; k and v of a row that is written go to the pool and,
  // when asked for, to the packed copy
  auto packed_row = [&](int head) -> T* {
    if (head < H) return q_out + (int64_t(b) * H + head) * D + c * E;
    T* out = head < H + H_kv ? k_out : v_out;
    return out == nullptr ? nullptr : out + (int64_t(b) * H_kv + (head - H) % H_kv) * D + c * E;
  };
  const bool idle = slot == IdxT(-1);
  if (idle || pb < 0 || pb >= n_pos || !(slot >= 0 && int64_t(slot) < n_slots)) {  // uniform: see the kernel above
    if (!idle && blockIdx.y == 0 && threadIdx.x == 0 && err != nullptr) atomicCAS(err, 0, b + 1);
    for (int head = head0; head < n_heads; head += step) {
      T* row = packed_row(head);
      if (row != nullptr) store16(row, make_uint4(0u, 0u, 0u, 0u));
    }
    return;
  }
  const int half = rotary >> 1;  // 32, 64 or 128: a lane's 8 elements are on one side of it
  const int e0 = c * E;
  const int a0 = e0 < half ? e0 : (e0 < rotary ? e0 - half : 0);
  const uint4 cv = load16(cos_tab + pb * half + a0), sv = load16(sin_tab + pb * half + a0);
  const uint4 wq = load16(q_w + e0), wk = load16(k_w + e0);

  auto finish = [&](int head, const uint4& raw) {
    uint4 result = raw;  // a v head is copied as it is
    if (head < H + H_kv) {
      const uint4 w = head < H ? wq : wk;
      float x[E], sq[E];
#pragma unroll
      for (int j = 0; j < E; ++j) {
        x[j] = Vec16<T>::get(raw, j);
        sq[j] = x[j] * x[j];  // exact: a product of 16-bit values
      }
      if (norm_mode == kNormQwen3) {
        rt8<T>(sq);
        const float ms = rt<T>(head_squares<D>(sq, c) * (1.0f / D));
        div_rt8<T>(x, rt<T>(sqrtf(rt<T>(ms + eps))));
#pragma unroll
        for (int j = 0; j < E; ++j) x[j] *= Vec16<T>::get(w, j);
      } else {
        const float r = 1.0f / sqrtf(head_squares<D>(sq, c) * (1.0f / D) + eps);
#pragma unroll
        for (int j = 0; j < E; ++j) x[j] = (x[j] * r) * (1.0f + Vec16<T>::get(w, j));
      }
      result = rt8<T>(x);  // the normed head
      if (e0 < rotary) {
        // the rotation partner is this element of lane c ^ (half / 8); the first half's lanes take
        // x cos - partner sin, the second's partner sin + x cos
        float p[E];
#pragma unroll
        for (int j = 0; j < E; ++j) {
          p[j] = half == 64 ? dpp<kDppRowRor8>(x[j]) : half == 32 ? swap4(x[j]) : swap16(x[j]);
          p[j] *= Vec16<T>::get(sv, j);
          x[j] *= Vec16<T>::get(cv, j);
        }
        rt8<T>(p);
        rt8<T>(x);
#pragma unroll
        for (int j = 0; j < E; ++j) x[j] = e0 < half ? x[j] - p[j] : x[j] + p[j];
        result = rt8<T>(x);
      }
    }
    T* row = packed_row(head);
    if (row != nullptr) store16(row, result);
    if (head >= H) {
      T* pool = head < H + H_kv ? k_pool : v_pool;
      store16_nt(pool + (int64_t(slot) * H_kv + (head - H) % H_kv) * D + e0, result);
    }
  };
  // two heads' loads at a time ahead of their arithmetic
  for (int head = head0; head < n_heads; head += 2 * step) {
    const int next = head + step;
    const uint4 r0 = load16_nt(src + int64_t(head) * D);
    const uint4 r1 = load16_nt(src + int64_t(next < n_heads ? next : head) * D);
    finish(head, r0);
    if (next < n_heads) finish(next, r1);
  }
}

// Launch arguments shared by every instantiation.
struct EpilogueArgs {
  const void* qkv; int64_t row_stride; int parts; const void* q_w; const void* k_w; const void* cos_tab;
  const void* sin_tab; int64_t n_pos; int rotary; const int64_t* pos; const void* slots; int slot_bits;
  void* q_out; void* k_pool; void* v_pool; void* k_out; void* v_out; int B; int H; int H_kv; int64_t n_slots;
  float eps; int norm_mode; int32_t* err; hipStream_t s;
};

// Whether the 16-byte kernel is the faster one. Below a number of q/k/v values a launch is latency, and
// a lane's eight elements are a longer chain than one or two; a row of few heads leaves most of a
// workgroup empty. bf16 at D 64 and 128: from 2^20 values (H 16 / H_kv 8 / D 128: 256 rows 4.61 -> 4.56 us, 512 6.5 ->
// 5.6, 8192 64 -> 38) and 8 heads (H 4 / H_kv 2 1.05-1.5x, H 2 / H_kv 1 0.92-1.0x). At D 256 the older kernel's lane has
// four elements and loses less, least with the Qwen3.5 norm (one division per head, not one per element): H 8 / H_kv
// 2, 1366 rows 1.06x and 0.98x, 8192 rows 1.18x and 1.07x. fp16 costs a pack for every two roundings and a
// correction for every quotient (D 128: 2^20 values 0.95-0.99x, 2^21 1.02-1.06x; D 256, H 8 / H_kv 2: 2^24 values 0.99x
// and 0.93x, 2^26 1.23x).
template <typename T, int D>
bool vec_faster(int64_t values, int n_heads, int norm_mode) {
  const bool bf16 = std::is_same<T, bf16_t>::value, qwen3 = norm_mode == kNormQwen3;
  if (D == 256) {
    if (bf16) return n_heads >= 10 && values >= (qwen3 ? int64_t(3) << 20 : int64_t(1) << 24);
    return n_heads >= 10 && values >= (qwen3 ? int64_t(1) << 25 : int64_t(1) << 26);
  }
  if (bf16 || D == 64) return n_heads >= 8 && values >= int64_t(1) << 20;
  return n_heads >= 10 && values >= int64_t(1) << 21;
}
// Rows from which one workgroup walks all heads of a row (8192 rows 39.2 against 45.5 us with
// the heads shared out over the grid's y axis); below, they are shared out so that a small
// batch still spreads over the chip (300 rows 4.4 against 5.4 us).
constexpr int kRowPerGroup = 1024;

// Every address the 16-byte kernel touches is a multiple of 16 bytes (rows and heads are
// multiples of 64 elements; the caller's pointers and row stride are what can be off).
bool vec16_ok(const EpilogueArgs& a) {
  uintptr_t all = 0;
  for (const void* p : {a.qkv, a.q_w, a.k_w, a.cos_tab, a.sin_tab, static_cast<const void*>(a.q_out),
                        static_cast<const void*>(a.k_pool), static_cast<const void*>(a.v_pool),
                        static_cast<const void*>(a.k_out), static_cast<const void*>(a.v_out)}) {
    all |= reinterpret_cast<uintptr_t>(p);
  }
  return all % 16 == 0 && a.row_stride % 8 == 0;
}

template <typename T, int D>
int launch_d(const EpilogueArgs& a) {
  if constexpr (sizeof(T) == 2) {
    const int n_heads = a.H + 2 * a.H_kv;
    if (a.parts == 0 && vec_faster<T, D>(int64_t(a.B) * n_heads * D, n_heads, a.norm_mode) && vec16_ok(a)) {
      constexpr int HPW = 256 * 8 / D;  // heads per workgroup pass
      const unsigned groups = (n_heads + HPW - 1) / HPW;
      const dim3 grid(a.B, a.B >= kRowPerGroup ? 1 : groups);
      auto go = [&](auto idx_tag) {
        using IdxT = decltype(idx_tag);
        hipLaunchKernelGGL((qk_norm_rope_write_vec_kernel<T, D, IdxT>), grid, dim3(256), 0, a.s,
                           static_cast<const T*>(a.qkv), a.row_stride, static_cast<const T*>(a.q_w),
                           static_cast<const T*>(a.k_w), static_cast<const T*>(a.cos_tab),
                           static_cast<const T*>(a.sin_tab), a.n_pos, a.rotary, a.pos,
                           static_cast<const IdxT*>(a.slots), static_cast<T*>(a.q_out), static_cast<T*>(a.k_pool),
                           static_cast<T*>(a.v_pool), static_cast<T*>(a.k_out), static_cast<T*>(a.v_out), a.H, a.H_kv,
                           a.n_slots, a.eps, a.norm_mode, a.err);
      };
      if (a.slot_bits == 32) go(int32_t{}); else go(int64_t{});
      return launch_status("mi_qk_norm_rope_write");
    }
  }
  constexpr int kWaves = 4;
  const dim3 grid(a.B, (a.H + 2 * a.H_kv + kWaves - 1) / kWaves);
  const int64_t plane = int64_t(a.B) * a.row_stride;
  auto go = [&](auto idx_tag, auto unroll) {
    using IdxT = decltype(idx_tag);
    hipLaunchKernelGGL((qk_norm_rope_write_kernel<T, D, IdxT, decltype(unroll)::value>), grid, dim3(64 * kWaves), 0,
                       a.s, a.qkv, a.row_stride, a.parts, plane, static_cast<const T*>(a.q_w),
                       static_cast<const T*>(a.k_w), static_cast<const T*>(a.cos_tab),
                       static_cast<const T*>(a.sin_tab), a.n_pos, a.rotary, a.pos, static_cast<const IdxT*>(a.slots),
                       static_cast<T*>(a.q_out), static_cast<T*>(a.k_pool), static_cast<T*>(a.v_pool),
                       static_cast<T*>(a.k_out), static_cast<T*>(a.v_out), a.B, a.H, a.H_kv, a.n_slots, a.eps,
                       a.norm_mode, a.err);
  };
  auto by_slots = [&](auto unroll) {
    if (a.slot_bits == 32) go(int32_t{}, unroll); else go(int64_t{}, unroll);
  };
  switch (parts_unroll(a.parts)) {
    case -1: by_slots(std::integral_constant<int, -1>{}); break;
    case 2: by_slots(std::integral_constant<int, 2>{}); break;
    case 8: by_slots(std::integral_constant<int, 8>{}); break;
    default: by_slots(std::integral_constant<int, 0>{}); break;
  }
  return launch_status("mi_qk_norm_rope_write");
}

template <typename T>
int launch_t(int D, const EpilogueArgs& a) {
  switch (D) {
    case 64: return launch_d<T, 64>(a);
    case 128: return launch_d<T, 128>(a);
    case 256: return launch_d<T, 256>(a);
    default:
      return fail(MI_ERR_UNSUPPORTED, "mi_qk_norm_rope_write: head_dim %d is not supported (64, 128, 256)", D);
  }
}

}  // namespace
}  // namespace miattn

extern "C" int mi_qk_norm_rope_write(const void* qkv, int64_t row_stride, int qkv_parts, const void* q_norm_w,
                                     const void* k_norm_w, const void* cos_tab, const void* sin_tab,
                                     int64_t n_pos, int rotary_dim, const int64_t* pos, const void* slot_ids,
                                     int slot_bits, void* q_out, void* k_pool, void* v_pool, void* k_out,
                                     void* v_out, int B, int H, int H_kv, int D, int64_t n_slots, float eps,
                                     int norm_mode, int dtype, int32_t* error_word, void* stream) {
  using namespace miattn;
  if (B < 0 || H < 1 || H_kv < 1 || H % H_kv != 0) {
    return fail(MI_ERR_INVALID, "mi_qk_norm_rope_write: n_head (%d) must be a multiple of n_kv_head (%d)", H, H_kv);
  }
  if (slot_bits != 32 && slot_bits != 64) {
    return fail(MI_ERR_INVALID, "mi_qk_norm_rope_write: slot_bits must be 32 or 64, got %d", slot_bits);
  }
  if (n_pos < 1) return fail(MI_ERR_INVALID, "mi_qk_norm_rope_write: the RoPE table is empty");
  if (qkv_parts < 0) return fail(MI_ERR_INVALID, "mi_qk_norm_rope_write: qkv_parts %d < 0", qkv_parts);
  if (row_stride < int64_t(H + 2 * H_kv) * D) {
    return fail(MI_ERR_INVALID, "mi_qk_norm_rope_write: row stride %lld < %d packed q/k/v elements",
                (long long)row_stride, (H + 2 * H_kv) * D);
  }
  // the rotation partner of element e < rotary/2 is e + rotary/2: in the same lane when
  // rotary/2 is a multiple of 64, in lane ^ 32 when it is 32
  if (!(rotary_dim == 64 || rotary_dim == 128 || rotary_dim == 256) || rotary_dim > D) {
    return fail(MI_ERR_UNSUPPORTED, "mi_qk_norm_rope_write: rotary_dim %d must be 64, 128 or 256 and <= head_dim %d",
                rotary_dim, D);
  }
  if (norm_mode != 0 && norm_mode != 1) {
    return fail(MI_ERR_INVALID, "mi_qk_norm_rope_write: norm_mode %d is not 0 or 1", norm_mode);
  }
  if (qkv == nullptr || q_norm_w == nullptr || k_norm_w == nullptr || cos_tab == nullptr || sin_tab == nullptr ||
      pos == nullptr || slot_ids == nullptr || q_out == nullptr || k_pool == nullptr || v_pool == nullptr) {
    return fail(MI_ERR_INVALID, "mi_qk_norm_rope_write: NULL pointer argument");
  }
  if (B == 0) return MI_OK;
  const EpilogueArgs a{qkv, row_stride, qkv_parts, q_norm_w, k_norm_w, cos_tab, sin_tab, n_pos, rotary_dim, pos,
                       slot_ids, slot_bits, q_out, k_pool, v_pool, k_out, v_out, B, H, H_kv, n_slots, eps, norm_mode,
                       error_word, static_cast<hipStream_t>(stream)};
  switch (dtype) {
    case MI_BF16: return launch_t<bf16_t>(D, a);
    case MI_F16: return launch_t<f16_t>(D, a);
    case MI_F32: return launch_t<float>(D, a);
    default:
      return fail(MI_ERR_INVALID, "mi_qk_norm_rope_write: unknown dtype %d", dtype);
  }
}
