// Paged KV-cache producer for MI355X (gfx950): rotary embedding of Q and K
// and the paged write of K and V into fp8 (OCP e4m3fn) or 16-bit caches.
//
//  kv_rope_write8<T, CT, CS, ROWS>   the fast path: every Q and K head row of the
//    call is one row of the work; a lane owns eight contiguous dims (16-byte
//    loads and stores), D/8 lanes a row, and each lane takes ROWS rows (one or
//    two by the call's size) with all their loads issued before any arithmetic;
//    row numbers are 32-bit (the 64-bit divisions cost a small call ~0.1 us).  A neox pair partner lies
//    half/8 lanes away in the same row and is exchanged with a lane shuffle;
//    cos and sin arrive as 8 (neox) or 4 (interleaved) consecutive values.
//    Taken when rows, caches and the cos/sin table are 16-byte aligned,
//    head_dim % 8 == 0 and, for neox, rotary_dim % 16 == 0.  Row loads and
//    all row and cache stores are non-temporal: every byte is touched once
//    per call and each wave writes whole 128-byte lines (70.3 vs 75.2 us for
//    a 16K-token chunk of the config-3 shape).
//
//  kv_rope_write<T, CT>   the general path: grid (num_tokens, ceil(max(Hq, Hkv) / 4)), 4 waves.
//    Wave w of workgroup (t, g) owns head h = 4 g + w of token t; lane l owns
//    the four contiguous dims [4 l, 4 l + 4) (head_dim <= 256).  A neox pair
//    partner lies rotary_dim / 2 dims away (another lane's four dims, loaded
//    directly: every load of the wave precedes its stores, so the in-place
//    update is safe); an interleaved partner lies inside the lane's four dims.
//    Arithmetic in fp32 with contraction off -- each product and the sum are
//    rounded separately -- then rounded to the model dtype.  fp8 caches take
//    RNE_e4m3fn(clamp(x / scale, +-448)) via v_cvt_pk_fp8_f32 (one dword per
//    lane); 16-bit caches take the dtype value (8 bytes per lane).
//
//  kv_amax8<T, CS>   the fp8 cache scales, fast path (the layouts of
//    kv_rope_write8): workgroups of 16 waves over chunks of tokens, all heads,
//    K and V read once in whole rows; a workgroup folds its maxima in LDS and
//    combines its scales by atomic maximum (a maximum has no order: the result
//    is deterministic).  kv_amax<T>: the general path, by (head, K or V, chunk).
//
// Reference semantics (paths relative to the reference repo root):
//   integrations/vllm/l20_rope_kv.py:26-137 (interleaved), :140-253 (neox),
//   :256-309 (entry point; 16-bit caches only there);
//   scripts/smoke_cuda_paged_fp8_decode_op.py:13-19 (the fp8 quantiser).

#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>
#include <stdio.h>

#include <algorithm>
#include <type_traits>

#include "l20_kv_write.h"

// Error reporting shared with the decode entry points (l20_pd_last_error).
namespace l20pd_host {
int32_t set_error(int32_t code, const char *msg);
void clear_error();
}  // namespace l20pd_host

namespace l20kv {

typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr float kFp8Max = 448.0f;

struct Params {
  void *q;
  int64_t q_st, q_sh;
  int hq;
  void *k;
  int64_t k_st, k_sh;
  const void *v;
  int64_t v_st, v_sh;
  const int64_t *pos;
  const void *cs;
  int64_t cs_sp;
  int cs_dtype;  // 0 bf16, 1 fp16, 2 fp32
  int rot, neox;
  const int64_t *slots;
  void *kc;
  int64_t kc_sp, kc_st, kc_sh;
  void *vc;
  int64_t vc_sp, vc_st, vc_sh;
  int64_t num_pages;
  float k_scale, v_scale;
  const float *k_scale_ph, *v_scale_ph;
  int tokens, hkv, d;
};

template <typename T> __device__ __forceinline__ float to_f32(T x) { return (float)x; }
template <typename T> __device__ __forceinline__ T from_f32(float x) { return (T)x; }

// Four consecutive elements of type T (8 bytes) as fp32.
template <typename T> __device__ __forceinline__ void load4(const T *p, float (&x)[4]) {
  const i32x2 w = *reinterpret_cast<const i32x2 *>(p);
  const T *e = reinterpret_cast<const T *>(&w);
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = to_f32(e[i]);
}

// Four fp32 -> four T (RNE), packed as two dwords.
template <typename T> __device__ __forceinline__ i32x2 pack4(const float (&x)[4]);
template <> __device__ __forceinline__ i32x2 pack4<__bf16>(const float (&x)[4]) {
  return i32x2{__builtin_bit_cast(int, __builtin_convertvector(f32x2{x[0], x[1]}, bf16x2)),
               __builtin_bit_cast(int, __builtin_convertvector(f32x2{x[2], x[3]}, bf16x2))};
}
template <> __device__ __forceinline__ i32x2 pack4<_Float16>(const float (&x)[4]) {
  return i32x2{__builtin_bit_cast(int, __builtin_convertvector(f32x2{x[0], x[1]}, f16x2)),
               __builtin_bit_cast(int, __builtin_convertvector(f32x2{x[2], x[3]}, f16x2))};
}

// The fp32 values of four packed T (what a store then load would give).
template <typename T> __device__ __forceinline__ void unpack4(i32x2 w, float (&x)[4]) {
  const T *e = reinterpret_cast<const T *>(&w);
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = to_f32(e[i]);
}

__device__ __forceinline__ float cs_load(const Params &p, int64_t position, int idx) {
  const int64_t off = position * p.cs_sp + idx;
  if (p.cs_dtype == 2) return reinterpret_cast<const float *>(p.cs)[off];
  if (p.cs_dtype == 1) return (float)reinterpret_cast<const _Float16 *>(p.cs)[off];
  return (float)reinterpret_cast<const __bf16 *>(p.cs)[off];
}

// Rotate the lane's four dims [e0, e0 + 4) of one head row in fp32.
template <typename T>
__device__ __forceinline__ void rope4(const Params &p, const T *row, int64_t position, int e0, float (&x)[4]) {
#pragma clang fp contract(off)
  load4(row + e0, x);
  if (e0 >= p.rot) return;
  const int half = p.rot >> 1;
  float pr[4], c[4], s[4], sg[4];
  if (p.neox) {
    const bool first = e0 < half;
    load4(row + (first ? e0 + half : e0 - half), pr);
    const int t0 = first ? e0 : e0 - half;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      c[i] = cs_load(p, position, t0 + i);
      s[i] = cs_load(p, position, half + t0 + i);
      sg[i] = first ? -1.0f : 1.0f;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      pr[i] = x[i ^ 1];
      c[i] = cs_load(p, position, (e0 + i) >> 1);
      s[i] = cs_load(p, position, half + ((e0 + i) >> 1));
      sg[i] = (i & 1) ? 1.0f : -1.0f;
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = x[i] * c[i];
    const float b = (pr[i] * s[i]) * sg[i];
    x[i] = a + b;
  }
}

// ---- fast path helpers: eight consecutive elements of T as one 16-byte word ----
template <typename T> __device__ __forceinline__ void unpack8(i32x4 w, float (&x)[8]) {
  const T *e = reinterpret_cast<const T *>(&w);
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = to_f32(e[i]);
}
template <typename T> __device__ __forceinline__ i32x4 pack8(const float (&x)[8]) {
  const float lo[4] = {x[0], x[1], x[2], x[3]};
  const float hi[4] = {x[4], x[5], x[6], x[7]};
  const i32x2 a = pack4<T>(lo), b = pack4<T>(hi);
  return i32x4{a[0], a[1], b[0], b[1]};
}
// The cos and sin of one row's eight dims as loaded (table type CS: 0 bf16, 1
// fp16, 2 fp32), unpacked where they are used: eight consecutive values each
// for a neox pair layout, four (one per pair) for an interleaved one.  Kept as
// loaded, 16-bit tables take 8 registers a row and not 16 (kv_rope_write8 on a
// 16K-token chunk, 32 heads of 128: 65.5 -> 63.2 us).
template <int CS> struct CosSin {
  i32x4 c[CS == 2 ? 2 : 1], s[CS == 2 ? 2 : 1];
};
template <int CS, int N>
__device__ __forceinline__ void load_cs(const void *base, int64_t off, i32x4 (&w)[CS == 2 ? 2 : 1]) {
  if constexpr (CS == 2) {
    const i32x4 *src = reinterpret_cast<const i32x4 *>(reinterpret_cast<const float *>(base) + off);
    w[0] = src[0];
    if constexpr (N == 8) w[1] = src[1];
  } else {
    const uint16_t *src = reinterpret_cast<const uint16_t *>(base) + off;
    if constexpr (N == 8) {
      w[0] = *reinterpret_cast<const i32x4 *>(src);
    } else {
      const i32x2 v = *reinterpret_cast<const i32x2 *>(src);
      w[0] = i32x4{v[0], v[1], 0, 0};
    }
  }
}
// dims [e0, e0 + 8) (e0 < rot) of the row at `pos`
template <int CS>
__device__ __forceinline__ void load_row_cs(const Params &p, int64_t pos, int e0, int half, CosSin<CS> &w) {
  const int64_t base = pos * p.cs_sp;
  if (p.neox) {
    const int t0 = e0 < half ? e0 : e0 - half;
    load_cs<CS, 8>(p.cs, base + t0, w.c);
    load_cs<CS, 8>(p.cs, base + half + t0, w.s);
  } else {
    load_cs<CS, 4>(p.cs, base + (e0 >> 1), w.c);
    load_cs<CS, 4>(p.cs, base + half + (e0 >> 1), w.s);
  }
}
template <int CS> __device__ __forceinline__ void unpack_cs(const i32x4 (&w)[CS == 2 ? 2 : 1], float (&x)[8]) {
  if constexpr (CS == 2) {
    const f32x4 a = __builtin_bit_cast(f32x4, w[0]), b = __builtin_bit_cast(f32x4, w[1]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[i] = a[i];
      x[4 + i] = b[i];
    }
  } else if constexpr (CS == 1) {
    unpack8<_Float16>(w[0], x);
  } else {
    unpack8<__bf16>(w[0], x);
  }
}

// Rotate eight dims x in place; pw holds the neox partner's eight dims, first
// says that x is in the first half of the rotary dims.
template <typename T, int CS>
__device__ __forceinline__ void rotate8(const Params &p, float (&x)[8], i32x4 pw, const CosSin<CS> &w, bool first) {
#pragma clang fp contract(off)
  float y[8], c[8], sn[8];
  unpack_cs<CS>(w.c, c);
  unpack_cs<CS>(w.s, sn);
  if (p.neox) {
    float pr[8];
    unpack8<T>(pw, pr);
    const float sg = first ? -1.0f : 1.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float a = x[i] * c[i];
      const float b = (pr[i] * sn[i]) * sg;
      y[i] = a + b;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float a = x[i] * c[i >> 1];
      const float b = (x[i ^ 1] * sn[i >> 1]) * ((i & 1) ? 1.0f : -1.0f);
      y[i] = a + b;
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] = y[i];
}

// Four values -> four e4m3fn codes in one dword: RNE of clamp(x / scale).
__device__ __forceinline__ int quant4(const float (&x)[4], float scale) {
  float y[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) y[i] = fminf(fmaxf(__fdiv_rn(x[i], scale), -kFp8Max), kFp8Max);
  int w = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], 0, false);
  w = __builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], w, true);
  return w;
}

// Rows [0, rows_q) are Q head rows (token r / Hq, head r % Hq), the next
// rows_k are K head rows (token r / Hkv): rotated in place, and for K also the
// K and V cache writes.  Four waves; a lane group of lpr = D/8 lanes per row.
// POS_FIRST: the positions load ahead of the rows, so that the cos/sin loads wait for
// them alone.  Only for two rows on long streams (launch_fast): 16384 tokens of 28 + 4
// heads, fp8 and bf16 caches, 63.6 -> 62.7 and 63.3 -> 62.5 us; 1050 tokens would go
// from 6.8 to 7.7, and one row gains nothing (4.56, 4.64 at 500).
template <typename T, int CT, int CS, int ROWS, bool POS_FIRST>
__global__ __launch_bounds__(256) void kv_rope_write8(Params p, uint32_t rows_q, uint32_t rows_all) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int lpr = p.d >> 3;     // lanes per row
  const int rpw = 64 / lpr;     // rows per wave and pass
  const int g = lane / lpr;
  const int l = lane - g * lpr;
  const int e0 = 8 * l;
  const int half = p.rot >> 1;
  const bool rot_lane = e0 < p.rot;
  const uint32_t first = blockIdx.x * (uint32_t)(4 * rpw * ROWS);

  // ---- loads of all of this lane's rows ----
  i32x4 xw[ROWS], vw[ROWS];
  int64_t pos[ROWS], slot[ROWS];
  float ksc[ROWS], vsc[ROWS];  // the K row's cache scales (loaded with the row)
  T *row[ROWS];
  int head[ROWS];
  bool live[ROWS], is_k[ROWS];
  if constexpr (POS_FIRST) {
    int64_t tok[ROWS];
#pragma unroll
    for (int u = 0; u < ROWS; ++u) {
      const uint32_t r = first + (uint32_t)((u * 4 + wave) * rpw + g);
      live[u] = g < rpw && r < rows_all;
      is_k[u] = r >= rows_q;
      const uint32_t n = is_k[u] ? r - rows_q : r, heads = (uint32_t)(is_k[u] ? p.hkv : p.hq);
      tok[u] = n / heads;
      head[u] = (int)(n % heads);
      pos[u] = 0;
      if (live[u] && rot_lane) pos[u] = p.pos[tok[u]];
    }
#pragma unroll
    for (int u = 0; u < ROWS; ++u) {
      row[u] = is_k[u] ? reinterpret_cast<T *>(p.k) + tok[u] * p.k_st + (int64_t)head[u] * p.k_sh
                       : reinterpret_cast<T *>(p.q) + tok[u] * p.q_st + (int64_t)head[u] * p.q_sh;
      if (!live[u]) continue;
      xw[u] = __builtin_nontemporal_load(reinterpret_cast<const i32x4 *>(row[u] + e0));
      if (is_k[u]) {
        vw[u] = __builtin_nontemporal_load(reinterpret_cast<const i32x4 *>(
            reinterpret_cast<const T *>(p.v) + tok[u] * p.v_st + (int64_t)head[u] * p.v_sh + e0));
        slot[u] = p.slots[tok[u]];
        if constexpr (CT == 0) {
          ksc[u] = p.k_scale_ph ? p.k_scale_ph[head[u]] : p.k_scale;
          vsc[u] = p.v_scale_ph ? p.v_scale_ph[head[u]] : p.v_scale;
        }
      }
    }
  } else {
#pragma unroll
    for (int u = 0; u < ROWS; ++u) {
      const uint32_t r = first + (uint32_t)((u * 4 + wave) * rpw + g);
      live[u] = g < rpw && r < rows_all;
      is_k[u] = r >= rows_q;
      int64_t t = 0;
      int h = 0;
      if (live[u]) {
        if (!is_k[u]) {
          const uint32_t q = r / (uint32_t)p.hq;
          t = q;
          h = (int)(r - q * (uint32_t)p.hq);
          row[u] = reinterpret_cast<T *>(p.q) + t * p.q_st + (int64_t)h * p.q_sh;
        } else {
          const uint32_t rk = r - rows_q;
          const uint32_t q = rk / (uint32_t)p.hkv;
          t = q;
          h = (int)(rk - q * (uint32_t)p.hkv);
          row[u] = reinterpret_cast<T *>(p.k) + t * p.k_st + (int64_t)h * p.k_sh;
          vw[u] = __builtin_nontemporal_load(reinterpret_cast<const i32x4 *>(reinterpret_cast<const T *>(p.v) + t * p.v_st +
                                                   (int64_t)h * p.v_sh + e0));
          slot[u] = p.slots[t];
          if constexpr (CT == 0) {
            ksc[u] = p.k_scale_ph ? p.k_scale_ph[h] : p.k_scale;
            vsc[u] = p.v_scale_ph ? p.v_scale_ph[h] : p.v_scale;
          }
        }
        xw[u] = __builtin_nontemporal_load(reinterpret_cast<const i32x4 *>(row[u] + e0));
        pos[u] = p.pos[t];
      }
      head[u] = h;
    }
  }
  // ---- cos / sin of the lanes' dims ----
  CosSin<CS> cs[ROWS];
#pragma unroll
  for (int u = 0; u < ROWS; ++u) {
    if (live[u] && rot_lane) load_row_cs<CS>(p, pos[u], e0, half, cs[u]);
  }
  // ---- rotate, store back, write the caches ----
#pragma unroll
  for (int u = 0; u < ROWS; ++u) {
    // the neox partner's words, from the lane half/8 away in the same row (every lane shuffles)
    const int src = g * lpr + (e0 < half ? l + (half >> 3) : l - (half >> 3));
    i32x4 pw;
#pragma unroll
    for (int i = 0; i < 4; ++i) pw[i] = __shfl(xw[u][i], (p.neox && rot_lane) ? src : lane);
    if (!live[u]) continue;
    float x[8];
    unpack8<T>(xw[u], x);
    if (rot_lane) rotate8<T, CS>(p, x, pw, cs[u], e0 < half);
    const i32x4 out = pack8<T>(x);
    __builtin_nontemporal_store(out, reinterpret_cast<i32x4 *>(row[u] + e0));
    if (!is_k[u]) continue;
    const int64_t sl = slot[u];
    const int64_t page = sl >> 4;
    if (sl < 0 || page >= p.num_pages) continue;  // not stored
    const int h = head[u];
    const int64_t ko = page * p.kc_sp + (sl & 15) * p.kc_st + (int64_t)h * p.kc_sh + e0;
    const int64_t vo = page * p.vc_sp + (sl & 15) * p.vc_st + (int64_t)h * p.vc_sh + e0;
    if constexpr (CT == 0) {
      float kv[8], v[8];
      unpack8<T>(out, kv);  // quantise the stored model-dtype values
      unpack8<T>(vw[u], v);
      const float ks = ksc[u], vs = vsc[u];
      const float k_lo[4] = {kv[0], kv[1], kv[2], kv[3]}, k_hi[4] = {kv[4], kv[5], kv[6], kv[7]};
      const float v_lo[4] = {v[0], v[1], v[2], v[3]}, v_hi[4] = {v[4], v[5], v[6], v[7]};
      __builtin_nontemporal_store(i32x2{quant4(k_lo, ks), quant4(k_hi, ks)}, reinterpret_cast<i32x2 *>(reinterpret_cast<uint8_t *>(p.kc) + ko));
      __builtin_nontemporal_store(i32x2{quant4(v_lo, vs), quant4(v_hi, vs)}, reinterpret_cast<i32x2 *>(reinterpret_cast<uint8_t *>(p.vc) + vo));
    } else {
      *reinterpret_cast<i32x4 *>(reinterpret_cast<T *>(p.kc) + ko) = out;
      *reinterpret_cast<i32x4 *>(reinterpret_cast<T *>(p.vc) + vo) = vw[u];
    }
  }
}

template <typename T, int CT>
__global__ __launch_bounds__(256) void kv_rope_write(Params p) {
  const int t = blockIdx.x;
  const int h = blockIdx.y * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int e0 = 4 * lane;
  if (e0 >= p.d) return;
  const int64_t position = p.pos[t];
  float x[4];
  if (p.q && h < p.hq) {
    T *row = reinterpret_cast<T *>(p.q) + (int64_t)t * p.q_st + (int64_t)h * p.q_sh;
    rope4<T>(p, row, position, e0, x);
    *reinterpret_cast<i32x2 *>(row + e0) = pack4<T>(x);
  }
  if (h >= p.hkv) return;
  T *krow = reinterpret_cast<T *>(p.k) + (int64_t)t * p.k_st + (int64_t)h * p.k_sh;
  rope4<T>(p, krow, position, e0, x);
  const i32x2 kw = pack4<T>(x);
  *reinterpret_cast<i32x2 *>(krow + e0) = kw;
  const int64_t slot = p.slots[t];
  if (slot < 0) return;
  const int64_t page = slot >> 4;
  const int64_t r = slot & 15;
  if (page >= p.num_pages) return;  // outside the cache: nothing to write
  float v[4];
  load4(reinterpret_cast<const T *>(p.v) + (int64_t)t * p.v_st + (int64_t)h * p.v_sh + e0, v);
  const int64_t ko = page * p.kc_sp + r * p.kc_st + (int64_t)h * p.kc_sh + e0;
  const int64_t vo = page * p.vc_sp + r * p.vc_st + (int64_t)h * p.vc_sh + e0;
  if constexpr (CT == 0) {
    float kv[4];
    unpack4<T>(kw, kv);  // quantise the stored model-dtype values
    const float ks = p.k_scale_ph ? p.k_scale_ph[h] : p.k_scale;
    const float vs = p.v_scale_ph ? p.v_scale_ph[h] : p.v_scale;
    *reinterpret_cast<int *>(reinterpret_cast<uint8_t *>(p.kc) + ko) = quant4(kv, ks);
    *reinterpret_cast<int *>(reinterpret_cast<uint8_t *>(p.vc) + vo) = quant4(v, vs);
  } else {
    *reinterpret_cast<i32x2 *>(reinterpret_cast<T *>(p.kc) + ko) = kw;
    *reinterpret_cast<i32x2 *>(reinterpret_cast<T *>(p.vc) + vo) = pack4<T>(v);
  }
}

// ---------------------------------------------------------------------------
// fp8 cache scales
// ---------------------------------------------------------------------------
// max(amax / 448, 1e-12).  Correctly rounded division is monotone, so the
// maximum of the workgroups' scales is the scale of the overall maximum: the
// workgroups combine scales, and no pass over the maxima follows.
__device__ __forceinline__ float scale_of(float amax) { return fmaxf(__fdiv_rn(amax, kFp8Max), 1e-12f); }

constexpr int kScaleThreads = 1024;
constexpr int kScaleMaxGroups = kScaleThreads / 4;  // lane groups of a workgroup at the smallest head_dim (32)
// Rows per lane in flight (fp32 tables take twice the registers).
constexpr int scale_rows(int cs) { return cs == 2 ? 2 : 4; }

// Every scale to its lower bound, ahead of the workgroups' atomic maxima.
__global__ void kv_scales_init(float *k_scales, float *v_scales, int hkv) {
  const int h = blockIdx.x * blockDim.x + threadIdx.x;
  if (h < hkv) k_scales[h] = v_scales[h] = 1e-12f;
}

// One workgroup's maxima -> the scales.  A positive float orders as its bits.
// single: the only workgroup of the call, which stores (no kv_scales_init ran).
// Consecutive lanes hold consecutive heads, so up to 64 heads leave in one instruction
// over consecutive words: device-scope atomics on one line are served one request at a time.
__device__ __forceinline__ void publish_scale(float *out, int h, float amax, bool single) {
  const float s = scale_of(amax);
  if (single) out[h] = s;
  else atomicMax(reinterpret_cast<unsigned int *>(out) + h, __builtin_bit_cast(unsigned int, s));
}

// The fast path: amax of the stored K (rotated, dtype-rounded) and V of a chunk
// of tokens, every head.  HBM-bound: K and V are read once, in whole rows (a
// lane owns eight contiguous dims, D/8 lanes a row, scale_rows rows of K and
// V in flight per lane), and every lane group keeps one head, so the maxima stay
// in registers until the workgroup's LDS fold.  blockIdx.y: block of hb heads.
// 16K tokens of 4 KV heads at head_dim 128 (38 MB): 12.3 us, 3.1 TB/s, where one
// workgroup per (head, K or V) took 3158 us; 13.0 us per call with the initialising
// launch.  256 workgroups of 16 waves, the whole chunk in flight at once.  Per call
// with an earlier order of its loads: 15.1 us, 13.2 without the atomics, 512
// workgroups of 8 waves 17.0, 1024 of 4 22.3 (more atomics on one line).
template <typename T, int CS>
__global__ __launch_bounds__(kScaleThreads) void kv_amax8(Params p, float *k_out, float *v_out, int hb, int chunk,
                                                         int per_head, int single) {
#pragma clang fp contract(off)
  constexpr int kRows = scale_rows(CS);
  __shared__ float s_max[2][kScaleMaxGroups];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int lpr = p.d >> 3;     // lanes per row
  const int rpw = 64 / lpr;     // rows per wave and pass
  const int g = lane / lpr;
  const int l = lane - g * lpr;
  const int e0 = 8 * l;
  const int half = p.rot >> 1;
  const bool rot_lane = e0 < p.rot;
  const int tpp = (kScaleThreads / 64) * rpw / hb;  // tokens per pass
  const int group = wave * rpw + g;
  const int off = group / hb;  // the group's token of a pass
  const int head = blockIdx.y * hb + (group - off * hb);
  const bool used = g < rpw && off < tpp && head < p.hkv;
  const int64_t t_end = min((int64_t)p.tokens, ((int64_t)blockIdx.x + 1) * chunk);
  const int64_t held = min(head, p.hkv - 1);
  const T *kbase = reinterpret_cast<const T *>(p.k) + held * p.k_sh + e0;
  const T *vbase = reinterpret_cast<const T *>(p.v) + held * p.v_sh + e0;
  // the neox partner's words, from the lane half/8 away in the same row
  const int src = (p.neox && rot_lane) ? g * lpr + (e0 < half ? l + (half >> 3) : l - (half >> 3)) : lane;
  float mk = 0.0f, mv = 0.0f;
  for (int64_t t0 = (int64_t)blockIdx.x * chunk; t0 < t_end; t0 += kRows * tpp) {  // uniform: every lane shuffles
    i32x4 kw[kRows], vw[kRows];
    int64_t pos[kRows], slot[kRows];
    // Every load of the pass without a branch (past the chunk: its last token again),
    // positions and slots first: a slot compared where it is loaded, in a branch,
    // waits there for all loads so far (16K tokens of 4 heads: 13.5 -> 12.3 us).
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
      const int64_t t = min(t0 + (int64_t)u * tpp + off, t_end - 1);
      pos[u] = p.pos[t];
      slot[u] = p.slots[t];
    }
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
      const int64_t t = min(t0 + (int64_t)u * tpp + off, t_end - 1);
      kw[u] = *reinterpret_cast<const i32x4 *>(kbase + t * p.k_st);
      vw[u] = *reinterpret_cast<const i32x4 *>(vbase + t * p.v_st);
    }
    bool live[kRows];
#pragma unroll
    for (int u = 0; u < kRows; ++u)
      live[u] = used && t0 + (int64_t)u * tpp + off < t_end && slot[u] >= 0 &&
                (slot[u] >> 4) < p.num_pages;  // else not stored
    CosSin<CS> cs[kRows];
#pragma unroll
    for (int u = 0; u < kRows; ++u)
      if (live[u] && rot_lane) load_row_cs<CS>(p, pos[u], e0, half, cs[u]);
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
      i32x4 pw;
#pragma unroll
      for (int i = 0; i < 4; ++i) pw[i] = __shfl(kw[u][i], src);
      if (!live[u]) continue;
      float x[8];
      unpack8<T>(kw[u], x);
      if (rot_lane) rotate8<T, CS>(p, x, pw, cs[u], e0 < half);
      unpack8<T>(pack8<T>(x), x);  // the stored model-dtype values
#pragma unroll
      for (int i = 0; i < 8; ++i) mk = fmaxf(mk, fabsf(x[i]));
      unpack8<T>(vw[u], x);
#pragma unroll
      for (int i = 0; i < 8; ++i) mv = fmaxf(mv, fabsf(x[i]));
    }
  }
  // the row's lanes
  float rk = mk, rv = mv;
  if ((lpr & (lpr - 1)) == 0) {
    for (int o = 1; o < lpr; o <<= 1) {
      rk = fmaxf(rk, __shfl_xor(rk, o));
      rv = fmaxf(rv, __shfl_xor(rv, o));
    }
  } else {  // head_dim 96: 12 lanes
    for (int i = 0; i < lpr; ++i) {
      rk = fmaxf(rk, __shfl(mk, min(g * lpr + i, 63)));
      rv = fmaxf(rv, __shfl(mv, min(g * lpr + i, 63)));
    }
  }
  if (l == 0 && g < rpw) {
    s_max[0][group] = used ? rk : 0.0f;
    s_max[1][group] = used ? rv : 0.0f;
  }
  __syncthreads();
  const int groups = (kScaleThreads / 64) * rpw;
  if (per_head) {
    const int i = threadIdx.x;  // head i of the block
    if (i >= hb || blockIdx.y * hb + i >= p.hkv) return;
    float k = 0.0f, v = 0.0f;
    for (int o = 0; o < tpp; ++o) {
      k = fmaxf(k, s_max[0][o * hb + i]);
      v = fmaxf(v, s_max[1][o * hb + i]);
    }
    publish_scale(k_out, blockIdx.y * hb + i, k, single);
    publish_scale(v_out, blockIdx.y * hb + i, v, single);
  } else {
    float k = 0.0f, v = 0.0f;  // the maximum over heads, in every entry
    for (int o = 0; o < groups; ++o) {
      k = fmaxf(k, s_max[0][o]);
      v = fmaxf(v, s_max[1][o]);
    }
    for (int h = threadIdx.x; h < p.hkv; h += kScaleThreads) {
      publish_scale(k_out, h, k, single);
      publish_scale(v_out, h, v, single);
    }
  }
}

// The general path (any layout the checks accept): workgroup (h, K or V, chunk
// of tokens), 16 waves over the chunk's tokens, four dims per lane.
template <typename T>
__global__ __launch_bounds__(1024) void kv_amax(Params p, float *k_out, float *v_out, int chunk, int per_head) {
  __shared__ float s_red[16];
  const int h = blockIdx.x;
  const bool is_k = blockIdx.y == 0;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int e0 = 4 * lane;
  const int64_t t_end = min((int64_t)p.tokens, ((int64_t)blockIdx.z + 1) * chunk);
  float m = 0.0f;
  if (e0 < p.d) {
    for (int64_t t = (int64_t)blockIdx.z * chunk + wave; t < t_end; t += 16) {
      const int64_t slot = p.slots[t];
      if (slot < 0 || (slot >> 4) >= p.num_pages) continue;  // not stored
      float x[4];
      if (is_k) {
        const T *row = reinterpret_cast<const T *>(p.k) + t * p.k_st + (int64_t)h * p.k_sh;
        rope4<T>(p, row, p.pos[t], e0, x);
        const i32x2 w = pack4<T>(x);
        unpack4<T>(w, x);
      } else {
        load4(reinterpret_cast<const T *>(p.v) + t * p.v_st + (int64_t)h * p.v_sh + e0, x);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) m = fmaxf(m, fabsf(x[i]));
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  if (lane == 0) s_red[wave] = m;
  __syncthreads();
  float r = 0.0f;
  for (int w = 0; w < 16; ++w) r = fmaxf(r, s_red[w]);
  float *out = is_k ? k_out : v_out;
  if (per_head) {
    if (threadIdx.x == 0) publish_scale(out, h, r, false);
  } else {
    for (int i = threadIdx.x; i < p.hkv; i += 1024) publish_scale(out, i, r, false);
  }
}

}  // namespace l20kv

namespace {

using l20pd_host::set_error;

int32_t check(const l20_pd_kv_write_args *a) {
  if (!a) return set_error(L20_PD_EINVAL, "null argument block");
  if (a->dtype != L20_PD_BF16 && a->dtype != L20_PD_FP16)
    return set_error(L20_PD_EINVAL, "query, key and value must be bf16 or fp16");
  if (a->cs_dtype != L20_PD_BF16 && a->cs_dtype != L20_PD_FP16 && a->cs_dtype != L20_PD_FP32)
    return set_error(L20_PD_EINVAL, "cos_sin_cache must be bf16, fp16 or fp32");
  const bool fp8 = a->cache_dtype == L20_PD_KV_FP8_E4M3;
  if (!fp8 && a->cache_dtype != L20_PD_KV_FP16 && a->cache_dtype != L20_PD_KV_BF16)
    return set_error(L20_PD_EINVAL, "unknown K/V cache dtype");
  if (!fp8 && (a->cache_dtype == L20_PD_KV_BF16) != (a->dtype == L20_PD_BF16))
    return set_error(L20_PD_EINVAL, "a 16-bit cache must have the model dtype");
  if (a->head_dim <= 0 || a->head_dim > 256 || a->head_dim % 4)
    return set_error(L20_PD_EINVAL, "head_dim must be a multiple of 4 up to 256");
  if (a->rotary_dim < 0 || a->rotary_dim > a->head_dim || a->rotary_dim % 8)
    return set_error(L20_PD_EINVAL, "invalid cos_sin_cache rotary dimension");
  if (a->num_tokens < 0 || a->num_kv_heads <= 0 || (a->query && a->num_q_heads <= 0))
    return set_error(L20_PD_EINVAL, "token and head counts must be positive");
  if ((int64_t)std::max(a->num_q_heads, a->num_kv_heads) > 65535 * 4)
    return set_error(L20_PD_EINVAL, "too many heads");
  if (a->num_tokens == 0) return L20_PD_OK;
  if (!a->key || !a->value || !a->positions || !a->slot_mapping || !a->key_cache || !a->value_cache ||
      (a->rotary_dim > 0 && !a->cos_sin_cache))
    return set_error(L20_PD_EINVAL, "null tensor pointer");
  // 8-byte row chunks of the 16-bit tensors, 4-byte (fp8) or 8-byte (16-bit) cache chunks
  const uint64_t qkv = (uint64_t)(uintptr_t)a->key | (uint64_t)(uintptr_t)a->value |
                       (uint64_t)(a->k_stride_token * 2) | (uint64_t)(a->k_stride_head * 2) |
                       (uint64_t)(a->v_stride_token * 2) | (uint64_t)(a->v_stride_head * 2) |
                       (a->query ? ((uint64_t)(uintptr_t)a->query | (uint64_t)(a->q_stride_token * 2) |
                                    (uint64_t)(a->q_stride_head * 2))
                                 : 0);
  if (qkv % 8) return set_error(L20_PD_EINVAL, "query/key/value pointers and strides must be 8-byte aligned");
  const int64_t es = fp8 ? 1 : 2;
  const uint64_t cb = (uint64_t)(uintptr_t)a->key_cache | (uint64_t)(uintptr_t)a->value_cache |
                      (uint64_t)(a->kc_stride_page * es) | (uint64_t)(a->kc_stride_token * es) |
                      (uint64_t)(a->kc_stride_head * es) | (uint64_t)(a->vc_stride_page * es) |
                      (uint64_t)(a->vc_stride_token * es) | (uint64_t)(a->vc_stride_head * es);
  if (cb % (uint64_t)(4 * es)) return set_error(L20_PD_EINVAL, "cache pointers and strides must be aligned to 4 elements");
  if (a->num_pages <= 0) return set_error(L20_PD_EINVAL, "K/V cache has no pages");
  return L20_PD_OK;
}

l20kv::Params params(const l20_pd_kv_write_args &a) {
  l20kv::Params p{};
  p.q = a.query;
  p.q_st = a.q_stride_token;
  p.q_sh = a.q_stride_head;
  p.hq = a.query ? a.num_q_heads : 0;
  p.k = a.key;
  p.k_st = a.k_stride_token;
  p.k_sh = a.k_stride_head;
  p.v = a.value;
  p.v_st = a.v_stride_token;
  p.v_sh = a.v_stride_head;
  p.pos = a.positions;
  p.cs = a.cos_sin_cache;
  p.cs_sp = a.cs_stride_position;
  p.cs_dtype = a.cs_dtype == L20_PD_FP32 ? 2 : (a.cs_dtype == L20_PD_FP16 ? 1 : 0);
  p.rot = a.rotary_dim;
  p.neox = a.is_neox != 0;
  p.slots = a.slot_mapping;
  p.kc = a.key_cache;
  p.kc_sp = a.kc_stride_page;
  p.kc_st = a.kc_stride_token;
  p.kc_sh = a.kc_stride_head;
  p.vc = a.value_cache;
  p.vc_sp = a.vc_stride_page;
  p.vc_st = a.vc_stride_token;
  p.vc_sh = a.vc_stride_head;
  p.num_pages = a.num_pages;
  p.k_scale = a.k_scale;
  p.v_scale = a.v_scale;
  p.k_scale_ph = a.k_scale_per_head;
  p.v_scale_ph = a.v_scale_per_head;
  p.tokens = a.num_tokens;
  p.hkv = a.num_kv_heads;
  p.d = a.head_dim;
  return p;
}

// The fast path's layout requirements (16-byte rows and cache chunks, lane-aligned neox halves).
bool fast_path_ok(const l20_pd_kv_write_args &a) {
  if (a.head_dim % 8 || (a.is_neox && a.rotary_dim % 16)) return false;
  const uint64_t qkv = (uint64_t)(uintptr_t)a.key | (uint64_t)(uintptr_t)a.value |
                       (uint64_t)(a.k_stride_token * 2) | (uint64_t)(a.k_stride_head * 2) |
                       (uint64_t)(a.v_stride_token * 2) | (uint64_t)(a.v_stride_head * 2) |
                       (a.query ? ((uint64_t)(uintptr_t)a.query | (uint64_t)(a.q_stride_token * 2) |
                                   (uint64_t)(a.q_stride_head * 2))
                                : 0);
  if (qkv % 16) return false;
  const bool fp8 = a.cache_dtype == L20_PD_KV_FP8_E4M3;
  const int64_t es = fp8 ? 1 : 2;
  const uint64_t cb = (uint64_t)(uintptr_t)a.key_cache | (uint64_t)(uintptr_t)a.value_cache |
                      (uint64_t)(a.kc_stride_page * es) | (uint64_t)(a.kc_stride_token * es) |
                      (uint64_t)(a.kc_stride_head * es) | (uint64_t)(a.vc_stride_page * es) |
                      (uint64_t)(a.vc_stride_token * es) | (uint64_t)(a.vc_stride_head * es);
  if (cb % (uint64_t)(8 * es)) return false;
  if (a.rotary_dim > 0) {
    const int64_t cs_es = a.cs_dtype == L20_PD_FP32 ? 4 : 2;
    const uint64_t cs = (uint64_t)(uintptr_t)a.cos_sin_cache | (uint64_t)(a.cs_stride_position * cs_es) |
                        (uint64_t)(a.rotary_dim / 2 * cs_es);
    // neox: 8 values per 16-byte load; interleaved: 4 values (8 bytes, or 16 for fp32)
    if (cs % (uint64_t)(a.is_neox ? 16 : 4 * cs_es)) return false;
  }
  return true;
}

template <typename T, int CT, int ROWS, bool POS_FIRST>
void launch_fast_rows(const l20kv::Params &p, int cs_dtype, uint32_t rows_q, uint32_t rows_all, hipStream_t s) {
  const int64_t rows_per_wg = (int64_t)4 * (64 / (p.d / 8)) * ROWS;
  const dim3 grid((unsigned)((rows_all + rows_per_wg - 1) / rows_per_wg));
  if constexpr (!POS_FIRST)  // never with fp32 tables (rows_per_lane)
    if (cs_dtype == 2) {
      hipLaunchKernelGGL((l20kv::kv_rope_write8<T, CT, 2, ROWS, false>), grid, dim3(256), 0, s, p, rows_q, rows_all);
      return;
    }
  if (cs_dtype == 1)
    hipLaunchKernelGGL((l20kv::kv_rope_write8<T, CT, 1, ROWS, POS_FIRST>), grid, dim3(256), 0, s, p, rows_q, rows_all);
  else
    hipLaunchKernelGGL((l20kv::kv_rope_write8<T, CT, 0, ROWS, POS_FIRST>), grid, dim3(256), 0, s, p, rows_q, rows_all);
}

// Rows per lane, by `one`, the workgroups of one row per lane.  A call is a chain of
// dependent loads, so what decides is whether its workgroups are on the chip at once:
// 8 a CU of one row per lane (2048), 6 of two (1536, the rows of 3072 of one; 5 with
// fp8 caches and fp32 tables, whose words take twice the registers).  Up to 2048 one
// row, up to 3072 two, beyond them one again (the shorter last round), until the
// stream is long enough for the loads in flight to count: 20480 with fp8 caches, whose
// quantiser needs the waves, 4096 with 16-bit ones, never with fp32 tables.  us per
// call with one and two rows, in a graph, by `one`, 28 + 4 heads of 128 with an fp8 and
// a bf16 cache, 16-bit tables: 1024 4.2, 5.0 and 3.8, 4.2; 1900 5.2, 6.0 and 5.5, 5.6;
// 2100 7.0, 6.5 and 6.5, 6.2; 2800 7.9, 7.3 and 7.5, 7.3; 3300 8.5, 10.1 and 8.4, 9.5;
// and, two with the positions first, 4050 10.4, 11.0 and 10.2, 10.0; 9000 20.9, 21.3 and
// 21.0, 19.9; 16000 33.6, 34.6 and 34.0, 33.1; 20000 41.0, 41.2 and 41.2, 40.4; 25500
// 51.3, 50.5 and 51.0, 51.1; 32768 64.6, 63.1 and 64.0, 62.1.  32 + 8 heads, fp32
// tables: 2100 7.5, 7.8 and 7.0, 7.4; 2500 9.2, 8.4 and 8.5, 8.2; 3000 9.9, 10.9 and
// 9.6, 9.1; 3200 10.4, 11.4 and 9.8, 10.1; 9000 21.3, 24.2 and 22.0, 24.3; 16000 34.6,
// 38.0 and 34.7, 38.0; 32768 66.0, 73.4 and 65.2, 68.5.
int rows_per_lane(int64_t one, bool fp8_cache, bool fp32_table) {
  if (one <= 2048) return 1;
  if (one <= (fp8_cache && fp32_table ? 2560 : 3072)) return 2;
  return fp32_table || one <= (fp8_cache ? 20480 : 4096) ? 1 : 2;
}
template <typename T, int CT>
void launch_fast(const l20kv::Params &p, int cs_dtype, uint32_t rows_q, uint32_t rows_all, hipStream_t s) {
  const int64_t one = ((int64_t)rows_all + 4 * (64 / (p.d / 8)) - 1) / (4 * (64 / (p.d / 8)));
  if (rows_per_lane(one, CT == 0, cs_dtype == 2) == 1)
    launch_fast_rows<T, CT, 1, false>(p, cs_dtype, rows_q, rows_all, s);
  else if (one <= 3072)
    launch_fast_rows<T, CT, 2, false>(p, cs_dtype, rows_q, rows_all, s);
  else
    launch_fast_rows<T, CT, 2, true>(p, cs_dtype, rows_q, rows_all, s);
}

template <typename T>
void launch_amax8(const l20kv::Params &p, dim3 grid, float *k_scales, float *v_scales, int hb, int chunk, int per_head,
                  bool single, hipStream_t s) {
  const dim3 block(l20kv::kScaleThreads);
  if (p.cs_dtype == 2)
    hipLaunchKernelGGL((l20kv::kv_amax8<T, 2>), grid, block, 0, s, p, k_scales, v_scales, hb, chunk, per_head, single);
  else if (p.cs_dtype == 1)
    hipLaunchKernelGGL((l20kv::kv_amax8<T, 1>), grid, block, 0, s, p, k_scales, v_scales, hb, chunk, per_head, single);
  else
    hipLaunchKernelGGL((l20kv::kv_amax8<T, 0>), grid, block, 0, s, p, k_scales, v_scales, hb, chunk, per_head, single);
}

int32_t launched() {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    char msg[256];
    snprintf(msg, sizeof(msg), "HIP launch failed: %s", hipGetErrorString(e));
    return set_error(L20_PD_ELAUNCH, msg);
  }
  return L20_PD_OK;
}

}  // namespace

extern "C" {

int32_t l20_pd_kv_write_check(const l20_pd_kv_write_args *args) {
  l20pd_host::clear_error();
  return check(args);
}

int32_t l20_pd_rope_and_cache(const l20_pd_kv_write_args *a, void *stream) {
  l20pd_host::clear_error();
  const int32_t rc = check(a);
  if (rc != L20_PD_OK || a->num_tokens == 0) return rc;
  const l20kv::Params p = params(*a);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const bool bf = a->dtype == L20_PD_BF16;
  // (row numbers in 32 bits, with room for the last workgroup's)
  if (fast_path_ok(*a) && (int64_t)a->num_tokens * ((int64_t)p.hq + p.hkv) < ((int64_t)1 << 31)) {
    const uint32_t rows_q = (uint32_t)((int64_t)a->num_tokens * p.hq);
    const uint32_t rows_all = (uint32_t)((int64_t)a->num_tokens * ((int64_t)p.hq + p.hkv));
    const bool fp8 = a->cache_dtype == L20_PD_KV_FP8_E4M3;
    if (bf) {
      if (fp8) launch_fast<__bf16, 0>(p, p.cs_dtype, rows_q, rows_all, s);
      else launch_fast<__bf16, 1>(p, p.cs_dtype, rows_q, rows_all, s);
    } else {
      if (fp8) launch_fast<_Float16, 0>(p, p.cs_dtype, rows_q, rows_all, s);
      else launch_fast<_Float16, 1>(p, p.cs_dtype, rows_q, rows_all, s);
    }
    return launched();
  }
  const int heads = std::max(p.hq, p.hkv);
  const dim3 grid((unsigned)a->num_tokens, (unsigned)((heads + 3) / 4));
  if (a->cache_dtype == L20_PD_KV_FP8_E4M3) {
    if (bf)
      hipLaunchKernelGGL((l20kv::kv_rope_write<__bf16, 0>), grid, dim3(256), 0, s, p);
    else
      hipLaunchKernelGGL((l20kv::kv_rope_write<_Float16, 0>), grid, dim3(256), 0, s, p);
  } else {
    if (bf)
      hipLaunchKernelGGL((l20kv::kv_rope_write<__bf16, 1>), grid, dim3(256), 0, s, p);
    else
      hipLaunchKernelGGL((l20kv::kv_rope_write<_Float16, 1>), grid, dim3(256), 0, s, p);
  }
  return launched();
}

int32_t l20_pd_kv_fp8_scales(const l20_pd_kv_write_args *a, float *k_scales, float *v_scales, int32_t per_head,
                             void *stream) {
  l20pd_host::clear_error();
  const int32_t rc = check(a);
  if (rc != L20_PD_OK) return rc;
  if (!k_scales || !v_scales) return set_error(L20_PD_EINVAL, "null scale output");
  l20_pd_kv_write_args b = *a;
  b.query = nullptr;  // not read: its layout does not decide the path
  const l20kv::Params p = params(b);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const bool bf = a->dtype == L20_PD_BF16;
  const int tokens = std::max(1, p.tokens);
  // At least 32 dims (the fold's LDS rows): smaller heads take the general path.
  const bool fast = a->num_tokens > 0 && p.d >= 32 && fast_path_ok(b);
  // Fast path: one pass of the grid where it can be (16K tokens, 4 KV heads:
  // 256 workgroups of 64 tokens), at most 256 workgroups (an MI355X's CUs) for each
  // block of hb heads, since the atomics on one line of scales are served one at a
  // time (~11 ns each).
  const int groups = (l20kv::kScaleThreads / 64) * (fast ? 64 / (p.d / 8) : 1);
  const int hb = std::min(p.hkv, groups);
  const int step = l20kv::scale_rows(p.cs_dtype) * (groups / hb);  // tokens per workgroup and loop pass
  int64_t chunk, blocks;
  if (fast) {
    blocks = std::min<int64_t>(256, ((int64_t)tokens + step - 1) / step);
    chunk = (((int64_t)tokens + blocks - 1) / blocks + step - 1) / step * step;
  } else {
    // 16 waves of at least 4 tokens each; (K, V) x heads x chunks workgroups about the CUs
    blocks = std::max<int64_t>(1, std::min<int64_t>(((int64_t)tokens + 63) / 64, 128 / std::min(p.hkv, 128)));
    chunk = ((int64_t)tokens + blocks - 1) / blocks;
  }
  blocks = ((int64_t)tokens + chunk - 1) / chunk;
  const dim3 grid = fast ? dim3((unsigned)blocks, (unsigned)((p.hkv + hb - 1) / hb))
                         : dim3((unsigned)p.hkv, 2, (unsigned)blocks);
  const bool single = fast && grid.x == 1 && grid.y == 1;
  if (!single) {
    hipLaunchKernelGGL(l20kv::kv_scales_init, dim3((unsigned)((p.hkv + 255) / 256)), dim3(256), 0, s, k_scales,
                       v_scales, p.hkv);
    const int32_t r = launched();
    if (r != L20_PD_OK) return r;
  }
  if (fast) {
    if (bf) launch_amax8<__bf16>(p, grid, k_scales, v_scales, hb, (int)chunk, per_head, single, s);
    else launch_amax8<_Float16>(p, grid, k_scales, v_scales, hb, (int)chunk, per_head, single, s);
  } else if (bf) {
    hipLaunchKernelGGL((l20kv::kv_amax<__bf16>), grid, dim3(1024), 0, s, p, k_scales, v_scales, (int)chunk, per_head);
  } else {
    hipLaunchKernelGGL((l20kv::kv_amax<_Float16>), grid, dim3(1024), 0, s, p, k_scales, v_scales, (int)chunk, per_head);
  }
  return launched();
}

}  // extern "C"
