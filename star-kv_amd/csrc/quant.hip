// Latent-cache writer on gfx950: quantise (or copy) new latent rows in place
// into a preallocated cache.
//
// Replaces the per-step cache growth of the reference -- HF DynamicLayer.update
// (HF:cache_utils.py:127-146, a torch.cat of the whole cache per token, reached
// from model.py:411-419) -- and the quantise-on-write of the quantised module
// (LlamaLoRaAttention_headwise_quant.py:107-127, whose quantize_r_split_int8_
// int4_packed the reference does not ship).  A "row" is one K latent vector
// (b, h, s) of rank r_h or one V latent vector (b, s) of rank Rv; one wave
// quantises one row:
//   int8 block:  s = fp16(amax / 127), q = clip(rint(x / s), -127, 127)
//   int4 block:  s = fp16(amax / 7),   n = clip(rint(x / s), -8, 7), nibble n + 8
//                (rank 2k in the low nibble of byte k)
//   group-64:    z = fp16(min), s = fp16((max - z) / 15), n = clip(rint((x - z) / s), 0, 15)
// with s = 1 when it would be 0, divisions correctly rounded and rint
// rounding half to even -- the rounding steps of the CPU oracle's quantisers.
// The cache is described by the same starkv_klatent / starkv_vlatent structs
// the attention entry points read.
#include "common.hpp"

namespace starkv {

__device__ inline float wave_max(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ inline float wave_min(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
  return v;
}

template <typename T>
__device__ inline float ldx(const T* p, int j) { return to_f32(p[j]); }

__device__ inline _Float16 fp16_scale(float amax, float qmax) {
  _Float16 s = (_Float16)__fdiv_rn(amax, qmax);
  return (float)s == 0.f ? (_Float16)1.0f : s;
}

// Quantise ranks [j0, j1) of the row at x (act dtype) as one symmetric block:
// int8 bytes into q8 (j - j0) or int4 nibbles into q4 ((j - j0) / 2); scale to *sp.
template <typename T>
__device__ void quant_block(const T* x, int j0, int j1, bool int8, uint8_t* q, uint16_t* sp, int lane) {
  float amax = 0.f;
  for (int j = j0 + lane; j < j1; j += 64) amax = fmaxf(amax, fabsf(ldx(x, j)));
  amax = wave_max(amax);
  const _Float16 s16 = fp16_scale(amax, int8 ? 127.f : 7.f);
  const float s = (float)s16;
  if (lane == 0) *sp = __builtin_bit_cast(uint16_t, s16);
  if (int8) {
    for (int j = j0 + lane; j < j1; j += 64) {
      const float n = fminf(fmaxf(rintf(__fdiv_rn(ldx(x, j), s)), -127.f), 127.f);
      q[j - j0] = (uint8_t)(int8_t)(int)n;
    }
  } else {
    for (int k = j0 + 2 * lane; k < j1; k += 128) {       // one byte = ranks k, k+1
      const float n0 = fminf(fmaxf(rintf(__fdiv_rn(ldx(x, k), s)), -8.f), 7.f);
      const float n1 = k + 1 < j1 ? fminf(fmaxf(rintf(__fdiv_rn(ldx(x, k + 1), s)), -8.f), 7.f) : 0.f;
      q[(k - j0) >> 1] = (uint8_t)(((int)n0 + 8) | (((int)n1 + 8) << 4));
    }
  }
}

// Group-64 asymmetric int4 of the row: nibbles into q, scale / zero of group g at sp[g] / zp[g].
// one group of 64 ranks (ranks g0 .. g0 + 63 of the row)
template <typename T>
__device__ void quant_g64(const T* x, int R, int g0, uint8_t* q, uint16_t* sp, uint16_t* zp, int lane) {
  {
    const int j = g0 + lane;
    const bool ok = j < R;
    const float v = ok ? ldx(x, j) : 0.f;
    const float lo = wave_min(ok ? v : INFINITY), hi = wave_max(ok ? v : -INFINITY);
    const _Float16 z16 = (_Float16)lo;
    const float z = (float)z16;
    _Float16 s16 = (_Float16)__fdiv_rn(hi - z, 15.f);
    if ((float)s16 == 0.f) s16 = (_Float16)1.0f;
    const float s = (float)s16;
    if (lane == 0) {
      sp[g0 / 64] = __builtin_bit_cast(uint16_t, s16);
      zp[g0 / 64] = __builtin_bit_cast(uint16_t, z16);
    }
    const int n = ok ? (int)fminf(fmaxf(rintf(__fdiv_rn(v - z, s)), 0.f), 15.f) : 0;
    const int n_odd = __shfl_xor(n, 1, 64);
    if (ok && !(lane & 1)) q[j >> 1] = (uint8_t)(n | (n_odd << 4));
  }
}

// one row per wave; 4 waves per workgroup (blk: the workgroup's index)
template <typename T>
__device__ inline void k_append_rows(const KAppendArgs& a, int64_t blk) {
  const int lane = threadIdx.x & 63;
  const int64_t row = blk * 4 + (threadIdx.x >> 6);
  if (row >= (int64_t)a.B * a.H * a.T) return;
  const int t = (int)(row % a.T), h = (int)((row / a.T) % a.H), b = (int)(row / ((int64_t)a.T * a.H));
  const int s = (a.pos0_dev ? *a.pos0_dev : a.pos0) + t, r = a.rank[h];
  if (s < 0 || s >= a.cap) {                        // only a run-time position can land here
    if (a.err != nullptr && lane == 0) *a.err = 1;
    return;
  }
  const T* x = (const T*)a.src + b * a.src_sb + a.src_off[h] + (int64_t)t * a.src_st;
  if (a.fmt == STARKV_FMT_DENSE) {
    T* d = (T*)a.data + b * a.stride_b + a.off[h] + (int64_t)s * a.pitch[h];
    for (int j = lane; j < r; j += 64) d[j] = x[j];
    return;
  }
  const int ra = min(r, a.split);
  uint8_t* qa = (uint8_t*)a.data + b * a.stride_b + a.off[h] + (int64_t)s * a.pitch[h];
  uint16_t* sa = (uint16_t*)a.scale + b * a.sc_sb + h * a.sc_sh + s;
  quant_block(x, 0, ra, a.a_int8, qa, sa, lane);
  if (r > a.split) {
    uint8_t* qb = (uint8_t*)a.data2 + b * a.stride2_b + a.off2[h] + (int64_t)s * a.pitch2[h];
    uint16_t* sb = (uint16_t*)a.scale2 + b * a.sc2_sb + h * a.sc2_sh + s;
    quant_block(x, a.split, r, false, qb, sb, lane);
  }
}

// one row per wave; group-64 int4: one (row, group) per wave
template <typename T>
__device__ inline void v_append_rows(const VAppendArgs& a, int64_t blk) {
  const int lane = threadIdx.x & 63;
  const int64_t wid = blk * 4 + (threadIdx.x >> 6);
  const int64_t row = wid / a.gw;
  const int grp = (int)(wid - row * a.gw);
  if (row >= (int64_t)a.B * a.T) return;
  const int t = (int)(row % a.T), b = (int)(row / a.T);
  const int s = (a.pos0_dev ? *a.pos0_dev : a.pos0) + t, R = a.R;
  if (s < 0 || s >= a.cap) {                        // only a run-time position can land here
    if (a.err != nullptr && lane == 0) *a.err = 1;
    return;
  }
  const T* x = (const T*)a.src + b * a.src_sb + (int64_t)t * a.src_st;
  if (a.vq == VQ_DENSE) {
    T* d = (T*)a.data + b * a.stride_b + (int64_t)s * a.stride_s;
    for (int j = lane; j < R; j += 64) d[j] = x[j];
    return;
  }
  uint8_t* q = (uint8_t*)a.data + b * a.stride_b + (int64_t)s * a.stride_s;
  uint16_t* sp = (uint16_t*)a.scale + b * a.sc_sb + (int64_t)s * a.sc_ss;
  if (a.vq == VQ_G64) {
    quant_g64(x, R, 64 * grp, q, sp, (uint16_t*)a.zero + b * a.sc_sb + (int64_t)s * a.sc_ss, lane);
    return;
  }
  quant_block(x, 0, min(R, a.split), a.a_int8, q, sp, lane);
  if (R > a.split) {
    uint8_t* q2 = (uint8_t*)a.data2 + b * a.stride2_b + (int64_t)s * a.stride2_s;
    uint16_t* s2 = (uint16_t*)a.scale2 + b * a.sc2_sb + (int64_t)s * a.sc2_ss;
    quant_block(x, a.split, R, false, q2, s2, lane);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_append_kernel(const KAppendArgs a) {
  k_append_rows<T>(a, blockIdx.x);
}
template <typename T>
__global__ __launch_bounds__(256) void v_append_kernel(const VAppendArgs a) {
  v_append_rows<T>(a, blockIdx.x);
}

// A decode step's three small writes in one launch: workgroups [0, nbk) write
// the K rows, [nbk, nbk + nbv) the V rows, the rest rotate the query rows
// (64 threads per row, as rope_apply_kernel).
template <typename T>
__global__ __launch_bounds__(256) void step_append_kernel(const StepAppendArgs a) {
  int64_t blk = blockIdx.x;
  if (blk < a.nbk) {
    k_append_rows<T>(a.k, blk);
    return;
  }
  blk -= a.nbk;
  if (blk < a.nbv) {
    v_append_rows<T>(a.v, blk);
    return;
  }
  blk -= a.nbv;
  rope_apply_row<T>(a.r, blk * 256 + threadIdx.x);
}

// ---------------------------------------------------------------------------
// Many rows at once (a prompt).  The row-per-wave kernels above read 2 bytes
// per lane and spend most lanes on the short K rows; these read and write
// whole 8-rank chunks.
//
// Bytes bound this work, and past them the divisions: 8 + 4 latent bytes per
// 4 stored ones leave ~16 VALU operations per element at the copy rate, which
// two correctly rounded divisions would take alone.  The codes need only the
// quotient's rounding to an integer, so a chunk multiplies by the correctly
// rounded reciprocal of its scale and corrects the product by its exact
// residual.  Symmetric blocks: x and s have at most 11 significant bits, so
// the quotient is a tie n + 1/2 exactly or lies 2^-19 away from it
// (relatively), and one correction, exact at ties, rounds as the division
// does.  Group-64: x - z has 24 bits; two corrections give the correctly
// rounded quotient itself (Markstein's theorem: a faithful quotient and a
// correctly rounded reciprocal).  A scale outside fp16's range divides.
// Measured at B8 T2048 (32 heads, ranks sum 1640, Rv 1640, int8 K / group-64
// V, 151 MB): 348 -> 55 us a call, 51 us on the GPU (3.0 TB/s).
// ---------------------------------------------------------------------------
template <typename T>
__device__ inline void chunk_f32(uint4 u, float (&f)[8]) {
  const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if constexpr (__is_same(T, _Float16)) {
      const kh2 h = __builtin_bit_cast(kh2, w[k]);
      f[2 * k] = (float)h[0];
      f[2 * k + 1] = (float)h[1];
    } else {
      f[2 * k] = __uint_as_float(w[k] << 16);
      f[2 * k + 1] = __uint_as_float(w[k] & 0xffff0000u);
    }
  }
}

// nv (1..8) 16-bit elements from element j0 of a row on, zero past them.  Any
// 2-byte alignment (unaligned vector loads); a tail reads the 8 elements that
// end with it, so nothing outside the row is touched.
__device__ inline uint4 load_chunk(const uint16_t* row, int j0, int nv) {
  uint4 u;
  if (nv == 8) {
    __builtin_memcpy(&u, row + j0, 16);
    return u;
  }
  if (j0 >= 8) {
    __builtin_memcpy(&u, row + j0 + nv - 8, 16);
    const int drop = 16 * (8 - nv);                     // bits of the elements before j0
    const uint64_t lo = (uint64_t)u.x | ((uint64_t)u.y << 32), hi = (uint64_t)u.z | ((uint64_t)u.w << 32);
    const uint64_t l = drop < 64 ? (lo >> drop) | (hi << (64 - drop)) : hi >> (drop - 64);
    const uint64_t h = drop < 64 ? hi >> drop : 0;
    return make_uint4((uint32_t)l, (uint32_t)(l >> 32), (uint32_t)h, (uint32_t)(h >> 32));
  }
  uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (e < nv) w[e >> 1] |= (uint32_t)row[j0 + e] << (16 * (e & 1));
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// the codes' integers ride in the low bits of y + 1.5 * 2^23 (+ a bias), the
// addition rounding half to even as rint does
constexpr float RINT_MAGIC = 12582912.f;
__device__ inline uint32_t rint_bits(float y, float bias) { return __float_as_uint(y + (RINT_MAGIC + bias)); }

// eight nibbles (codes + bias in 0..15) of the quotients y, already clamped
__device__ inline uint32_t pack_nibbles(const float (&y)[8], float bias) {
  uint32_t w = 0;
#pragma unroll
  for (int e = 0; e < 8; ++e) w |= (rint_bits(y[e], bias) & 15u) << (4 * e);
  return w;
}

// n bytes (1..8) of w to q, any alignment
__device__ inline void store_bytes(uint8_t* q, uint64_t w, int n) {
  if (n == 8) {
    __builtin_memcpy(q, &w, 8);
  } else if (n == 4) {
    const uint32_t v = (uint32_t)w;
    __builtin_memcpy(q, &v, 4);
  } else {
    for (int i = 0; i < n; ++i) q[i] = (uint8_t)(w >> (8 * i));
  }
}

struct BlockPlan {
  int nc, pp, nb;                       // chunks of a position's heads, positions per pass, blocks per batch
  int ns;                               // scales per head (1, or 2 with a lower block)
  uint16_t cstart[K_MAX_KV];            // first chunk of head h (0xffff past the last head)
};

// All heads of a run of positions per workgroup, so the packed source rows
// ([B, T, sum of ranks]) are read as they lie: thread -> (position, 8-rank
// chunk) of one pass, KC chunks per thread where a position has more than 256,
// 8 / KC passes held in registers while the blocks' maxima meet in LDS.
template <typename T, int KC, bool DENSE>
__global__ __launch_bounds__(256) void append_block_kernel(const KAppendArgs a, const BlockPlan p) {
  constexpr int U = 8 / KC;
  extern __shared__ uint32_t sm[];
  const int tid = threadIdx.x;
  const int b = blockIdx.x / p.nb, t0 = (blockIdx.x - b * p.nb) * (p.pp * U);
  const int P = p.pp * U;
  const int nslot = a.H * p.ns * P;
  float* const scale = (float*)sm;                       // [head][block][position]: maxima, then scales
  float* const recip = scale + nslot;
  const int pos = a.pos0_dev ? *a.pos0_dev : a.pos0;
  const int pp = KC == 1 ? tid / p.nc : 0;
  int head[KC], j0[KC], nv[KC];
  uint4 x[KC][U];
#pragma unroll
  for (int k = 0; k < KC; ++k) {
    const int c = (KC == 1 ? tid - pp * p.nc : tid) + 256 * k;
    int h = -1;
#pragma unroll
    for (int i = 0; i < K_MAX_KV; ++i) h += c >= p.cstart[i];
    head[k] = h;
    j0[k] = 8 * (c - p.cstart[h]);
    nv[k] = c < p.nc && pp < p.pp ? min(8, a.rank[h] - j0[k]) : 0;
    const uint16_t* src = (const uint16_t*)a.src + b * a.src_sb + a.src_off[h];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (nv[k] > 0) x[k][u] = load_chunk(src + (int64_t)min(t0 + u * p.pp + pp, a.T - 1) * a.src_st, j0[k], nv[k]);
  }
  if (a.err != nullptr)
    for (int i = t0 + tid; i < min(t0 + P, a.T); i += 256)
      if (pos + i < 0 || pos + i >= a.cap) *a.err = 1;
  if constexpr (DENSE) {
#pragma unroll
    for (int k = 0; k < KC; ++k)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int t = t0 + u * p.pp + pp, s = pos + t;
        if (nv[k] <= 0 || t >= a.T || s < 0 || s >= a.cap) continue;
        uint16_t* d = (uint16_t*)a.data + b * a.stride_b + a.off[head[k]] + (int64_t)s * a.pitch[head[k]] + j0[k];
        if (nv[k] == 8) {
          __builtin_memcpy(d, &x[k][u], 16);
        } else {
          const uint32_t w[4] = {x[k][u].x, x[k][u].y, x[k][u].z, x[k][u].w};
#pragma unroll
          for (int e = 0; e < 7; ++e)
            if (e < nv[k]) d[e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
        }
      }
    return;
  }
  for (int i = tid; i < nslot; i += 256) sm[i] = 0;
  __syncthreads();
  int slot[KC];
#pragma unroll
  for (int k = 0; k < KC; ++k) {
    slot[k] = (head[k] * p.ns + (j0[k] >= a.split)) * P + pp;
    if (nv[k] <= 0) continue;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float f[8], m = 0.f;
      chunk_f32<T>(x[k][u], f);
#pragma unroll
      for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(f[e]));
      atomicMax(&sm[slot[k] + u * p.pp], __float_as_uint(m));   // non-negative floats order as their bits
    }
  }
  __syncthreads();
  for (int i = tid; i < nslot; i += 256) {
    const int seg = i / P, t = t0 + (i - seg * P), s = pos + t;
    const int h = p.ns == 2 ? seg >> 1 : seg;
    const bool lower = p.ns == 2 && (seg & 1);
    const _Float16 s16 = fp16_scale(scale[i], !lower && a.a_int8 ? 127.f : 7.f);
    scale[i] = (float)s16;
    recip[i] = __fdiv_rn(1.f, (float)s16);
    if (t >= a.T || s < 0 || s >= a.cap || (lower && a.rank[h] <= a.split)) continue;
    uint16_t* sp = lower ? (uint16_t*)a.scale2 + b * a.sc2_sb + h * a.sc2_sh + (int64_t)s * a.sc2_ss
                         : (uint16_t*)a.scale + b * a.sc_sb + h * a.sc_sh + (int64_t)s * a.sc_ss;
    *sp = __builtin_bit_cast(uint16_t, s16);
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < KC; ++k) {
    if (nv[k] <= 0) continue;
    const int h = head[k];
    const bool lower = j0[k] >= a.split, i8 = !lower && a.a_int8;
    const int jb = lower ? j0[k] - a.split : j0[k];
    uint8_t* q = (lower ? (uint8_t*)a.data2 + b * a.stride2_b + a.off2[h] : (uint8_t*)a.data + b * a.stride_b + a.off[h]) +
                 (i8 ? jb : jb >> 1);
    const int64_t pitch = lower ? a.pitch2[h] : a.pitch[h];
    const float lo = i8 ? -127.f : -8.f, hi = i8 ? 127.f : 7.f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int t = t0 + u * p.pp + pp, s = pos + t;
      if (t >= a.T || s < 0 || s >= a.cap) continue;
      const float sc = scale[slot[k] + u * p.pp], rc = recip[slot[k] + u * p.pp];
      float f[8];
      chunk_f32<T>(x[k][u], f);
      if (sc < INFINITY) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float y = f[e] * rc;
          f[e] = fmaf(fmaf(-y, sc, f[e]), rc, y);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = __fdiv_rn(f[e], sc);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = fminf(fmaxf(f[e], lo), hi);
      uint8_t* d = q + (int64_t)s * pitch;
      if (i8) {
        uint32_t w[2];
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          const uint32_t e01 = __builtin_amdgcn_perm(rint_bits(f[4 * v + 1], 0.f), rint_bits(f[4 * v], 0.f), 0x0C0C0400u);
          const uint32_t e23 = __builtin_amdgcn_perm(rint_bits(f[4 * v + 3], 0.f), rint_bits(f[4 * v + 2], 0.f), 0x04000C0Cu);
          w[v] = e01 | e23;
        }
        store_bytes(d, (uint64_t)w[0] | ((uint64_t)w[1] << 32), nv[k]);
      } else {
        store_bytes(d, pack_nibbles(f, 8.f), (nv[k] + 1) >> 1);   // past an odd rank: 0 / s, nibble 8
      }
    }
  }
}

// Group-64 V rows: thread -> 8-rank chunk, a group's eight threads reduce its
// minimum and maximum among themselves; U chunks in flight per thread.
template <typename T>
__global__ __launch_bounds__(256) void append_g64_kernel(const VAppendArgs a, int nb) {
  constexpr int U = 4;
  const int b = blockIdx.x / nb;
  const uint32_t first = (uint32_t)(blockIdx.x - b * nb) * (256 * U) + threadIdx.x;
  const uint32_t ncg = (uint32_t)((a.R + 63) >> 6) * 8, total = ncg * (uint32_t)a.T;
  const int pos = a.pos0_dev ? *a.pos0_dev : a.pos0;
  uint4 x[U];
  int tt[U], j0[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t i = min(first + 256 * u, total - 8 + (threadIdx.x & 7));   // past the end: the last group again
    const uint32_t t = i / ncg;
    tt[u] = (int)t;
    j0[u] = 8 * (int)(i - t * ncg);
    const int nv = min(8, a.R - j0[u]);
    x[u] = make_uint4(0, 0, 0, 0);
    if (nv > 0) x[u] = load_chunk((const uint16_t*)a.src + b * a.src_sb + (int64_t)t * a.src_st, j0[u], nv);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int nv = min(8, a.R - j0[u]), s = pos + tt[u];
    float f[8], lo = INFINITY, hi = -INFINITY;
    chunk_f32<T>(x[u], f);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      lo = e < nv ? fminf(lo, f[e]) : lo;
      hi = e < nv ? fmaxf(hi, f[e]) : hi;
    }
#pragma unroll
    for (int o = 4; o >= 1; o >>= 1) {
      lo = fminf(lo, __shfl_xor(lo, o, 8));
      hi = fmaxf(hi, __shfl_xor(hi, o, 8));
    }
    const _Float16 z16 = (_Float16)lo;
    const float z = (float)z16;
    _Float16 s16 = (_Float16)__fdiv_rn(hi - z, 15.f);
    if ((float)s16 == 0.f) s16 = (_Float16)1.0f;
    const float sc = (float)s16;
    if (s < 0 || s >= a.cap) {                        // only a run-time position can land here
      if (a.err != nullptr) *a.err = 1;
      continue;
    }
    if (first + 256 * u >= total) continue;
    if ((threadIdx.x & 7) == 0) {
      const int64_t o = b * a.sc_sb + (int64_t)s * a.sc_ss + (j0[u] >> 6);
      ((uint16_t*)a.scale)[o] = __builtin_bit_cast(uint16_t, s16);
      ((uint16_t*)a.zero)[o] = __builtin_bit_cast(uint16_t, z16);
    }
    if (nv <= 0) continue;
    if (fabsf(sc) < INFINITY) {
      const float rc = __fdiv_rn(1.f, sc);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = f[e] - z;
        float y = d * rc;
        y = fmaf(fmaf(-y, sc, d), rc, y);
        f[e] = fmaf(fmaf(-y, sc, d), rc, y);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = __fdiv_rn(f[e] - z, sc);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = e < nv ? fminf(fmaxf(f[e], 0.f), 15.f) : 0.f;
    store_bytes((uint8_t*)a.data + b * a.stride_b + (int64_t)s * a.stride_s + (j0[u] >> 1), pack_nibbles(f, 0.f),
                (nv + 1) >> 1);
  }
}

template <typename T, int KC>
static void launch_block_t(const KAppendArgs& a, const BlockPlan& p, hipStream_t st) {
  const dim3 grid((unsigned)(a.B * p.nb));
  const size_t lds = (size_t)a.H * p.ns * p.pp * (8 / KC) * 8;
  if (a.fmt == STARKV_FMT_DENSE) hipLaunchKernelGGL((append_block_kernel<T, KC, true>), grid, dim3(256), 0, st, a, p);
  else hipLaunchKernelGGL((append_block_kernel<T, KC, false>), grid, dim3(256), lds, st, a, p);
}

static void launch_block(const KAppendArgs& a, int dtype, hipStream_t st) {
  BlockPlan p = {};
  bool two = false;
  for (int h = 0; h < K_MAX_KV; ++h) {
    p.cstart[h] = h < a.H ? (uint16_t)p.nc : (uint16_t)0xffff;
    if (h >= a.H) continue;
    p.nc += (a.rank[h] + 7) / 8;
    two |= a.rank[h] > a.split;
  }
  p.ns = two ? 2 : 1;
  const int kc = p.nc <= 256 ? 1 : p.nc <= 512 ? 2 : 4;   // at most 64 * 16 (K) or 8192 / 8 (V) chunks
  p.pp = kc == 1 ? 256 / p.nc : 1;
  p.nb = (int)ceil_div(a.T, p.pp * (8 / kc));
  const bool h = dtype == STARKV_F16;
  if (kc == 1) h ? launch_block_t<_Float16, 1>(a, p, st) : launch_block_t<__bf16, 1>(a, p, st);
  else if (kc == 2) h ? launch_block_t<_Float16, 2>(a, p, st) : launch_block_t<__bf16, 2>(a, p, st);
  else h ? launch_block_t<_Float16, 4>(a, p, st) : launch_block_t<__bf16, 4>(a, p, st);
}

static void launch_v_rows(const VAppendArgs& a, int dtype, hipStream_t st) {
  if (a.vq == VQ_G64) {
    const int nb = (int)ceil_div((int64_t)a.T * ceil_div(a.R, 64) * 8, 256 * 4);
    const dim3 grid((unsigned)(a.B * nb));
    if (dtype == STARKV_F16) hipLaunchKernelGGL(append_g64_kernel<_Float16>, grid, dim3(256), 0, st, a, nb);
    else hipLaunchKernelGGL(append_g64_kernel<__bf16>, grid, dim3(256), 0, st, a, nb);
    return;
  }
  // a dense or per-token block row is one head whose scales step by sc_ss
  KAppendArgs k = {};
  k.src = a.src; k.src_sb = a.src_sb; k.src_st = a.src_st;
  k.B = a.B; k.H = 1; k.T = a.T; k.pos0 = a.pos0; k.cap = a.cap; k.pos0_dev = a.pos0_dev; k.err = a.err;
  k.fmt = a.vq == VQ_DENSE ? STARKV_FMT_DENSE : STARKV_FMT_INT4_REF;
  k.data = a.data; k.stride_b = a.stride_b; k.pitch[0] = a.stride_s;
  k.scale = a.scale; k.sc_sb = a.sc_sb; k.sc_ss = a.sc_ss;
  k.split = a.vq == VQ_DENSE ? a.R : a.split; k.a_int8 = a.a_int8;
  k.data2 = a.data2; k.stride2_b = a.stride2_b; k.pitch2[0] = a.stride2_s;
  k.scale2 = a.scale2; k.sc2_sb = a.sc2_sb; k.sc2_ss = a.sc2_ss;
  k.rank[0] = a.R;
  launch_block(k, dtype, st);
}

// Where the chunked kernels take over, from modelled times in ns.  Each has 6
// to 12 us of fixed time (a chain of loads, maxima and divisions, eight passes
// over one workgroup's positions).  The row-per-wave kernels start in 2.8 us
// and take 0.34 ns of the whole chip per row of K or 64-rank group of V (0.53
// with a lower block, 0.21 unquantised); the one wave of a block or dense row
// of V also takes 3.6 or 1.7 ns per rank, whatever the chip does beside it.
// Measured, row-per-wave against chunked, us:
//   K alone, 32 heads: int8 rank 48, 512 positions 8.4 / 8.3; rank 51, 768
//   11.0 / 11.5; rank 8, 768 11.1 / 11.4; split, rank 48, 512 12.3 / 9.9;
//   unquantised rank 51, 1024 9.1 / 8.3.
//   V alone: group-64 R1640, 512 positions 6.6 / 6.0; split R1640, 4096 12.4 /
//   12.9, 8192 22.7 / 18.8; split R512, 8192 10.0 / 11.4, 16384 15.6 / 14.0;
//   split R2560, 512 12.8 / 10.0; dense R512, 16384 8.1 / 9.4, 32768 17.7 /
//   14.1; dense R1640, 2048 6.5 / 6.5, 4096 11.1 / 8.0; dense R2560, 512 7.5 / 6.7.
//   both, in one launch against two: 32 heads, int8 / group-64 R1640, rank 51,
//   512 12.8 / 16.4, 1024 22.6 / 16.8; rank 8, R64, 1024 14.4 / 16.2, 2048 26.0
//   / 16.3; 8 heads of rank 64, R512, 2048 13.6 / 14.7; unquantised rank 96,
//   R2560, 1024 18.0 / 13.4.
// A workgroup holds pp * 8 / KC positions of one batch, 2 at the fewest: runs
// of fewer than 16 stay with the row-per-wave kernels.
static int64_t k_waves_ns(const KAppendArgs& a) {
  int64_t ps = 0;
  for (int h = 0; h < a.H; ++h) ps += a.fmt == STARKV_FMT_DENSE ? 210 : a.rank[h] > a.split ? 530 : 335;
  return ps * a.B * a.T / 1000;
}
static bool k_chunked(const KAppendArgs& a) {
  if (a.T < 16) return false;
  return a.fmt == STARKV_FMT_DENSE ? (int64_t)a.B * a.T * a.H >= 28672 : k_waves_ns(a) >= 8200;   // 24.5 K rows, 15.5 K with a lower block
}
static int64_t v_row_ns(const VAppendArgs& a) {
  return 2800 + (a.vq == VQ_G64 ? 0 : a.vq == VQ_DENSE ? a.R * 17 / 10 : 600 + a.R * 36 / 10);
}
static int64_t v_waves_ns(const VAppendArgs& a) {
  return 335 * (int64_t)a.B * a.T * (a.vq == VQ_G64 ? ceil_div(a.R, 64) : 1) / 1000;
}
static bool v_chunked(const VAppendArgs& a) {
  const int64_t rows = (int64_t)a.B * a.T, groups = ceil_div(a.R, 64);
  if (a.T < 16) return false;
  const bool dense = a.vq == VQ_DENSE;
  if (a.vq == VQ_G64 || groups >= (dense ? 40 : 28)) return rows * groups >= 16384;
  if (dense && groups >= 25) return rows * groups >= 53248;
  return rows >= 24576 || rows * groups >= (dense ? 196608 : 131072);
}
// K and V in launches of their own, either or both chunked
static bool step_apart(const KAppendArgs& k, const VAppendArgs& v) {
  const bool kc = k_chunked(k), vc = v_chunked(v), dense = k.fmt == STARKV_FMT_DENSE;
  if (!kc && !vc) return false;
  const int64_t kw = k_waves_ns(k), vw = v_waves_ns(v), vr = v_row_ns(v);
  bool two = false;
  for (int h = 0; h < k.H; ++h) two = two || (!dense && k.rank[h] > k.split);
  const int64_t kt = !kc ? 2800 + kw : dense ? 6500 : two ? 12000 : 11000;
  const int64_t vt = !vc ? vr + vw : v.vq == VQ_G64 ? 6000 : v.vq == VQ_DENSE ? 6500 : 10500;
  return kt + vt <= vr + kw + vw;
}

int launch_step_append(const StepAppendArgs& a0, int dtype, hipStream_t st) {
  StepAppendArgs a = a0;
  if (step_apart(a.k, a.v)) {
    int e = launch_k_append(a.k, dtype, st);
    if (!e) e = launch_v_append(a.v, dtype, st);
    return !e && a.has_rope ? launch_rope_apply(a.r, dtype, st) : e;
  }
  a.v.gw = a.v.vq == VQ_G64 ? (int)ceil_div(a.v.R, 64) : 1;
  a.nbk = ceil_div((int64_t)a.k.B * a.k.H * a.k.T, 4);
  a.nbv = ceil_div((int64_t)a.v.B * a.v.T * a.v.gw, 4);
  const int64_t nbr = a.has_rope ? ceil_div((int64_t)a.r.B * a.r.H * a.r.T * 64, 256) : 0;
  const int64_t n = a.nbk + a.nbv + nbr;
  if (n == 0) return 0;
  if (dtype == STARKV_F16) hipLaunchKernelGGL(step_append_kernel<_Float16>, dim3((unsigned)n), dim3(256), 0, st, a);
  else hipLaunchKernelGGL(step_append_kernel<__bf16>, dim3((unsigned)n), dim3(256), 0, st, a);
  return (int)hipGetLastError();
}

int launch_k_append(const KAppendArgs& a, int dtype, hipStream_t st) {
  const int64_t rows = (int64_t)a.B * a.H * a.T;
  if (rows == 0) return 0;
  if (k_chunked(a)) {
    launch_block(a, dtype, st);
    return (int)hipGetLastError();
  }
  const dim3 grid((unsigned)ceil_div(rows, 4));
  if (dtype == STARKV_F16) hipLaunchKernelGGL(k_append_kernel<_Float16>, grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL(k_append_kernel<__bf16>, grid, dim3(256), 0, st, a);
  return (int)hipGetLastError();
}

int launch_v_append(const VAppendArgs& a, int dtype, hipStream_t st) {
  const int64_t rows = (int64_t)a.B * a.T;
  if (rows == 0) return 0;
  if (v_chunked(a)) {
    launch_v_rows(a, dtype, st);
    return (int)hipGetLastError();
  }
  VAppendArgs r = a;
  r.gw = a.vq == VQ_G64 ? (int)ceil_div(a.R, 64) : 1;
  const dim3 grid((unsigned)ceil_div(rows * r.gw, 4));
  if (dtype == STARKV_F16) hipLaunchKernelGGL(v_append_kernel<_Float16>, grid, dim3(256), 0, st, r);
  else hipLaunchKernelGGL(v_append_kernel<__bf16>, grid, dim3(256), 0, st, r);
  return (int)hipGetLastError();
}

}  // namespace starkv
