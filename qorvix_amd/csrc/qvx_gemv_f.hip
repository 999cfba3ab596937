// qvx_gemv_f.hip -- GEMV with fp32 activations on gfx950: unquantised weights (F32, F16, BF16), and every
// block format where the integer kernels do not take the call (Q4_1, Q5_1, Q8_1, unaligned weights, row
// pitches they cannot read).
//
// out[v, r] = sum_k W[r, k] * X[v, k]: the reference's qmatmul / qmatmulN (runtime/src/qmatmul.cpp:28-115
// over dequant.cpp's formulas, runtime/src/dequant.cpp:38-255).  Each weight value is the exact
// dequantised fp32 value; products and sums are fp32 FMAs.
//
// One summation order for every form, so qvx_qmatmul_n stays bit-identical to qvx_qmatmul: the row is cut
// into chunks of consecutive elements (16 bytes of an unquantised row; 8 elements of a block format,
// which always share one block and one scale); lane l of a wave sums chunks l, l + 64, ... in order, one
// chain of FMAs in element order; the 64 lane sums are combined by a butterfly (xor 32, 16, ..., 1).
//
// Streaming form (k_gemv_float, up to 4 vectors a launch): one workgroup of 16 waves per CU, the
// activations staged once into LDS as fp32 where they fit.  A wave takes whole rows, a lane its chunks
// in blocks of kU whose loads are all issued before any is used.  A block format's chunk is a few loads
// of 4 to 16 bytes at whatever alignment the block has.
//
// Tiled form (k_gemv_float_many, larger batches): described at the kernel.
#include "qvx_deq.hpp"
#include "qvx_gemv_valu.hpp"

namespace qvx {

namespace {

constexpr size_t kLdsX = 128 * 1024;  // activation staging budget per workgroup

// N bytes from any address.
template <typename V>
__device__ inline V ldu(const uint8_t* p) {
  V v;
  __builtin_memcpy(&v, p, sizeof(V));
  return v;
}

// ---- weight chunks -----------------------------------------------------------------------------------
// Src<T>: E elements a chunk; kU chunks a lane of the streaming form requests at a time; kSeg bytes a segment of
// 64 chunks; kAligned = 16-byte aligned rows; Raw = a chunk's bytes in registers; load() issues its loads (chunk l of the segment at p: the
// lane's part of the address is the same in every segment); widen() forms the fp32 values.
template <uint32_t T> struct Src;

template <uint32_t T> struct SrcPlain {  // 16 bytes of fp32 / fp16 / bf16 values
  static constexpr int E = T == T_F32 ? 4 : 8, kU = 8, kSeg = 1024;
  static constexpr bool kAligned = true;
  typedef uint4 Raw;
  static __device__ inline Raw load(const uint8_t* p, int l) { return *reinterpret_cast<const uint4*>(p + 16 * l); }
  static __device__ inline void widen(const Raw& w, float (&f)[E]) {
    const uint32_t d[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (T == T_F32) {
        f[i] = __uint_as_float(d[i]);
      } else if constexpr (T == T_F16) {
        f[2 * i] = f16lo(d[i]);
        f[2 * i + 1] = f16hi(d[i]);
      } else {
        f[2 * i] = __uint_as_float(d[i] << 16);
        f[2 * i + 1] = __uint_as_float(d[i] & 0xFFFF0000u);
      }
    }
  }
};
template <> struct Src<T_F32> : SrcPlain<T_F32> {};
template <> struct Src<T_F16> : SrcPlain<T_F16> {};
template <> struct Src<T_BF16> : SrcPlain<T_BF16> {};

// Unquantised weights at any alignment: 8 elements a chunk.
template <uint32_t T> struct SrcLoose;
template <> struct SrcLoose<T_F32> {
  static constexpr bool kAligned = false;
  static constexpr int E = 8, kU = 4, kSeg = 2048;
  struct Raw { uint4 a, b; };
  static __device__ inline Raw load(const uint8_t* p, int l) {
    return {ldu<uint4>(p + 32 * l), ldu<uint4>(p + 32 * l + 16)};
  }
  static __device__ inline void widen(const Raw& w, float (&f)[8]) {
    const uint32_t d[8] = {w.a.x, w.a.y, w.a.z, w.a.w, w.b.x, w.b.y, w.b.z, w.b.w};
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = __uint_as_float(d[i]);
  }
};
template <> struct SrcLoose<T_F16> : SrcPlain<T_F16> {
  static constexpr bool kAligned = false;
  static __device__ inline Raw load(const uint8_t* p, int l) { return ldu<uint4>(p + 16 * l); }
};
template <> struct SrcLoose<T_BF16> : SrcPlain<T_BF16> {
  static constexpr bool kAligned = false;
  static __device__ inline Raw load(const uint8_t* p, int l) { return ldu<uint4>(p + 16 * l); }
};

// Four codes less their offset, as signed bytes.
template <int OFF>
__device__ inline uint32_t less4(uint32_t q) {
  return (q + (0x80u - OFF) * 0x01010101u) ^ 0x80808080u;
}

// The formats of 32-element blocks: codes q at byte kQ (8 bits: element e at kQ + e; 4 bits: low nibbles
// elements 0..15, high 16..31), fifth bits at byte kH (-1: none), scale d at byte 0, offset m at byte 2
// (kM) or a constant kOff subtracted from the code.
template <int BB, int kQ, bool kByte, int kH, bool kM, int kOff>
struct Src32 {
  static constexpr bool kAligned = false;
  static constexpr int E = 8, kU = 4, kSeg = 16 * BB;
  struct Raw { uint2 q; uint32_t h, dm; };
  static __device__ inline Raw load(const uint8_t* p, int l) {
    const uint8_t* b = p + (l >> 2) * BB;
    const int e0 = 8 * (l & 3);
    Raw r;
    r.q = ldu<uint2>(b + kQ + (kByte ? e0 : (e0 & 15)));
    if (!kByte) r.q.x >>= e0 < 16 ? 0 : 4, r.q.y >>= e0 < 16 ? 0 : 4;
    r.h = 0;
    if constexpr (kH >= 0) r.h = ldu<uint32_t>(b + kH) >> e0;
    r.dm = kM ? ldu<uint32_t>(b) : (uint32_t)ldu<uint16_t>(b);
    return r;
  }
  // A value is the code's product with d, not a sum in which an infinite scale would meet its own opposite.
  static __device__ inline void widen(const Raw& r, float (&f)[8]) {
    const float d = f16lo(r.dm), m = f16hi(r.dm);
    uint32_t q[2] = {r.q.x, r.q.y};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if constexpr (!kByte) q[i] &= 0x0F0F0F0Fu;
      if constexpr (kH >= 0) q[i] |= Lane<T_Q5_0>::spread4(r.h >> (4 * i));
      if constexpr (kOff > 0) q[i] = less4<kOff>(q[i]);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t b = q[k >> 2] >> (8 * (k & 3));
      if constexpr (kM) f[k] = __builtin_fmaf((float)(b & 0xFFu), d, m);  // the product is exact: one rounding
      else f[k] = (float)(int)(int8_t)b * d;
    }
  }
};
template <> struct Src<T_Q8_0> : Src32<34, 2, true, -1, false, 0> {};
template <> struct Src<T_Q8_1> : Src32<36, 4, true, -1, false, 0> {};
template <> struct Src<T_Q4_0> : Src32<18, 2, false, -1, false, 8> {};
template <> struct Src<T_Q4_1> : Src32<20, 4, false, -1, true, 0> {};
template <> struct Src<T_Q5_0> : Src32<22, 6, false, 2, false, 16> {};
template <> struct Src<T_Q5_1> : Src32<24, 8, false, 4, true, 0> {};

// Q4_K / Q5_K: d, dmin and the 12 bytes of 6-bit scales and mins, Q5_K's fifth bits, the nibbles.
template <bool kFive>
struct SrcK45 {
  static constexpr bool kAligned = false;
  static constexpr int E = 8, kU = 4, BB = kFive ? 176 : 144, kSeg = 2 * BB;
  struct Raw { uint4 hd; uint2 q, h; uint32_t j; };
  static __device__ inline Raw load(const uint8_t* p, int c) {
    const uint8_t* b = p + (c >> 5) * BB;
    const int e0 = 8 * (c & 31), g = e0 >> 6, l = e0 & 31, hi = (e0 >> 5) & 1;
    Raw r;
    r.hd = ldu<uint4>(b);
    r.q = ldu<uint2>(b + BB - 128 + 32 * g + l);
    r.h = make_uint2(0, 0);
    if constexpr (kFive) r.h = ldu<uint2>(b + 16 + l);
    r.j = (uint32_t)(2 * g + hi);
    return r;
  }
  static __device__ inline void widen(const Raw& r, float (&f)[8]) {
    const uint32_t j = r.j, j4 = 8u * (j & 3u), sh = 4u * (j & 1u);
    const uint32_t y = r.hd.y >> j4, z = r.hd.z >> j4, w = r.hd.w >> j4;  // scale bytes j%4, 4 + j%4, 8 + j%4
    const uint32_t sc = j < 4 ? y & 63u : (w & 15u) | (((y >> 6) & 3u) << 4);
    const uint32_t mn = j < 4 ? z & 63u : ((w >> 4) & 15u) | (((z >> 6) & 3u) << 4);
    const float ds = f16lo(r.hd.x) * (float)sc, dm = f16hi(r.hd.x) * (float)mn;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t b = 8u * (uint32_t)(k & 3);
      uint32_t q = ((k < 4 ? r.q.x : r.q.y) >> (b + sh)) & 15u;
      if constexpr (kFive) q |= (((k < 4 ? r.h.x : r.h.y) >> (b + j)) & 1u) << 4;
      f[k] = __builtin_fmaf(ds, (float)q, -dm);  // the product is exact: one rounding
    }
  }
};
template <> struct Src<T_Q4_K> : SrcK45<false> {};
template <> struct Src<T_Q5_K> : SrcK45<true> {};

template <> struct Src<T_Q6_K> {
  static constexpr bool kAligned = false;
  static constexpr int E = 8, kU = 4, kSeg = 420;
  struct Raw { uint2 l, h; uint32_t sc, d; };
  static __device__ inline Raw load(const uint8_t* p, int c) {
    const uint8_t* b = p + (c >> 5) * 210;
    const int e0 = 8 * (c & 31), h = e0 >> 7, quarter = (e0 >> 5) & 3, l = e0 & 31;
    Raw r;
    r.l = ldu<uint2>(b + 64 * h + 32 * (quarter & 1) + l);
    r.h = ldu<uint2>(b + 128 + 32 * h + l);
    r.sc = b[192 + 8 * h + 2 * quarter + (l >> 4)];
    r.d = ldu<uint16_t>(b + 208);
    const uint32_t nsh = (quarter & 2) ? 4u : 0u, hsh = 2u * (uint32_t)quarter;
    r.l.x >>= nsh, r.l.y >>= nsh;
    r.h.x >>= hsh, r.h.y >>= hsh;
    return r;
  }
  static __device__ inline void widen(const Raw& r, float (&f)[8]) {
    const float ds = f16lo(r.d) * (float)(int)(int8_t)r.sc;
    const uint32_t q[2] = {less4<32>((r.l.x & 0x0F0F0F0Fu) | ((r.h.x & 0x03030303u) << 4)),
                           less4<32>((r.l.y & 0x0F0F0F0Fu) | ((r.h.y & 0x03030303u) << 4))};
#pragma unroll
    for (int k = 0; k < 8; ++k) f[k] = (float)(int)(int8_t)(q[k >> 2] >> (8 * (k & 3))) * ds;
  }
};

// Workgroup barrier for LDS only: this wave's LDS accesses complete, then s_barrier (__syncthreads would
// also wait for the global loads in flight, which the kernels below keep across their barriers).
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// A chunk's activations in LDS: the XP = E / 4 float4s of chunk c lie in XP planes of `plane` words, so the
// 64 lanes of a read hit consecutive words.
template <int E>
__device__ inline void read_x(const float4* xs, int plane, int c, float (&x)[E]) {
#pragma unroll
  for (int q = 0; q < E / 4; ++q) {
    const float4 t = xs[q * plane + c];
    x[4 * q] = t.x, x[4 * q + 1] = t.y, x[4 * q + 2] = t.z, x[4 * q + 3] = t.w;
  }
}

// The butterfly over a wave's lane sums, xor 32, 16, 8, 4, 2, 1: every lane ends with the same bits.  Once the
// lanes that differ in bit 3 agree, a rotation by 4 within the row of 16 reaches the lane at xor 4.
__device__ inline float row_sum16(float s) {
  s += dpp<0x128>(s);  // row_ror:8
  s += dpp<0x124>(s);  // row_ror:4
  s += dpp<kXor2>(s);
  s += dpp<kXor1>(s);
  return s;
}
// a + (a of lane xor N) in the lanes with bit N clear, b + (b of lane xor N) in the others.
template <int N>
__device__ inline float pair_sum(float a, float b) {
  const int ia = __builtin_bit_cast(int, a), ib = __builtin_bit_cast(int, b);
  const auto t = N == 32 ? __builtin_amdgcn_permlane32_swap(ia, ib, false, false)
                         : __builtin_amdgcn_permlane16_swap(ia, ib, false, false);
  return __builtin_bit_cast(float, (int)t[0]) + __builtin_bit_cast(float, (int)t[1]);
}

// ---- streaming form ----------------------------------------------------------------------------------
// STAGE: the NV vectors are staged in LDS; otherwise (rows too long for it) they are read from global
// memory, nv <= NV of them.
template <typename S, int NV, bool STAGE>
__global__ __launch_bounds__(1024) void k_gemv_float(const uint8_t* __restrict__ W, const float* __restrict__ X,
                                                     float* __restrict__ Y, int rows, int cols, size_t row_bytes,
                                                     int nv) {
  constexpr int E = S::E, kU = S::kU, XP = E / 4;
  extern __shared__ float4 xs4[];  // [NV][XP][cols / E]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
  const int nchunk = cols / E, stride = (int)gridDim.x * nw;
  // Requests the next kU chunks of the wave's rows, in order; the first before the activations are staged.
  // Block formats keep the next ones in flight while the last are decoded and summed (Q6_K 32000 x 3072:
  // 96 -> 47 us); unquantised chunks, eight 16-byte loads a block already, do without (4096 x 4096 fp16:
  // 9.3 us with, 8.7 without).
  constexpr bool kAhead = S::kU < 8;
  // Lanes past the row's last chunk repeat it (their sums skip it), so no load is in a branch.
  const int nseg = (nchunk + 63) / 64, lastc = min(lane, nchunk - 64 * (nseg - 1) - 1);
  int r = (int)blockIdx.x * nw + wave, g0 = 0;
  auto request = [&](typename S::Raw (&w)[kU]) __attribute__((always_inline)) {
    const uint8_t* rp = W + (size_t)min(r, rows - 1) * row_bytes;
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int g = min(g0 + u, nseg - 1);
      w[u] = S::load(rp + (size_t)g * S::kSeg, g == nseg - 1 ? lastc : lane);
    }
    g0 += kU;
    if (g0 >= nseg) g0 = 0, r += stride;
  };
  typename S::Raw w[kU], wn[kU];
  request(w);
  bool fresh = true;  // w holds the block about to be summed
  if constexpr (STAGE) {
    const int n4 = nv * cols / 4, per = cols / 4;
    for (int i = threadIdx.x; i < n4; i += (int)blockDim.x) {
      const int v = NV == 1 ? 0 : i / per, j = i - v * per;
      xs4[v * per + (j % XP) * nchunk + j / XP] = reinterpret_cast<const float4*>(X)[i];
    }
    lds_barrier();
  }
  for (int row = (int)blockIdx.x * nw + wave; row < rows; row += stride) {
    float acc[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[v] = 0.0f;
    for (int b0 = 0; b0 < nchunk; b0 += 64 * kU) {
      if constexpr (kAhead) request(wn);
      else if (!fresh) request(w);
      fresh = false;
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        if (b0 + 64 * u >= nchunk) break;  // uniform
        const int c = b0 + 64 * u + lane;
        if (c < nchunk) {
          float f[E];
          S::widen(w[u], f);
#pragma unroll
          for (int v = 0; v < NV; ++v) {
            float x[E];
            if constexpr (STAGE) {
              read_x<E>(xs4 + v * (cols / 4), nchunk, c, x);
            } else {
              const float4* xp = reinterpret_cast<const float4*>(X + (size_t)min(v, nv - 1) * cols + E * c);
#pragma unroll
              for (int q = 0; q < XP; ++q) {
                const float4 t = xp[q];
                x[4 * q] = t.x, x[4 * q + 1] = t.y, x[4 * q + 2] = t.z, x[4 * q + 3] = t.w;
              }
            }
#pragma unroll
            for (int e = 0; e < E; ++e) acc[v] = __builtin_fmaf(f[e], x[e], acc[v]);
          }
        }
      }
      if constexpr (kAhead)
#pragma unroll
        for (int u = 0; u < kU; ++u) w[u] = wn[u];
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const float s = row_sum16(pair_sum<16>(pair_sum<32>(acc[v], acc[v]), pair_sum<32>(acc[v], acc[v])));
      if (lane == 0 && v < nv) Y[(size_t)v * rows + row] = s;
    }
  }
}

// ---- tiled form --------------------------------------------------------------------------------------
// A workgroup of 8 waves computes 32 rows x 8 vectors, a wave 4 rows: lane l holds the 4 x 8 lane sums of its
// chunks, so a chunk's weights serve 8 vectors and its activations 4 rows.  The activations come through a
// two-stage LDS ring of two segments (128 chunks) of every vector, shared by the waves; the next stage's
// activations and weights are requested before a stage is summed.  At the end the 32 sums of 64 lanes meet in
// 8 registers: permlane swaps add two sums at a time over xor 32 and 16 (lanes 16 q .. 16 q + 15 then hold
// sums 8 (q % 2) + 16 (q / 2) + j), DPP adds the rest -- the butterfly's own pairs.
// Of a 384-wide encoder's launches VALU instructions fill 0.21 of the cycles and waves wait 0.47 of theirs: short rows leave
// half of a stage empty, and ramp, the first stage's loads and the butterfly are most of a launch.  Measured on MI355X, graph-replayed:
// fp16 384 x 1536 at 256 vectors 12.6 us, where 64 launches of the streaming form took 290; 14336 x 4096 at
// 16 vectors 110 -> 57 us; Q6_K 32000 x 3072 at 16 570 -> 114 us (the byte-by-byte decode this file's block
// chunks replaced; its one-vector call 126 -> 43, 2048 x 5632 24 -> 7.8).
constexpr int kTV = 8, kTR = 4, kTS = 2, kTW = 8;  // vectors, rows a wave, segments a stage, waves
template <typename S>
__global__ __launch_bounds__(64 * kTW) void k_gemv_float_many(const uint8_t* __restrict__ W, const float* __restrict__ X,
                                                              const float* __restrict__ bias, float* __restrict__ Y,
                                                              int rows, int cols, int nvec, size_t row_bytes) {
  constexpr int E = S::E, XP = E / 4, kStage = 64 * kTS * XP;  // float4s of a vector a stage
  constexpr int NX = kTV * kStage / (64 * kTW);
  static_assert(kTV * kStage % (64 * kTW) == 0, "whole float4s a thread");
  __shared__ float4 xs[2][kTV * kStage];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r0 = ((int)blockIdx.x * kTW + wave) * kTR, v0 = (int)blockIdx.y * kTV;
  const int nchunk = cols / E, nst = (nchunk + 64 * kTS - 1) / (64 * kTS);
  const int nseg = (nchunk + 63) / 64, lastc = min(lane, nchunk - 64 * (nseg - 1) - 1);  // as the streaming form's

  auto load_x = [&](int st, float4 (&x)[NX]) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < NX; ++k) {
      const int p = tid + 64 * kTW * k, v = min(v0 + p / kStage, nvec - 1), j = st * kStage + p % kStage;
      x[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (j < nchunk * XP) x[k] = reinterpret_cast<const float4*>(X + (size_t)v * cols)[j];
    }
  };
  auto store_x = [&](int h, const float4 (&x)[NX]) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < NX; ++k) {
      const int p = tid + 64 * kTW * k, j = p % kStage;
      xs[h][p / kStage * kStage + (j % XP) * (64 * kTS) + j / XP] = x[k];
    }
  };
  auto load_w = [&](int st, typename S::Raw (&w)[kTS][kTR]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kTS; ++u)
#pragma unroll
      for (int i = 0; i < kTR; ++i) {
        const int g = min(kTS * st + u, nseg - 1);
        w[u][i] = S::load(W + (size_t)min(r0 + i, rows - 1) * row_bytes + (size_t)g * S::kSeg,
                          g == nseg - 1 ? lastc : lane);
      }
  };

  float acc[kTR * kTV];
#pragma unroll
  for (int o = 0; o < kTR * kTV; ++o) acc[o] = 0.0f;
  typename S::Raw w[kTS][kTR];
  float4 x[NX];
  load_x(0, x);
  load_w(0, w);
  store_x(0, x);
  lds_barrier();
  for (int st = 0; st < nst; ++st) {
    const bool more = st + 1 < nst;
    if (more) load_x(st + 1, x);
#pragma unroll
    for (int u = 0; u < kTS; ++u) {
      float f[kTR][E];
#pragma unroll
      for (int i = 0; i < kTR; ++i) S::widen(w[u][i], f[i]);
      const int c = 64 * (kTS * st + u) + lane;
      const int gn = min(kTS * (st + 1) + u, nseg - 1);  // this segment's registers take the next stage's
#pragma unroll
      for (int i = 0; i < kTR; ++i)
        w[u][i] = S::load(W + (size_t)min(r0 + i, rows - 1) * row_bytes + (size_t)gn * S::kSeg,
                          gn == nseg - 1 ? lastc : lane);
      if (c < nchunk) {
#pragma unroll
        for (int v = 0; v < kTV; ++v) {
          float xv[E];
          read_x<E>(&xs[st & 1][v * kStage], 64 * kTS, 64 * u + lane, xv);
#pragma unroll
          for (int i = 0; i < kTR; ++i)
#pragma unroll
            for (int e = 0; e < E; ++e) acc[i * kTV + v] = __builtin_fmaf(f[i][e], xv[e], acc[i * kTV + v]);
        }
      }
    }
    if (more) store_x((st + 1) & 1, x);
    lds_barrier();
  }
  // 32 sums -> 16 -> 8 registers -> one sum a row of 16 lanes and register
  float s[8];
#pragma unroll
  for (int j = 0; j < 8; ++j)
    s[j] = row_sum16(pair_sum<16>(pair_sum<32>(acc[j], acc[j + 16]), pair_sum<32>(acc[j + 8], acc[j + 24])));
  const int q = lane >> 4, j = lane & 15;
  float t = s[0];
#pragma unroll
  for (int k = 1; k < 8; ++k) t = j == k ? s[k] : t;
  const int o = j + 8 * (q & 1) + 16 * (q >> 1), r = r0 + o / kTV, v = v0 + o % kTV;
  if (j < 8 && r < rows && v < nvec) Y[(size_t)v * rows + r] = bias ? t + bias[r] : t;
}

template <typename S>
void launch_many(const uint8_t* w, const float* X, const float* bias, float* Y, int nvec, int rows, int cols,
                 size_t row_bytes, hipStream_t s) {
  const dim3 grid((unsigned)((rows + kTR * kTW - 1) / (kTR * kTW)), (unsigned)((nvec + kTV - 1) / kTV));
  k_gemv_float_many<S><<<grid, 64 * kTW, 0, s>>>(w, X, bias, Y, rows, cols, nvec, row_bytes);
}

template <typename S, int NV, bool STAGE>
bool launch_nv(const uint8_t* w, const float* X, float* Y, int rows, int cols, size_t row_bytes, int nv,
               hipStream_t s) {
  auto kern = &k_gemv_float<S, NV, STAGE>;
  const size_t lds = STAGE ? (size_t)NV * cols * 4 : 0;
  static LdsLimit lim;
  if (!lds_ready(reinterpret_cast<const void*>(kern), lim, lds)) return false;
  // 16 waves a workgroup, 8 or 4 where that would leave CUs without one, but not of aligned unquantised weights of
  // 512 rows or more with much to stage, which 4 waves take longer over than the CUs save (fp16 1024 x 11008 at 2
  // vectors 13.8 us with 4, 11.0 with 16, at 5888 columns 13.6 and 15 the other way; fp32 1024 x 5888 at 4 14.3 and 11.0, at 11008 and 2 16.7 and
  // 19.5; Q6_K 64 x 11008 at 2 14.6 and 16.6).
  const bool stage = S::kAligned && rows >= 2 * kCUs && rows < 8 * kCUs &&
                     (S::E == 4 ? cols <= 8192 && lds >= 64 * 1024 : cols > 8192 && lds >= 80 * 1024);
  const int nw = rows >= 16 * kCUs || stage ? 16 : rows >= 8 * kCUs ? 8 : 4;
  const int nwg = (int)std::min<int64_t>(kCUs, ((int64_t)rows + nw - 1) / nw);
  kern<<<(unsigned)nwg, (unsigned)(64 * nw), lds, s>>>(w, X, Y, rows, cols, row_bytes, nv);
  return true;
}

constexpr int kGridY = 65535;  // most tiles of vectors a launch may have

template <typename S>
bool launch_src(const void* w, const float* X, float* Y, const float* bias, int nvec, int rows, int cols,
                size_t row_bytes, bool tiled, hipStream_t s) {
  const auto* wb = static_cast<const uint8_t*>(w);
  if (tiled) {
    for (int64_t v0 = 0; v0 < nvec; v0 += kTV * (int64_t)kGridY)
      launch_many<S>(wb, X + v0 * cols, bias, Y + v0 * rows, (int)std::min<int64_t>(kTV * (int64_t)kGridY, nvec - v0),
                     rows, cols, row_bytes, s);
    return true;
  }
  // vectors per launch: as many (4, 2 or 1) as the LDS budget stages, four unstaged ones otherwise; 3 and 5 to 8 too
  // on rows of up to 1024 elements, whose launches are all ramp (Q6_K 1024 x 256 at 5 7.3 -> 4.9 us, at 7, three launches,
  // 10.3 -> 4.9; but fp16 256 x 2816 at 5 in one launch 9.3 us, in two 8.0).
  const size_t fit = kLdsX / ((size_t)cols * 4);
  for (int v0 = 0; v0 < nvec;) {
    const int left = nvec - v0, most = cols <= 1024 ? 8 : fit >= 4 || fit == 0 ? 4 : fit >= 2 ? 2 : 1;
    const int nv = left == 3 && fit > 0 && cols > 1024 ? 2 : std::min(left, most);
    const float* Xv = X + (size_t)v0 * cols;
    float* Yv = Y + (size_t)v0 * rows;
    bool ok;
    if (fit > 0)
      ok = nv > 4    ? launch_nv<S, 8, true>(wb, Xv, Yv, rows, cols, row_bytes, nv, s)
           : nv > 2  ? launch_nv<S, 4, true>(wb, Xv, Yv, rows, cols, row_bytes, nv, s)
           : nv == 2 ? launch_nv<S, 2, true>(wb, Xv, Yv, rows, cols, row_bytes, nv, s)
                     : launch_nv<S, 1, true>(wb, Xv, Yv, rows, cols, row_bytes, nv, s);
    else
      ok = nv > 2    ? launch_nv<S, 4, false>(wb, Xv, Yv, rows, cols, row_bytes, nv, s)
           : nv == 2 ? launch_nv<S, 2, false>(wb, Xv, Yv, rows, cols, row_bytes, nv, s)
                     : launch_nv<S, 1, false>(wb, Xv, Yv, rows, cols, row_bytes, nv, s);
    if (!ok) return false;
    v0 += nv;
  }
  return true;
}

}  // namespace

// Whether a batch takes the tiled form (its launch adds the bias) rather than the streaming form four vectors a
// launch.  Up to 8 vectors that is two launches, which are shorter on fewer rows than fill the chip with
// tiles (fp16 at 5: 1024 x 4096 10.4 us against 16.4, 4096 x 4096 16.2 against 18.1, 14336 x 4096 47.9
// against 34.8).
bool gemv_float_tiled(int nvec, int rows) { return nvec >= 9 || (nvec >= 5 && rows >= 8192); }

// GEMV over unquantised weights with 16-byte-aligned weights and activations and 16-byte row pitch, in
// chunks of 16 bytes.  Returns false, having launched nothing, for another type, a row that is not
// whole chunks, or a row whose activations do not fit the LDS budget (the loose form takes those).
// bias only with a tiled call.
bool launch_gemv_float(uint32_t t, const void* w, const float* X, float* Y, const float* bias, int nvec, int rows,
                       int cols, size_t row_bytes, hipStream_t s) {
  if (cols % (t == T_F32 ? 4 : 8) != 0 || (size_t)cols * 4 > kLdsX) return false;
  const bool tiled = gemv_float_tiled(nvec, rows);
  switch (t) {
    case T_F32: return launch_src<Src<T_F32>>(w, X, Y, bias, nvec, rows, cols, row_bytes, tiled, s);
    case T_F16: return launch_src<Src<T_F16>>(w, X, Y, bias, nvec, rows, cols, row_bytes, tiled, s);
    case T_BF16: return launch_src<Src<T_BF16>>(w, X, Y, bias, nvec, rows, cols, row_bytes, tiled, s);
    default: return false;
  }
}

// GEMV over weights at any alignment, in chunks of 8 elements: cols % 8 == 0, X 16-byte aligned (and fp32
// weights dword aligned).  bias only with a tiled call.
bool launch_gemv_loose(uint32_t t, const void* w, const float* X, float* Y, const float* bias, int nvec, int rows,
                       int cols, size_t row_bytes, hipStream_t s) {
  if (cols % 8 != 0 || (reinterpret_cast<uintptr_t>(X) & 15u) != 0 ||
      (t == T_F32 && (reinterpret_cast<uintptr_t>(w) & 3u) != 0))
    return false;
  const bool tiled = gemv_float_tiled(nvec, rows);
  switch (t) {
    case T_F32: return launch_src<SrcLoose<T_F32>>(w, X, Y, bias, nvec, rows, cols, row_bytes, tiled, s);
    case T_F16: return launch_src<SrcLoose<T_F16>>(w, X, Y, bias, nvec, rows, cols, row_bytes, tiled, s);
    case T_BF16: return launch_src<SrcLoose<T_BF16>>(w, X, Y, bias, nvec, rows, cols, row_bytes, tiled, s);
    case T_Q8_0: return launch_src<Src<T_Q8_0>>(w, X, Y, bias, nvec, rows, cols, row_bytes, tiled, s);
    case T_Q8_1: return launch_src<Src<T_Q8_1>>(w, X, Y, bias, nvec, rows, cols, row_bytes, tiled, s);
    case T_Q4_0: return launch_src<Src<T_Q4_0>>(w, X, Y, bias, nvec, rows, cols, row_bytes, tiled, s);
    case T_Q4_1: return launch_src<Src<T_Q4_1>>(w, X, Y, bias, nvec, rows, cols, row_bytes, tiled, s);
    case T_Q5_0: return launch_src<Src<T_Q5_0>>(w, X, Y, bias, nvec, rows, cols, row_bytes, tiled, s);
    case T_Q5_1: return launch_src<Src<T_Q5_1>>(w, X, Y, bias, nvec, rows, cols, row_bytes, tiled, s);
    case T_Q4_K: return launch_src<Src<T_Q4_K>>(w, X, Y, bias, nvec, rows, cols, row_bytes, tiled, s);
    case T_Q5_K: return launch_src<Src<T_Q5_K>>(w, X, Y, bias, nvec, rows, cols, row_bytes, tiled, s);
    case T_Q6_K: return launch_src<Src<T_Q6_K>>(w, X, Y, bias, nvec, rows, cols, row_bytes, tiled, s);
    default: return false;
  }
}

}  // namespace qvx
