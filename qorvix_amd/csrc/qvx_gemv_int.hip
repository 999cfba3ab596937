// qvx_gemv_int.hip -- batched GEMV over Q8_0 / Q4_0 / Q5_0 weights on the matrix cores of gfx950.
//
// out[v, r] = sum_k dequant(W)[r, k] * X[v, k] (+ bias[r]) for a batch of vectors: the reference's
// qmatmulN at its encoders' sizes (runtime/src/qmatmul.cpp:64-115, "dequantize each block once for all
// nVec dot products", runtime/include/qorvix/runtime/qmatmul.hpp:24-32), each output bit-identical to
// the one-vector VALU kernel (k_gemv, qvx_gemv_valu.hpp):
//  * the same 64-element slots and the same 15-bit fixed-point activations (convert_quant), converted
//    once per call by k_int_conv instead of once per workgroup;
//  * the same exact integer sums per 32-element block: one v_mfma_i32_32x32x32_i8 multiplies the qh and
//    ql bytes of 16 vectors with the signed codes of 32 weight rows, T = (qh sum) * 128 + (ql sum);
//  * the same float fold, fma(d1, T1, d0 * T0) * sx, rounded before it is summed (the one-vector kernel
//    takes Q4_0 as 16 (n - 8) and multiplies by 1/16 at the end: exact scalings by a power of two);
//  * the same reduction: a balanced pairwise tree over each 64 consecutive slots (over the next power of
//    two, at least 8, for shorter rows), the 64-slot sums added in order.  The one-vector kernel's
//    padding lanes add their mirrored last slot times 0: a zero of that slot's sign, or NaN where the
//    slot's sum is not finite, which takes a non-finite scale.  Here padding slots add -0, the same sum (a
//    zero sum is -0 only where every slot's is, the last one's included), and a padded row whose last
//    slot's scales are not finite is NaN.
#include "qvx_gemv_valu.hpp"

namespace qvx {

namespace {

constexpr int kC = 4;  // slots a chunk: one LDS stage a wave's K part

// Workgroup barrier for LDS only (__syncthreads would also wait for the operands in flight).
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x16_t __attribute__((ext_vector_type(16)));

// Per format: bytes of a 64-element slot, and a lane's operands of one slot of its row: the codes of
// elements 16g .. 16g + 15 of the slot's two 32-element blocks as signed bytes, and the block scales.
// w = the slot's bytes in LDS (dword aligned).
template <uint32_t T> struct IntFmt;
// A zero where a slot's two scales are finite, else NaN.  p = the slot in memory (2-byte aligned).
template <uint32_t T>
__device__ inline float scales_zero(const uint8_t* p) {
  const float d0 = f16lo(ldg2(p)), d1 = f16lo(ldg2(p + IntFmt<T>::kSlot / 2));
  return __builtin_fmaf(d1, 0.0f, d0 * 0.0f);
}
template <> struct IntFmt<T_Q8_0> {
  static constexpr int kSlot = 68;
  static __device__ inline void codes(const uint32_t* w, int g, uint32_t (&c0)[4], uint32_t (&c1)[4], float& d0,
                                      float& d1) {
    uint32_t a[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) a[i] = w[4 * g + i];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      c0[i] = align_bytes(a[i + 1], a[i], 2);
      c1[i] = w[9 + 4 * g + i];
    }
    d0 = f16lo(w[0]);
    d1 = f16hi(w[8]);
  }
};
// (n + bias) ^ 0x80 per byte: the code less its offset as a signed byte
__device__ inline uint32_t signed4(uint32_t n, uint32_t bias) { return (n + bias) ^ 0x80808080u; }
template <> struct IntFmt<T_Q4_0> {
  static constexpr int kSlot = 36;
  static __device__ inline void codes(const uint32_t* w, int g, uint32_t (&c0)[4], uint32_t (&c1)[4], float& d0,
                                      float& d1) {
    uint32_t a[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) a[i] = w[i];
    const uint32_t sh = 4u * (uint32_t)g;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      c0[i] = signed4((align_bytes(a[i + 1], a[i], 2) >> sh) & 0x0F0F0F0Fu, 0x78787878u);
      c1[i] = signed4((a[5 + i] >> sh) & 0x0F0F0F0Fu, 0x78787878u);
    }
    d0 = f16lo(a[0]);
    d1 = f16hi(a[4]);
  }
};
template <> struct IntFmt<T_Q5_0> {
  static constexpr int kSlot = 44;
  static __device__ inline void codes(const uint32_t* w, int g, uint32_t (&c0)[4], uint32_t (&c1)[4], float& d0,
                                      float& d1) {
    uint32_t a[11];
#pragma unroll
    for (int i = 0; i < 11; ++i) a[i] = w[i];
    const uint32_t sh = 4u * (uint32_t)g;
    const uint32_t h0 = align_bytes(a[1], a[0], 2) >> (4u * sh), h1 = a[6] >> (4u * sh);  // 16 fifth bits
    using L5 = Lane<T_Q5_0>;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      c0[i] = signed4(((align_bytes(a[i + 2], a[i + 1], 2) >> sh) & 0x0F0F0F0Fu) | L5::spread4(h0 >> (4 * i)),
                      0x70707070u);
      c1[i] = signed4(((a[7 + i] >> sh) & 0x0F0F0F0Fu) | L5::spread4(h1 >> (4 * i)), 0x70707070u);
    }
    d0 = f16lo(a[0]);
    d1 = f16hi(a[5]);
  }
};

// ---- activations -------------------------------------------------------------------------------------
// Workspace of a call: per 16-vector tile and slot, the two A fragments (block b: lane l's 16 bytes hold
// elements 16 (l/32) .. +15 of vector (l%32)/2's qh (l even) or ql bytes), then the 16 steps sx in
// the order the accumulators hold the vectors: entry 8g + 2j + b is vector 4j + 2g + b.
constexpr size_t kFragBytes = 2 * 1024;
inline size_t int_ws_bytes(int nvec, int S) {
  const size_t nvt = ((size_t)nvec + 15) / 16;
  return nvt * S * (kFragBytes + 64);
}
// Whether a call takes this form rather than the VALU kernel, which takes four vectors a launch, two or one for
// the rest (5 vectors are two launches, 7 are three).  This form's time hardly depends on the batch, but grows with K
// where its workgroups are few: a wave's K part is a serial chain.  Measured on MI355X, graph-replayed over distinct
// weights, the VALU kernel against this form:
//  * from 9 vectors it is faster on most shapes (4096 x 4096 at 12: Q8_0 23.6 -> 18.9 us, Q4_0 24.0 -> 12.8; 1024 x 4096
//    Q8_0 at 12 15.2 -> 15.0), not on few long rows: Q8_0 1024 x 4096 at 9 14.5 against 15.5, 1024 x 8192 at 12 21.3
//    against 23.9, 256 x 28672 at 12 56 against 65 and at 16 75 against 72, 2048 x 14336 at 9 1.16 times as long; Q5_0 256
//    x 14336 at 9 1.07;
//  * of 5 to 8, the 4- and 5-bit formats on weights of 16 Mi elements (Q4_0 4096 x 4096 at 8: 16.1 -> 12.6; 1024 x
//    4096: 10.7 against 11.1), past 8192 columns only from 2048 rows on, 5 and 6 from 4096 (2048 x 14336 at 5 1.36
//    times as long, 4096 x 14336 at 5 27.9 against 31.1 and at 6 equal);
//  * Q8_0 at 7 and 8 (5 and 6 are two launches of the VALU kernel, the second a short one: 8192 x 6144 at 6 1.42 times
//    as long) on 4096 rows and weights of 32 Mi elements (11008 x 4096 at 8: 33.8 -> 27.5), at 8 to 48 Mi where columns
//    are no more than 8192 (32000 x 4096 at 7 0.87 of the time, at 8 1.07).
inline bool int_batch(uint32_t t, int nvec, int rows, int cols) {
  const int64_t n = (int64_t)rows * cols, Mi = (int64_t)1 << 20;
  if (t == T_Q8_0) {
    if (nvec >= 9) {
      const int least = cols < 4096 || rows > 2048 ? 9 : rows > 1024 || cols <= 4096 ? 11 : cols < 14336 ? 13 : 17;
      return nvec >= least;
    }
    if (nvec < 7 || rows < 4096 || n < 32 * Mi) return false;
    return cols > 8192 ? rows > 4096 || n < 48 * Mi : n < 48 * Mi || (nvec == 7 && rows > 8192);
  }
  if (nvec >= 9) return nvec >= 11 || t != T_Q5_0 || rows > 1024 || cols < 6144;
  if (nvec < 5 || n < 16 * Mi) return false;
  if (cols <= 8192) return true;
  return rows >= (nvec <= 6 ? 4096 : 2048) && (nvec > 5 || rows > 4096 || cols < 14336);
}
// Vectors converted at a time: all of a call, or as many whole tiles as keep the workspace within 64 MiB.
inline int int_chunk_vectors(int nvec, int S) {
  const size_t per = int_ws_bytes(16, S);
  const int most = 16 * (int)std::max<size_t>(4, ((size_t)64 << 20) / per);
  return std::min(nvec, most);
}

__global__ __launch_bounds__(256) void k_int_conv(const float* __restrict__ X, int nvec, int cols, int S,
                                                  uint8_t* __restrict__ frag, float* __restrict__ step, int ntask) {
  const int t0 = (int)blockIdx.x * 256 + (int)threadIdx.x, t = min(t0, ntask - 1);
  const int vs = t >> 3, part = t & 7, run = part >> 1, hf = part & 1;  // eight tasks a slot, as k_gemv's
  const int v = vs / S, s = vs - v * S;
  const float4* x = reinterpret_cast<const float4*>(X + (size_t)min(v, nvec - 1) * cols + 64 * s + 16 * run + 8 * hf);
  float4 x0 = x[0], x1 = x[1];
  if (v >= nvec) x0 = x1 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);  // the last tile's padding vectors
  Quant8 q;
  convert_quant<4>(x0, x1, q);
  if (t0 >= ntask) return;
  const int vt = v >> 4, vl = v & 15;
  uint8_t* f = frag + ((size_t)vt * S + s) * kFragBytes + (run >> 1) * 1024 + (2 * vl + 32 * (run & 1)) * 16 + 8 * hf;
  *reinterpret_cast<uint2*>(f) = make_uint2(q.h[0], q.h[1]);
  *reinterpret_cast<uint2*>(f + 16) = make_uint2(q.l[0], q.l[1]);
  if (part == 0) step[((size_t)vt * S + s) * 16 + 8 * ((vl >> 1) & 1) + 2 * (vl >> 2) + (vl & 1)] = q.sx;
}

// ---- the product -------------------------------------------------------------------------------------
// Workgroup: one tile of 32 rows, VT 16-vector tiles (blockIdx.y) and KS parts of every 64-slot block,
// a wave each; wave (vt, ks) folds slots [64 b + 64/KS * ks, + 64/KS) of each block b for its vectors,
// and the parts -- whole subtrees -- are added through LDS.  The 32 rows' bytes of the next kC slots of
// every part are copied into one half of an LDS ring while the other half is folded, so the weights are
// read from memory once per VT * 16 vectors.
// The fold is 8 VALU instructions per row, vector and slot of some 110 a wave issues, but over an encoder layer's launches
// (577 x 1024, Q8_0) VALU instructions fill 0.19 of the SIMDs' cycles and MFMAs 0.03: the 320 workgroups of a 1024-row
// weight lie unevenly on 256 CUs, one or two waves a SIMD, and each wave is a chain of chunks.  Measured on MI355X: 577
// vectors of 1024 on 1024 rows of Q8_0, 12.6 us beside a 4.8 us conversion, where 145 launches of the
// one-vector kernel took 580; 4096 rows 31 us; 4096 x 4096 at 64 vectors 121 -> 26 us with the conversion.
template <uint32_t T, int KS, int VT>
__global__ __launch_bounds__(64 * KS * VT, 2) void k_gemv_int(const uint8_t* __restrict__ W, const uint8_t* __restrict__ frag,
                                                   const float* __restrict__ step, const float* __restrict__ bias,
                                                   float* __restrict__ Y, int rows, int nvec, int S, int Sp,
                                                   uint32_t row_bytes, int nvt) {
  using F = IntFmt<T>;
  constexpr int kSeg = kC * F::kSlot;          // bytes of a row's chunk, a multiple of 16
  constexpr int kPieces = kSeg / 16;
  constexpr int kRow = (kSeg / 4) | 1;         // LDS dwords a row: odd, so 32 rows fall on distinct banks
  constexpr int kPart = 32 * kRow;
  static_assert(kSeg % 16 == 0, "whole 16-byte pieces a chunk");
  extern __shared__ uint32_t lds[];            // [2][KS][32][kRow], then [KS - 1][VT][8][64] part sums
  constexpr int nthr = 64 * KS * VT;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int vtl = wave / KS, ks = wave % KS, vt = (int)blockIdx.y * VT + vtl;
  const int ln = lane & 31, g = lane >> 5;
  const int r0 = (int)blockIdx.x * 32, nr = min(32, rows - r0);
  const uint8_t* wb = W + (size_t)r0 * row_bytes;
  float* psum = reinterpret_cast<float*>(lds + 2 * KS * kPart);

  // Geometry of the reduction: blocks of `span` slots (64, or the short row's power of two), a part of
  // span / KS slots a wave, nck chunks a part.
  const int span = min(Sp, 64), part = span / KS, nck = part / kC, lck = 31 - __clz(nck), nblk = (S + span - 1) / span;
  const bool many = Sp > 64;

  // Copies chunk c (block c / nck) of every part into ring half h, all threads, without a branch: rows
  // and chunks are whole 16-byte pieces, pieces past the row repeat its last one (their slots add
  // -0) and rows past the weight its last row.
  constexpr int kMaxPer = (KS * 32 * kPieces + nthr - 1) / nthr;  // pieces a thread
  auto load = [&](int c, uint4 (&q)[kMaxPer]) __attribute__((always_inline)) {
    const int b = c >> lck, i = c - (b << lck);
#pragma unroll
    for (int k = 0; k < kMaxPer; ++k) {
      const int p = min(tid + k * nthr, KS * 32 * kPieces - 1);
      const int pc = p % kPieces, rr = (p / kPieces) % 32, kk = p / (32 * kPieces);
      const uint32_t off = (uint32_t)(b * span + kk * part + i * kC) * F::kSlot + 16u * pc;
      q[k] = ldg16(wb + (size_t)min(rr, nr - 1) * row_bytes + min(off, row_bytes - 16));
    }
  };
  auto store = [&](int h, const uint4 (&q)[kMaxPer]) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < kMaxPer; ++k) {
      const int p = tid + k * nthr;
      if (p >= KS * 32 * kPieces) break;
      const int pc = p % kPieces, rr = (p / kPieces) % 32, kk = p / (32 * kPieces);
      uint32_t* d = lds + (h * KS + kk) * kPart + rr * kRow + 4 * pc;
      d[0] = q[k].x;
      d[1] = q[k].y;
      d[2] = q[k].z;
      d[3] = q[k].w;
    }
  };

  const int nchunk = nblk * nck;
  const uint8_t* fb = frag + (size_t)min(vt, nvt - 1) * S * kFragBytes + 16 * lane;
  const float* sb = step + (size_t)min(vt, nvt - 1) * S * 16 + 8 * g;

  // The activation operands of kC slots, each requested again for the next chunk as soon as it is used.
  i32x4_t A0[kC], A1[kC];
  float4 SA[kC], SB[kC];
  auto act = [&](int c, int u) __attribute__((always_inline)) {
    const int b = c >> lck, i = c - (b << lck);
    const size_t s = (size_t)min(b * span + ks * part + i * kC + u, S - 1);
    A0[u] = *reinterpret_cast<const i32x4_t*>(fb + s * kFragBytes);
    A1[u] = *reinterpret_cast<const i32x4_t*>(fb + s * kFragBytes + 1024);
    SA[u] = *reinterpret_cast<const float4*>(sb + s * 16);
    SB[u] = *reinterpret_cast<const float4*>(sb + s * 16 + 4);
  };

  // The running sums in LDS for Q8_0, whose forms of four and eight K parts spill (0.97 of the time over the range of
  // shapes; the 4- and 5-bit formats, which do not, take 1.02 times theirs).
  constexpr bool kTotLds = T == T_Q8_0 && KS >= 4;
  float tot[8], st[4][8];
#pragma unroll
  for (int k = 0; k < 8; ++k) tot[k] = 0.0f;
  uint4 q[kMaxPer];
  load(0, q);
#pragma unroll
  for (int u = 0; u < kC; ++u) act(0, u);
  store(0, q);
  lds_barrier();
  for (int c = 0; c < nchunk; ++c) {
    const int b = c >> lck, i = c - (b << lck);
    const bool more = c + 1 < nchunk;
    if (more) load(c + 1, q);
    const uint32_t* wl = lds + ((c & 1) * KS + ks) * kPart + ln * kRow;
    const int s0 = b * span + ks * part + i * kC;
    float v[8], v1[8];
    uint32_t c0[4], c1[4];
    float d0, d1;
    F::codes(wl, g, c0, c1, d0, d1);
#pragma unroll
    for (int u = 0; u < kC; ++u) {
      const int s = s0 + u;
      float p[8];
      const i32x16_t zero = {};
      const i32x16_t C0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(
          A0[u], i32x4_t{(int)c0[0], (int)c0[1], (int)c0[2], (int)c0[3]}, zero, 0, 0, 0);
      const i32x16_t C1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(
          A1[u], i32x4_t{(int)c1[0], (int)c1[1], (int)c1[2], (int)c1[3]}, zero, 0, 0, 0);
      const float sx[8] = {SA[u].x, SA[u].y, SA[u].z, SA[u].w, SB[u].x, SB[u].y, SB[u].z, SB[u].w};
      const float e0 = d0, e1 = d1;
      act(min(c + 1, nchunk - 1), u);
      if (u + 1 < kC) F::codes(wl + (u + 1) * (F::kSlot / 4), g, c0, c1, d0, d1);  // read while this slot is folded
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < 8; ++k) {  // vector 4 (k/2) + 2g + k%2: accumulators 2k (qh), 2k + 1 (ql)
        const int t0 = (int)(((uint32_t)C0[2 * k] << 7) + (uint32_t)C0[2 * k + 1]);
        const int t1 = (int)(((uint32_t)C1[2 * k] << 7) + (uint32_t)C1[2 * k + 1]);
        const float f = __builtin_fmaf(e1, (float)t1, e0 * (float)t0);
        p[k] = f * sx[k];
        asm volatile("" : "+v"(p[k]));  // rounded before the tree adds it
        if (s >= S) p[k] = -0.0f;
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        if (u == 0) v[k] = p[k];
        else if (u == 1) v[k] = v[k] + p[k];
        else if (u == 2) v1[k] = p[k];
        else v[k] = v[k] + (v1[k] + p[k]);
      }
    }
    // the part's tree over its chunks, a binary counter of pending left sums (uniform branches)
    auto add = [&](const float (&l)[8]) __attribute__((always_inline)) {
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = l[k] + v[k];
    };
    auto put = [&](float (&l)[8]) __attribute__((always_inline)) {
#pragma unroll
      for (int k = 0; k < 8; ++k) l[k] = v[k];
    };
    if (i & 1) {
      add(st[0]);
      if (i & 2) {
        add(st[1]);
        if (i & 4) {
          add(st[2]);
          if (i & 8) add(st[3]);
          else put(st[3]);
        } else {
          put(st[2]);
        }
      } else {
        put(st[1]);
      }
    } else {
      put(st[0]);
    }
    if (more) store((c + 1) & 1, q);
    if (i + 1 == nck) {  // the block's parts are complete
      if constexpr (KS > 1) {
        float* ps = psum + (vtl * KS + ks) * 512 + lane;
        if (ks > 0)
#pragma unroll
          for (int k = 0; k < 8; ++k) ps[64 * k] = v[k];
        lds_barrier();
        if (ks == 0) {
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            auto pt = [&](int j) { return ps[512 * j + 64 * k]; };  // part j's sum
            v[k] = v[k] + pt(1);
            if constexpr (KS >= 4) v[k] = v[k] + (pt(2) + pt(3));
            if constexpr (KS >= 8) v[k] = v[k] + ((pt(4) + pt(5)) + (pt(6) + pt(7)));
          }
        }
      }
      if constexpr (kTotLds) {
        float* ps = psum + vtl * KS * 512 + lane;  // part 0's place: it is not stored
        if (ks == 0)
#pragma unroll
          for (int k = 0; k < 8; ++k) ps[64 * k] = many ? (b > 0 ? ps[64 * k] : 0.0f) + v[k] : v[k];
      } else if (many) {
#pragma unroll
        for (int k = 0; k < 8; ++k) tot[k] += v[k];
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) tot[k] = v[k];
      }
    }
    lds_barrier();
  }
  const int r = r0 + ln;
  if (ks != 0 || vt >= nvt || r >= rows) return;
  const float bb = bias ? bias[r] : 0.0f;
  if constexpr (kTotLds)
#pragma unroll
    for (int k = 0; k < 8; ++k) tot[k] = psum[vtl * KS * 512 + 64 * k + lane];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int vv = 16 * vt + 4 * (k >> 1) + 2 * g + (k & 1);
    if (vv < nvec) Y[(size_t)vv * rows + r] = bias ? tot[k] + bb : tot[k];
  }
  // A padded row whose last scales are not finite.  (Read again and stored over the sums, as the loop has no
  // register to spare: with a NaN carried through it, or added to the sums, Q8_0 11008 x 4096 at 8 took 30.8 us, not 27.5.)
  if (S % span != 0) {
    const float pad = scales_zero<T>(wb + (size_t)ln * row_bytes + row_bytes - F::kSlot);
    if (pad != pad)
      for (int k = 0; k < 8; ++k) {
        const int vv = 16 * vt + 4 * (k >> 1) + 2 * g + (k & 1);
        if (vv < nvec) Y[(size_t)vv * rows + r] = pad;
      }
  }
}

template <uint32_t T, int KS, int VT>
bool launch_vt(const uint8_t* w, const uint8_t* frag, const float* step, const float* bias, float* Y, int rows,
               int nvec, int S, int Sp, size_t row_bytes, hipStream_t s) {
  constexpr int kRow = (kC * IntFmt<T>::kSlot / 4) | 1;
  auto kern = &k_gemv_int<T, KS, VT>;
  const int nvt = (nvec + 15) / 16;
  const size_t lds = (size_t)2 * KS * 32 * kRow * 4 + (KS > 1 ? (size_t)VT * KS * 512 * 4 : 0);
  static LdsLimit lim;
  if (!lds_ready(reinterpret_cast<const void*>(kern), lim, lds)) return false;
  kern<<<dim3((unsigned)((rows + 31) / 32), (unsigned)((nvt + VT - 1) / VT)), (unsigned)(64 * VT * KS), lds, s>>>(
      w, frag, step, bias, Y, rows, nvec, S, Sp, (uint32_t)row_bytes, nvt);
  return true;
}
// Tiles of vectors a workgroup: four where the K parts are not split, two at two parts, else one.
template <uint32_t T, int KS>
bool launch_ks(const uint8_t* w, const uint8_t* frag, const float* step, const float* bias, float* Y, int rows,
               int nvec, int S, int Sp, size_t row_bytes, hipStream_t s) {
  constexpr int VT = KS == 1 ? 4 : KS == 2 ? 2 : 1;
  return launch_vt<T, KS, VT>(w, frag, step, bias, Y, rows, nvec, S, Sp, row_bytes, s);
}

template <uint32_t T>
bool launch_int(const void* w, const float* X, float* Y, const float* bias, int nvec, int rows, int cols,
                size_t row_bytes, void* ws, hipStream_t s) {
  Geo geo{};
  if (!geometry<T>(cols, row_bytes, geo)) return false;
  const int S = geo.S;
  const int step_v = int_chunk_vectors(nvec, S);
  const auto* wb = static_cast<const uint8_t*>(w);
  for (int v0 = 0; v0 < nvec; v0 += step_v) {
    const int nv = std::min(step_v, nvec - v0), nvt = (nv + 15) / 16;
    auto* frag = static_cast<uint8_t*>(ws);
    auto* step = reinterpret_cast<float*>(frag + (size_t)nvt * S * kFragBytes);
    const int ntask = nvt * 16 * S * 8;
    k_int_conv<<<(unsigned)((ntask + 255) / 256), 256, 0, s>>>(X + (size_t)v0 * cols, nv, cols, S, frag, step, ntask);
    // K parts of at least a chunk: as many as it takes to put about one wave on each SIMD.  Between, four
    // (Q4_0 4096 x 4096 at 64 vectors: 18.6 us against 24.9 on two), but two for Q8_0 batches, whose four
    // parts a lone tile of vectors spill (11008 x 4096 at 17: 29.8 against 40.7).
    const int64_t waves = (int64_t)((rows + 31) / 32) * nvt;
    float* Yv = Y + (size_t)v0 * rows;
    const int ks = std::min(std::min(geo.Sp, 64) / kC, waves >= 1024                                  ? 1
                                                       : T == T_Q8_0 && nvt >= 2 && waves >= 512 ? 2
                                                       : waves >= 256                             ? 4
                                                                                                   : 8);
    const bool ok = ks == 1   ? launch_ks<T, 1>(wb, frag, step, bias, Yv, rows, nv, S, geo.Sp, row_bytes, s)
                    : ks < 4 ? launch_ks<T, 2>(wb, frag, step, bias, Yv, rows, nv, S, geo.Sp, row_bytes, s)
                    : ks < 8 ? launch_ks<T, 4>(wb, frag, step, bias, Yv, rows, nv, S, geo.Sp, row_bytes, s)
                             : launch_ks<T, 8>(wb, frag, step, bias, Yv, rows, nv, S, geo.Sp, row_bytes, s);
    if (!ok) return false;
  }
  return true;
}

template <uint32_t T>
size_t int_need(int nvec, int cols, size_t row_bytes) {
  Geo geo{};
  if (!geometry<T>(cols, row_bytes, geo)) return 0;
  return int_ws_bytes(int_chunk_vectors(nvec, geo.S), geo.S);
}

}  // namespace

// Workspace bytes of the batched form for a call, 0 where it does not take the call (too few vectors, or a
// shape the one-vector kernel, whose per-slot arithmetic is the contract, does not take).
size_t gemv_int_ws_bytes(uint32_t t, int nvec, int rows, int cols, size_t row_bytes) {
  if (!int_batch(t, nvec, rows, cols)) return 0;
  switch (t) {
    case T_Q8_0: return int_need<T_Q8_0>(nvec, cols, row_bytes);
    case T_Q4_0: return int_need<T_Q4_0>(nvec, cols, row_bytes);
    case T_Q5_0: return int_need<T_Q5_0>(nvec, cols, row_bytes);
    default: return 0;
  }
}

// out = W . X (+ bias) on the batched form; ws holds gemv_int_ws_bytes.  Returns false, having launched
// nothing, when a launch cannot be configured.
bool launch_gemv_int(uint32_t t, const void* w, const float* X, float* Y, const float* bias, int nvec, int rows,
                     int cols, size_t row_bytes, void* ws, hipStream_t s) {
  switch (t) {
    case T_Q8_0: return launch_int<T_Q8_0>(w, X, Y, bias, nvec, rows, cols, row_bytes, ws, s);
    case T_Q4_0: return launch_int<T_Q4_0>(w, X, Y, bias, nvec, rows, cols, row_bytes, ws, s);
    case T_Q5_0: return launch_int<T_Q5_0>(w, X, Y, bias, nvec, rows, cols, row_bytes, ws, s);
    default: return false;
  }
}

}  // namespace qvx
