// qvx_gemv_group.hip -- grouped one-vector GEMV on the integer VALU kernel (gfx950).
//
// The consecutive projections of one activation vector (the decoder's q / k / v and gate / up,
// runtime/src/text_model.cpp:147-164) in one launch, for members of one Q8_0 / Q4_0 / Q5_0 / Q5_K / Q6_K type:
// each is a short launch whose ramp, activation conversion and drain cost as much as its streaming, and a
// group pays them once.  The members' rows are dealt out as if stacked: every workgroup takes rows of one
// member only, as many rows a lane group for each, so one pass of workgroups over the chip holds the
// whole group.  A row's arithmetic does not depend on the workgroup that computes it (gemv_valu_body), so
// every output is bit-identical to its own qvx_qmatmul.  Measured on MI355X, graph-replayed over distinct
// weights: a Q8_0 layer (q, k, v 4096 x 4096, gate, up 11008 x 4096) in 3 launches instead of 6, the step of four
// layers and a head 252 -> 234 us.
#include "qvx_gemv_valu.hpp"

namespace qvx {

namespace {

constexpr int kMembers = 4;

struct VMember {
  const uint8_t* w;
  float* y;
  int rows, nwg;
  Geo geo;
};
struct VGroup {
  VMember m[kMembers];
  int n;
};

template <uint32_t T, int RMAX, int TPT, bool CH>
__global__ __launch_bounds__((gemv_threads<T, 1>())) void k_gemv_vgroup(const float* __restrict__ X, int cols, VGroup a) {
  constexpr int PF = prefetch_rows<T, 1>() < RMAX ? prefetch_rows<T, 1>() : RMAX;
  int b = blockIdx.x, i = 0;
  while (i + 1 < a.n && b >= a.m[i].nwg) b -= a.m[i++].nwg;
  const VMember& m = a.m[i];
  gemv_valu_body<T, 1, RMAX, TPT, PF, CH, false>(m.w, X, m.y, m.rows, cols, m.geo, nullptr, 0.0f, b, threadIdx.x,
                                                 threadIdx.y);
}

// The group's workgroups: the fewest rows a lane group that fit one pass over the chip.  Returns them (0: not
// a group this launch takes), per_group = the most rows a lane group has.
template <uint32_t T>
int deal(const GemvMember* m, int n, int cols, VGroup& a, int& per_group) {
  if (n < 2 || n > kMembers) return 0;
  Geo geo{};
  if (!geometry<T>(cols, m[0].row_bytes, geo)) return 0;
  const int threads = geo.Sp * geo.G, tasks = geo.S * 2 * Lane<T>::kR;
  if (tasks > 2 * threads) return 0;
  const int64_t most = (int64_t)kCUs * (threads >= 1024 ? 1 : 1024 / threads);
  int p = 1, nwg = 0;
  for (;; ++p) {
    nwg = 0;
    for (int i = 0; i < n; ++i) nwg += (int)std::min<int64_t>(((int64_t)m[i].rows + (int64_t)p * geo.G - 1) / ((int64_t)p * geo.G), 1 << 20);
    if (nwg <= std::max<int64_t>(most, n)) break;
  }
  per_group = 0;
  a.n = n;
  nwg = 0;
  for (int i = 0; i < n; ++i) {
    VMember& v = a.m[i];
    v.w = static_cast<const uint8_t*>(m[i].w);
    v.y = m[i].y;
    v.rows = m[i].rows;
    v.nwg = (int)(((int64_t)m[i].rows + (int64_t)p * geo.G - 1) / ((int64_t)p * geo.G));
    v.geo = geo;
    v.geo.base = m[i].rows / v.nwg;
    v.geo.rem = m[i].rows % v.nwg;
    per_group = std::max(per_group, (v.geo.base + (v.geo.rem ? 1 : 0) + geo.G - 1) / geo.G);
    nwg += v.nwg;
  }
  return nwg;
}

template <uint32_t T, int RMAX, int TPT, bool CH>
bool launch_one(const float* X, int cols, const VGroup& a, int nwg, hipStream_t s) {
  auto kern = &k_gemv_vgroup<T, RMAX, TPT, CH>;
  const Geo& geo = a.m[0].geo;
  const size_t lds = gemv_lds_bytes<T>(1, geo.S);
  static LdsLimit lim;
  if (!lds_ready(reinterpret_cast<const void*>(kern), lim, lds)) return false;
  kern<<<(unsigned)nwg, dim3((unsigned)geo.Sp, (unsigned)geo.G), lds, s>>>(X, cols, a);
  return true;
}

template <uint32_t T>
bool launch_group(const GemvMember* m, int n, const float* X, int cols, hipStream_t s, bool dry) {
  VGroup a{};
  int per = 0;
  const int nwg = deal<T>(m, n, cols, a, per);
  if (nwg == 0 || dry) return nwg != 0;
  // rows a lane group: 1, 2 or 4 at once, more in chunks of four
  const auto go = [&](auto tpt) {
    constexpr int TPT = decltype(tpt)::value;
    return per <= 1   ? launch_one<T, 1, TPT, false>(X, cols, a, nwg, s)
           : per <= 2 ? launch_one<T, 2, TPT, false>(X, cols, a, nwg, s)
           : per <= 4 ? launch_one<T, 4, TPT, false>(X, cols, a, nwg, s)
                      : launch_one<T, 4, TPT, true>(X, cols, a, nwg, s);
  };
  const Geo& geo = a.m[0].geo;
  return geo.S * 2 * Lane<T>::kR <= geo.Sp * geo.G ? go(std::integral_constant<int, 1>{})
                                                   : go(std::integral_constant<int, 2>{});
}

}  // namespace

// One launch for 2..4 members of one type, 16-byte-aligned weights, x and row pitches (as the standalone
// VALU kernel takes them).  Returns false, having launched nothing, for any other group; dry: only says
// whether it would take the group.
bool launch_gemv_vgroup(const GemvMember* m, int n, const float* X, int cols, hipStream_t s, bool dry) {
  if (n < 2) return false;
  for (int i = 1; i < n; ++i)
    if (m[i].type != m[0].type) return false;
  switch (m[0].type) {
    case T_Q8_0: return launch_group<T_Q8_0>(m, n, X, cols, s, dry);
    case T_Q4_0: return launch_group<T_Q4_0>(m, n, X, cols, s, dry);
    case T_Q5_0: return launch_group<T_Q5_0>(m, n, X, cols, s, dry);
    case T_Q5_K: return launch_group<T_Q5_K>(m, n, X, cols, s, dry);
    case T_Q6_K: return launch_group<T_Q6_K>(m, n, X, cols, s, dry);
    default: return false;
  }
}

}  // namespace qvx
