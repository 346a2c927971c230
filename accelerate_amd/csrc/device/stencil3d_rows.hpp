// Rank-3 stencils of many taps (stencilOp, Interpreter.hs:637-649), from registers.
//
// Through LDS (stencil3d.hpp) every tap of every result is a read of its own, and its product
// with a weight is computed anew: smoothing with 27 taps, 401 x 387 x 393 Float32, keeps the vector units busy for 91 % of 194 us, where the traffic needs
// 76, and 7 taps take 141.  Here a wave owns a strip of 64 * V columns and a
// band of R rows and marches through the planes with the window of three planes by R + 2 * HY rows in
// registers: a row is loaded V values a lane, its left and right neighbours come from the
// next lanes by wave shifts, and what two results share (a loaded value, a product) is computed once, within
// the band and within the three planes one turn of the loop covers.  162 us (7 taps 174), 24 instead of 37 on 200^3,
// 323 instead of 332 on 512^3: bound by loads, of which the bands' border rows come again for every neighbour, so
// it wins most where they come from the cache (the host chooses, see there).  (A wave that marches down the rows of one plane
// with the planes around it loads everything three times: 198 - 317 us.)
//
// Outside the array a tap is replaced as `bounded` says (Interpreter.hs:797-839): columns and rows
// in the registers, planes by the index of the plane that is loaded, or the constant.  As in
// the kernel for several sweeps, margins compute values nobody uses on taps that no element has, so the
// function must be defined for all of them.

#define ACC_SR_ROWS (Spec::R + 2 * Spec::HY)
#define ACC_SR_PZ (2 * Spec::HZ + 1)
#define ACC_SR_E (Spec::V + 2 * Spec::HX)

struct Stencil3dRowsParams {
  i64 d, h, w;     // extents
  i64 strips;      // strips of columns
  i64 bands;       // bands of S::R rows, a whole number of workgroups of them
  i64 chunks;      // chunks of planes
  i64 planes;      // planes per chunk
};

struct StencilRow { Spec::E e[ACC_SR_E]; };
struct StencilWin { StencilRow r[ACC_SR_PZ][ACC_SR_ROWS]; };  // the planes and rows around a step's results

// columns a strip starts before its first result: a whole number of lanes, so that column 0 is a lane's first
static constexpr int kMargin = (Spec::HX + Spec::V - 1) / Spec::V * Spec::V;
static constexpr int kCols = ACC_WAVE * Spec::V - 2 * kMargin;

template <bool XE> ACC_DEV StencilRow acc_row_expand(const Spec::Env& env, const Spec::E (&v)[Spec::V], int gx, int w) {
  typedef Spec S;
  const int V = S::V, HX = S::HX;
  StencilRow r;
#pragma unroll
  for (int k = 0; k < V; ++k) r.e[HX + k] = v[k];
#pragma unroll
  for (int j = 1; j <= HX; ++j) {
    r.e[HX - j] = acc_dpp<0x138, 0xf>(v[V - j]);
    r.e[HX + V - 1 + j] = acc_dpp<0x130, 0xf>(v[j - 1]);
  }
  if constexpr (XE && S::BOUNDARY == 0) {
#pragma unroll
    for (int i = -1; i >= -HX; --i) r.e[HX + i] = gx + i < 0 ? r.e[HX + i + 1] : r.e[HX + i];
#pragma unroll
    for (int i = 1; i < V + HX; ++i) r.e[HX + i] = gx + i >= w ? r.e[HX + i - 1] : r.e[HX + i];
  } else if constexpr (XE && S::BOUNDARY == 1) {
#pragma unroll
    for (int j = 1; j <= HX; ++j) r.e[HX - j] = gx == 0 ? r.e[HX + j] : r.e[HX - j];
#pragma unroll
    for (int i = 1; i < V + HX; ++i)
#pragma unroll
      for (int j = 1; j <= HX; ++j)
        if (i - 2 * j >= -HX) r.e[HX + i] = gx + i == w - 1 + j ? r.e[HX + i - 2 * j] : r.e[HX + i];
  } else if constexpr (XE && S::BOUNDARY == 3) {
    const S::E c = S::outside(env);
#pragma unroll
    for (int i = -HX; i < V + HX; ++i) r.e[HX + i] = (gx + i < 0 || gx + i >= w) ? c : r.e[HX + i];
  }
  return r;
}

// index j of an extent of n as the boundary condition reads it (constant: any index inside); j lies at
// most one extent outside
ACC_DEV int acc_bounded(int j, int n) {
  if constexpr (Spec::BOUNDARY == 1) {
    if (j < 0) j = -j;
    if (j >= n) j = n - (j - n + 2);
  } else if constexpr (Spec::BOUNDARY == 2) {
    if (j < 0) j += n;
    if (j >= n) j -= n;
  }
  return j < 0 ? 0 : (j >= n ? n - 1 : j);
}

template <bool XE> ACC_DEV void acc_rows_strip(const Spec::Env& env, const Spec::Out& out, const Stencil3dRowsParams& p,
                                               int strip, int y0, int z0, int z1) {
  typedef Spec S;
  typedef S::E E;
  const int V = S::V, HY = S::HY, HZ = S::HZ, PZ = ACC_SR_PZ, NR = ACC_SR_ROWS;
  const int d = (int)p.d, h = (int)p.h, w = (int)p.w;
  const int lo = strip * kCols, hi = lo + kCols < w ? lo + kCols : w;  // the strip's own columns
  const int gx = lo - kMargin + acc_lane() * V;
  int cols[S::V];
  if constexpr (XE) {
#pragma unroll
    for (int k = 0; k < V; ++k) {
      int c = gx + k;
      if constexpr (S::BOUNDARY == 2) {
        if (c < 0) c += w;
        if (c >= w) c -= w;
      }
      cols[k] = c < 0 ? 0 : (c >= w ? w - 1 : c);
    }
  }
  i64 rowAt[ACC_SR_ROWS];   // rows y0 - HY .. y0 + R + HY - 1 of a plane, as the boundary condition reads them
  bool rowOut[ACC_SR_ROWS];  // constant boundary: the whole row is the constant
#pragma unroll
  for (int j = 0; j < NR; ++j) {
    rowAt[j] = (i64)acc_bounded(y0 - HY + j, h) * w;
    rowOut[j] = S::BOUNDARY == 3 && (y0 - HY + j < 0 || y0 - HY + j >= h);
  }
  auto load = [&](int z, E (&v)[ACC_SR_ROWS][S::V]) __attribute__((always_inline)) {
    const E* plane = S::source(env) + (i64)acc_bounded(z, d) * h * w;
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      const E* row = plane + rowAt[j];
      if constexpr (XE) {
#pragma unroll
        for (int k = 0; k < V; ++k) v[j][k] = row[cols[k]];
      } else {
        const acc_run<E, S::V> r = *(const acc_run<E, S::V>*)(row + gx);
#pragma unroll
        for (int k = 0; k < V; ++k) v[j][k] = r.e[k];
      }
    }
  };
  StencilRow win[ACC_SR_PZ][ACC_SR_ROWS];  // plane z in slot (z - (z0 - HZ)) % PZ
  E pre[ACC_SR_ROWS][S::V];                // the next plane's rows, on their way
  load(z0 - HZ, pre);
  auto enter = [&](auto u_, int z) __attribute__((always_inline)) {
    constexpr int u = decltype(u_)::value;
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      win[u][j] = acc_row_expand<XE>(env, pre[j], gx, w);
      if constexpr (S::BOUNDARY == 3) {
        if (rowOut[j] || z < 0 || z >= d) {
          const E c = S::outside(env);
#pragma unroll
          for (int e = 0; e < ACC_SR_E; ++e) win[u][j].e[e] = c;
        }
      }
    }
    load(z + 1, pre);
  };
  auto step = [&](auto u_, int zin) __attribute__((always_inline)) {
    constexpr int u = decltype(u_)::value;
    enter(u_, zin);
    const int z = zin - HZ;
    StencilWin wv;
#pragma unroll
    for (int q = 0; q < PZ; ++q)
#pragma unroll
      for (int j = 0; j < NR; ++j) wv.r[q][j] = win[(u + 1 + q) % PZ][j];
#pragma unroll
    for (int b = 0; b < S::R; ++b) {
      S::Elt r[S::V];
#pragma unroll
      for (int k = 0; k < V; ++k) r[k] = S::apply_win(env, wv, b, k);
      if (z < z1 && y0 + b < h) {
        const i64 at = ((i64)z * h + y0 + b) * w + gx;
        if (gx >= lo && gx + V <= hi) {
          S::store_run(out, at, r);
        } else if (XE && gx >= lo) {
#pragma unroll
          for (int k = 0; k < V; ++k)
            if (gx + k < hi) S::store(out, at + k, r[k]);
        }
      }
    }
  };
  static_assert(ACC_SR_PZ == 3, "the loop below steps through three planes");
  enter(AccConst<0>(), z0 - 1);
  enter(AccConst<1>(), z0);
  for (int z = z0 + 1; z < z1 + 1; z += 3) {
    step(AccConst<2>(), z);
    step(AccConst<0>(), z + 1);
    step(AccConst<1>(), z + 2);
  }
}

extern "C" __global__ void __launch_bounds__(ACC_BLOCK)
acc_stencil3d_rows(Spec::Env env, Spec::Out out, Stencil3dRowsParams p) {
  typedef Spec S;
  const i64 b = acc_xcd_contiguous((i64)blockIdx.x, (i64)gridDim.x);
  // chunks of planes outermost, then strips, bands innermost: a workgroup's waves take neighbouring bands
  const i64 groups = p.bands / ACC_WAVES, per = groups * p.strips;
  const int chunk = (int)(b / per);
  const i64 rest = b - chunk * per;
  const int strip = (int)(rest / groups);
  const i64 y0 = ((rest - strip * groups) * ACC_WAVES + __builtin_amdgcn_readfirstlane(acc_wave())) * S::R;
  if (y0 >= p.h) return;
  const i64 z0 = chunk * p.planes, z1 = z0 + p.planes < p.d ? z0 + p.planes : p.d;
  const i64 x0 = (i64)strip * kCols - kMargin;
  if (x0 >= 0 && x0 + ACC_WAVE * S::V <= p.w) acc_rows_strip<false>(env, out, p, strip, (int)y0, (int)z0, (int)z1);
  else acc_rows_strip<true>(env, out, p, strip, (int)y0, (int)z0, (int)z1);
}
