// Several sweeps of one rank-2 stencil in a single pass over memory (a loop that applies a
// stencil to its own result, Interpreter.hs:222-229 around :637-649).
//
// One sweep moves the array in and out of HBM and is bound by that (8192 x 8192 Float32: 88-90
// us for 512 MiB); its arithmetic is a tenth of it.  Here a wave owns a strip of 64 * V columns
// and marches down the rows with T sweeps in flight: sweep t of row y is computed as soon as
// sweep t - 1 of row y + HY is, from the 2 * HY + 1 rows of sweep t - 1 that the wave keeps in
// registers.  Rows enter from memory once and leave after T sweeps; nothing goes through LDS and
// no wave waits for another.  The left and right neighbours come from the next lanes by
// wave shifts.  What a wave lacks beyond its strip it recomputes: a strip gives 64 * V - 2 * T * HX
// (rounded to V) columns, a chunk of rows starts and ends T * HY rows early and late.
//
// Measured (Jacobi, 8192 x 8192): Float32 90 us a sweep with a launch for each, 15.6 us in passes of 8.  A pass of
// 8 takes 118 - 125 us: its 61 million vector instructions are issued in 92 % of the busy cycles.  A pass of 4 has half as many
// and takes 118 - 123 us, for which 572 MiB (operand and result 512) come and go at 5.1 TB/s, so 8 it is where registers
// allow (146 of them, 3 waves a SIMD; halos of 2 take 4).  Float64 30 us a sweep.  All waves
// of a launch are resident at once: with 3072 of them 15.7 us a sweep, 2048 16.0, 1024 22.3, 4096, a second generation, 18.0.
//
// Boundary conditions hold in every sweep: a tap outside the array is replaced from the same
// sweep's rows and columns (clamp, mirror), by the constant, or, for wrap, by continuing the array
// periodically, which is the same numbers computed twice.  Lanes whose position lies outside the
// array, and the margins of a strip, compute values nobody uses, on taps that no element has (zeros
// among them): the code generator takes this path only for functions of the taps that are defined
// for all of them, which a division by a tap is not.

// results of one lane and row: S::V values of type S::E, with HX neighbours on either side
#define ACC_SW_P (2 * Spec::HY + 1)
#define ACC_SW_E (Spec::V + 2 * Spec::HX)

struct SweepParams {
  i64 h, w;       // extents
  i64 strips;     // strips of columns
  i64 items;      // strips * chunks of rows
  i64 rows;       // rows per chunk
};

template <int N> struct AccConst { static constexpr int value = N; };

struct SweepRow { Spec::E e[ACC_SW_E]; };

// v with its neighbours; XE: the strip reaches beyond the first or last column
template <bool XE> ACC_DEV SweepRow acc_sweep_expand(const Spec::Env& env, const Spec::E (&v)[Spec::V], int gx, int w) {
  typedef Spec S;
  const int V = S::V, HX = S::HX;
  SweepRow r;
#pragma unroll
  for (int k = 0; k < V; ++k) r.e[HX + k] = v[k];
#pragma unroll
  for (int j = 1; j <= HX; ++j) {
    r.e[HX - j] = acc_dpp<0x138, 0xf>(v[V - j]);          // from the lane to the left
    r.e[HX + V - 1 + j] = acc_dpp<0x130, 0xf>(v[j - 1]);  // from the lane to the right
  }
  if constexpr (XE && S::BOUNDARY != 2) {
    // a lane starts at column 0 or at a multiple of V from it, so only the last column can lie
    // inside a lane
    if constexpr (S::BOUNDARY == 0) {
#pragma unroll
      for (int i = -1; i >= -HX; --i) r.e[HX + i] = gx + i < 0 ? r.e[HX + i + 1] : r.e[HX + i];
#pragma unroll
      for (int i = 1; i < V + HX; ++i) r.e[HX + i] = gx + i >= w ? r.e[HX + i - 1] : r.e[HX + i];
    } else if constexpr (S::BOUNDARY == 1) {
#pragma unroll
      for (int j = 1; j <= HX; ++j) r.e[HX - j] = gx == 0 ? r.e[HX + j] : r.e[HX - j];
#pragma unroll
      for (int i = 1; i < V + HX; ++i)
#pragma unroll
        for (int j = 1; j <= HX; ++j)
          if (i - 2 * j >= -HX) r.e[HX + i] = gx + i == w - 1 + j ? r.e[HX + i - 2 * j] : r.e[HX + i];
    } else {
      const S::E c = S::outside(env);
#pragma unroll
      for (int i = -HX; i < V + HX; ++i) r.e[HX + i] = (gx + i < 0 || gx + i >= w) ? c : r.e[HX + i];
    }
  }
  return r;
}

// the window around row y of h; YE: the window may reach beyond the first or last row
template <bool YE> ACC_DEV void acc_sweep_window(const Spec::Env& env, SweepRow (&win)[ACC_SW_P], int y, int h) {
  typedef Spec S;
  const int HY = S::HY;
  if constexpr (YE && S::BOUNDARY != 2) {
#pragma unroll
    for (int e = 0; e < ACC_SW_E; ++e) {
      if constexpr (S::BOUNDARY == 0) {
#pragma unroll
        for (int i = 1; i <= HY; ++i) win[HY - i].e[e] = y - i < 0 ? win[HY - i + 1].e[e] : win[HY - i].e[e];
#pragma unroll
        for (int i = 1; i <= HY; ++i) win[HY + i].e[e] = y + i >= h ? win[HY + i - 1].e[e] : win[HY + i].e[e];
      } else if constexpr (S::BOUNDARY == 1) {
        // row -k is row k; only rows inside are copied, and they are never copied onto
        S::E o[ACC_SW_P];
#pragma unroll
        for (int q = 0; q < ACC_SW_P; ++q) o[q] = win[q].e[e];
#pragma unroll
        for (int i = 1; i <= HY; ++i)
#pragma unroll
          for (int k = 1; k <= HY; ++k) {
            if (i >= k) {  // the focus lies k rows inside of the reflection: row -i .. is i - k below 0
              const int up = -i + 2 * k, dn = i - 2 * k;  // y - i = -k  /  y + i = h - 1 + k
              win[HY - i].e[e] = y - i == -k ? o[HY + up] : win[HY - i].e[e];
              win[HY + i].e[e] = y + i == h - 1 + k ? o[HY + dn] : win[HY + i].e[e];
            }
          }
      } else {
        const S::E c = S::outside(env);
#pragma unroll
        for (int i = 1; i <= HY; ++i) {
          win[HY - i].e[e] = y - i < 0 ? c : win[HY - i].e[e];
          win[HY + i].e[e] = y + i >= h ? c : win[HY + i].e[e];
        }
      }
    }
  }
}

template <int T> struct SweepGeo {
  static constexpr int HXT = (T * Spec::HX + Spec::V - 1) / Spec::V * Spec::V;  // margin of a strip
  static constexpr int U = ACC_WAVE * Spec::V - 2 * HXT;                        // columns a strip gives
};

template <int T, bool XE> ACC_DEV void acc_sweep_strip(const Spec::Env& env, const Spec::Out& out, const SweepParams& p,
                                                       int strip, int y0, int y1) {
  typedef Spec S;
  typedef S::E E;
  const int V = S::V, HY = S::HY, NP = ACC_SW_P;
  const int h = (int)p.h, w = (int)p.w;
  const int gx = strip * SweepGeo<T>::U - SweepGeo<T>::HXT + acc_lane() * V;
  const E* __restrict__ src = S::source(env);
  E* __restrict__ dst = S::target(out);
  const int lo = strip * SweepGeo<T>::U;  // the strip's own columns [lo, hi)
  const int hi = lo + SweepGeo<T>::U < w ? lo + SweepGeo<T>::U : w;
  int cols[S::V];
  if constexpr (XE) {
#pragma unroll
    for (int k = 0; k < V; ++k) {
      int c = gx + k;
      if constexpr (S::BOUNDARY == 2) {
        // rows of a periodic array: a strip reaches T * HX + V columns out at most, w is longer
        if (c < 0) c += w;
        if (c >= w) c -= w;
      }
      cols[k] = c < 0 ? 0 : (c >= w ? w - 1 : c);
    }
  }
  auto load = [&](int y, E (&v)[S::V]) {
    if constexpr (S::BOUNDARY == 2) {
      if (y < 0) y += h;
      if (y >= h) y -= h;
    }
    y = y < 0 ? 0 : (y >= h ? h - 1 : y);
    const E* row = src + (i64)y * w;
    if constexpr (XE) {
#pragma unroll
      for (int k = 0; k < V; ++k) v[k] = row[cols[k]];
    } else {
      const acc_run<E, S::V> r = *(const acc_run<E, S::V>*)(row + gx);
#pragma unroll
      for (int k = 0; k < V; ++k) v[k] = r.e[k];
    }
  };

  const int ys = y0 - T * HY;       // first row that enters
  const int ye = y1 + T * HY;       // rows [ys, ye) enter
  E pre[ACC_SW_P][S::V];            // the next rows, on their way
#pragma unroll
  for (int u = 0; u < NP; ++u) load(ys + u, pre[u]);
  SweepRow win[T][ACC_SW_P];        // win[t][u]: the newest rows of sweep t; row r lies in slot (r - ys + t * HY) % NP
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int u = 0; u < NP; ++u)
#pragma unroll
      for (int e = 0; e < ACC_SW_E; ++e) win[t][u].e[e] = (E)0;

  auto step = [&](auto ye_, auto u_, int yin) __attribute__((always_inline)) {
    constexpr bool YE = decltype(ye_)::value != 0;
    constexpr int u = decltype(u_)::value;
    win[0][u] = acc_sweep_expand<XE>(env, pre[u], gx, w);
    load(yin + NP, pre[u]);
#pragma unroll
    for (int t = 1; t <= T; ++t) {
      const int y = yin - t * HY;
      SweepRow wv[ACC_SW_P];
#pragma unroll
      for (int q = 0; q < NP; ++q) wv[q] = win[t - 1][(u + 1 + q) % NP];
      acc_sweep_window<YE>(env, wv, y, h);
      E r[S::V];
#pragma unroll
      for (int k = 0; k < V; ++k) r[k] = S::apply_win(env, wv, k).c0;
      if (t < T) {
        win[t < T ? t : 0][u] = acc_sweep_expand<XE>(env, r, gx, w);
      } else if (y >= y0 && y < y1) {
        E* row = dst + (i64)y * w;
        if constexpr (XE) {
#pragma unroll
          for (int k = 0; k < V; ++k)
            if (gx + k >= lo && gx + k < hi) row[gx + k] = r[k];
        } else if (gx >= lo && gx < hi) {
          acc_run<E, S::V> o;
#pragma unroll
          for (int k = 0; k < V; ++k) o.e[k] = r[k];
          *(acc_run<E, S::V>*)(row + gx) = o;
        }
      }
    }
  };
  for (int y = ys; y < ye; y += NP) {
    // a sweep of these steps computes rows y - T * HY .. y + NP - 1 - HY, and looks HY rows further
    const bool edge = S::BOUNDARY != 2 && (y - (T + 1) * HY < 0 || y + NP - 1 >= h);
    if (edge) {
      step(AccConst<1>(), AccConst<0>(), y);
      if constexpr (ACC_SW_P > 1) {
        step(AccConst<1>(), AccConst<1>(), y + 1);
        step(AccConst<1>(), AccConst<2>(), y + 2);
      }
      if constexpr (ACC_SW_P > 3) {
        step(AccConst<1>(), AccConst<3>(), y + 3);
        step(AccConst<1>(), AccConst<4>(), y + 4);
      }
    } else {
      step(AccConst<0>(), AccConst<0>(), y);
      if constexpr (ACC_SW_P > 1) {
        step(AccConst<0>(), AccConst<1>(), y + 1);
        step(AccConst<0>(), AccConst<2>(), y + 2);
      }
      if constexpr (ACC_SW_P > 3) {
        step(AccConst<0>(), AccConst<3>(), y + 3);
        step(AccConst<0>(), AccConst<4>(), y + 4);
      }
    }
  }
}

template <int T> ACC_DEV void acc_sweep(const Spec::Env& env, const Spec::Out& out, const SweepParams& p) {
  typedef Spec S;
  // neighbouring strips share their margins: neighbours run on the same XCD
  const i64 b = acc_xcd_contiguous((i64)blockIdx.x, (i64)gridDim.x);
  const i64 item = b * ACC_WAVES + __builtin_amdgcn_readfirstlane(acc_wave());
  if (item >= p.items) return;
  const int chunk = (int)(item / p.strips), strip = (int)(item - chunk * p.strips);
  const int y0 = chunk * (int)p.rows;
  const int y1 = y0 + p.rows < p.h ? y0 + (int)p.rows : (int)p.h;
  const int x0 = strip * SweepGeo<T>::U - SweepGeo<T>::HXT;
  if (x0 >= 0 && x0 + ACC_WAVE * S::V <= p.w) acc_sweep_strip<T, false>(env, out, p, strip, y0, y1);
  else acc_sweep_strip<T, true>(env, out, p, strip, y0, y1);
}

#if ACC_SW_MAX >= 8
extern "C" __global__ void __launch_bounds__(ACC_BLOCK) acc_sweeps8(Spec::Env env, Spec::Out out, SweepParams p) {
  acc_sweep<8>(env, out, p);
}
#endif
extern "C" __global__ void __launch_bounds__(ACC_BLOCK) acc_sweeps4(Spec::Env env, Spec::Out out, SweepParams p) {
  acc_sweep<4>(env, out, p);
}
extern "C" __global__ void __launch_bounds__(ACC_BLOCK) acc_sweeps2(Spec::Env env, Spec::Out out, SweepParams p) {
  acc_sweep<2>(env, out, p);
}
