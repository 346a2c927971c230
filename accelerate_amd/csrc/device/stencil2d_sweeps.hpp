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
// Measured (Jacobi, 8192 x 8192): Float32 90 us a sweep with a launch for each, 16.3 us in passes of 8 that fetched the neighbours
// when a row was made, 12.8 us in passes of 10 that fetch them late: 17 vector instructions a sweep and row of which 16 are the
// function's, 63 million a pass of 126 us at 2.3 GHz, 81 % of what can be issued.  10 is what 3 waves a SIMD hold
// (154 registers; us for 100 sweeps, plain stores: passes of 8 1626, 10 1315, 12 1450, 16 1415, the last two with 2 waves; 12 held
// to 168 registers spills, 2160).  Results stored past the caches 1315 -> 1280, where operand and result exceed them (4000^2
// 464 -> 493).  Leaving out the sweeps whose rows a chunk does not need yet: 5 x 3 taps 56.9 -> 52.3 us a sweep, 2000^2 10.2 -> 8.7.  Rows
// fetched 6 or 9 instead of 3 ahead 1820 / 1840 us, strips that start at whole cache lines 1370 (their margins are wider).
// Float64 30 us a sweep, 6000^2 17.8 -> 13.9.  All waves of a launch are resident at once: with 3072 of them passes of 8 took 15.7 us
// a sweep, 2048 16.0, 1024 22.3, 4096, a second generation, 18.0.
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
  int fewer;      // not 0: one sweep less than the kernel's number (LATE only: 4 instructions a row)
  int stream;     // not 0: results go past the caches (acc_sweeps10)
};

struct SweepRow { Spec::E e[ACC_SW_E]; };

// v with its neighbours; XE: the strip reaches beyond the first or last column; OWN: the lane's own columns may lie outside
// too (they do not once acc_sweep_keep has been over them)
template <bool XE, bool OWN> ACC_DEV SweepRow acc_sweep_expand(const Spec::Env& env, const Spec::E (&v)[Spec::V], int gx,
                                                              int w) {
  typedef Spec S;
  const int V = S::V, HX = S::HX;
  SweepRow r;
#pragma unroll
  for (int k = 0; k < V; ++k) r.e[HX + k] = v[k];
#pragma unroll
  for (int j = 1; j <= HX; ++j) {
    r.e[HX - j] = acc_neighbour<0x138, S::LATE>(v[V - j]);          // from the lane to the left
    r.e[HX + V - 1 + j] = acc_neighbour<0x130, S::LATE>(v[j - 1]);  // from the lane to the right
  }
  if constexpr (XE && S::BOUNDARY != 2) {
    // a lane starts at column 0 or at a multiple of V from it, so only the last column can lie
    // inside a lane
    const int first = OWN ? 1 : V;
    if constexpr (S::BOUNDARY == 0) {
#pragma unroll
      for (int i = -1; i >= -HX; --i) r.e[HX + i] = gx + i < 0 ? r.e[HX + i + 1] : r.e[HX + i];
#pragma unroll
      for (int i = first; i < V + HX; ++i) r.e[HX + i] = gx + i >= w ? r.e[HX + i - 1] : r.e[HX + i];
    } else if constexpr (S::BOUNDARY == 1) {
#pragma unroll
      for (int j = 1; j <= HX; ++j) r.e[HX - j] = gx == 0 ? r.e[HX + j] : r.e[HX - j];
#pragma unroll
      for (int i = first; i < V + HX; ++i)
#pragma unroll
        for (int j = 1; j <= HX; ++j)
          if (i - 2 * j >= -HX) r.e[HX + i] = gx + i == w - 1 + j ? r.e[HX + i - 2 * j] : r.e[HX + i];
    } else {
      const S::E c = S::outside(env);
#pragma unroll
      for (int i = -HX; i < V + HX; ++i)
        if (OWN || i < 0 || i >= V) r.e[HX + i] = (gx + i < 0 || gx + i >= w) ? c : r.e[HX + i];
    }
  }
  return r;
}

// A row of a sweep as the wave keeps it until the last sweep that taps it.  Where the function taps neighbours in one row of
// its window only (LATE), they are fetched when they are used: an operand that comes from the next lane then costs no instruction
// of its own, and no registers in between.  Otherwise they are fetched once, when the row is made.
template <bool LATE> struct SweepKept { Spec::E e[Spec::V]; };
template <> struct SweepKept<false> { SweepRow row; };

template <bool XE, bool LATE = Spec::LATE>
ACC_DEV SweepKept<LATE> acc_sweep_keep(const Spec::Env& env, const Spec::E (&v)[Spec::V], int gx, int w) {
  SweepKept<LATE> k;
  const SweepRow r = acc_sweep_expand<XE, true>(env, v, gx, w);
  if constexpr (LATE) {
#pragma unroll
    for (int i = 0; i < Spec::V; ++i) k.e[i] = r.e[Spec::HX + i];
  } else {
    k.row = r;
  }
  return k;
}
template <bool XE, bool LATE> ACC_DEV SweepRow acc_sweep_row(const Spec::Env& env, const SweepKept<LATE>& k, int gx, int w) {
  if constexpr (LATE) return acc_sweep_expand<XE, false>(env, k.e, gx, w);
  else return k.row;
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

template <int T, bool XE, bool NT> ACC_DEV void acc_sweep_strip(const Spec::Env& env, const Spec::Out& out, const SweepParams& p,
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
  SweepKept<S::LATE> win[T][ACC_SW_P];  // win[t][u]: the newest rows of sweep t; row r lies in slot (r - ys + t * HY) % NP
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int u = 0; u < NP; ++u) win[t][u] = SweepKept<S::LATE>{};

  // Sweep t has its first row that is computed from nothing but loaded ones 2 * t * HY steps in: until then it is left out, two sweeps
  // at a time.
  // (not where the rows kept fill the registers: 5 x 5 taps of 8 bytes, 240 of them, Float64 6000^2 112 -> 103 us a sweep, 4096^2 54.4 -> 51.1,
  // 500 x 700 6.5 -> 7.4; Int64 6000^2 134 -> 131)
  constexpr int GROUP = T * NP * (int)sizeof(SweepKept<S::LATE>) / 4 > 192 ? T : 2;
  auto level = [&](auto ye_, auto u_, auto t_, int yin) __attribute__((always_inline)) {
    constexpr bool YE = decltype(ye_)::value != 0;
    constexpr int u = decltype(u_)::value, t = decltype(t_)::value;
    const int y = yin - t * HY;
    SweepRow wv[ACC_SW_P];
#pragma unroll
    for (int q = 0; q < NP; ++q) wv[q] = acc_sweep_row<XE>(env, win[t - 1][(u + 1 + q) % NP], gx, w);
    acc_sweep_window<YE>(env, wv, y, h);
    E r[S::V];
#pragma unroll
    for (int k = 0; k < V; ++k) r[k] = S::apply_win(env, wv, k).c0;
    if constexpr (t == T && S::LATE) {
      // one sweep less: the last one hands on what it finds
#pragma unroll
      for (int k = 0; k < V; ++k) r[k] = p.fewer ? wv[HY].e[S::HX + k] : r[k];
    }
    if constexpr (t < T) {
      win[t][u] = acc_sweep_keep<XE>(env, r, gx, w);
    } else if (y >= y0 && y < y1) {
      E* row = dst + (i64)y * w;
      if constexpr (XE) {
#pragma unroll
        for (int k = 0; k < V; ++k)
          if (gx + k >= lo && gx + k < hi) row[gx + k] = r[k];
      } else if (gx >= lo && gx < hi) {
        typedef E Run __attribute__((vector_size(16), aligned(sizeof(E))));
        Run o;
#pragma unroll
        for (int k = 0; k < V; ++k) o[k] = r[k];
        if constexpr (NT) __builtin_nontemporal_store(o, (Run*)(row + gx));
        else *(Run*)(row + gx) = o;
      }
    }
  };
  auto levels = [&](auto self, auto ye_, auto u_, auto t_, int yin) __attribute__((always_inline)) {
    constexpr int t = decltype(t_)::value;
    if constexpr (t <= T) {
      if (t > 1 && (t - 1) % GROUP == 0 && yin < ys + 2 * t * HY) return;
      level(ye_, u_, t_, yin);
      self(self, ye_, u_, AccConst<t + 1>(), yin);
    }
  };
  auto step = [&](auto ye_, auto u_, int yin) __attribute__((always_inline)) {
    constexpr int u = decltype(u_)::value;
    win[0][u] = acc_sweep_keep<XE>(env, pre[u], gx, w);
    load(yin + NP, pre[u]);
    levels(levels, ye_, u_, AccConst<1>(), yin);
  };
  auto steps = [&](auto self, auto ye_, auto u_, int y) __attribute__((always_inline)) {
    constexpr int u = decltype(u_)::value;
    if constexpr (u < ACC_SW_P) {
      step(ye_, u_, y + u);
      self(self, ye_, AccConst<u + 1>(), y);
    }
  };
  for (int y = ys; y < ye; y += NP) {
    // a sweep of these steps computes rows y - T * HY .. y + NP - 1 - HY, and looks HY rows further
    const bool edge = S::BOUNDARY != 2 && (y - (T + 1) * HY < 0 || y + NP - 1 >= h);
    if (edge) steps(steps, AccConst<1>(), AccConst<0>(), y);
    else steps(steps, AccConst<0>(), AccConst<0>(), y);
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
  const bool inside = x0 >= 0 && x0 + ACC_WAVE * S::V <= p.w;
  // (two copies of the sweeps' code: a choice between two stores at the end of them took 90 more registers.  Strips at the ends of
  // the rows, which store element by element, need no third: Jacobi compiles in 5.9 s instead of 6.7)
  if (T >= 10 && inside && p.stream) acc_sweep_strip<T, false, (T >= 10)>(env, out, p, strip, y0, y1);
  else if (inside) acc_sweep_strip<T, false, false>(env, out, p, strip, y0, y1);
  else acc_sweep_strip<T, true, false>(env, out, p, strip, y0, y1);
}

#if ACC_SW_MAX >= 10
extern "C" __global__ void __launch_bounds__(ACC_BLOCK) acc_sweeps10(Spec::Env env, Spec::Out out, SweepParams p) {
  acc_sweep<10>(env, out, p);
}
#endif
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
