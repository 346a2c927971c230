// Rank-3 stencils (stencilOp, Interpreter.hs:637-649) whose function can be evaluated plane by plane, from registers.
//
// A function of three planes of taps that goes through them in order (a sum from the first tap to the last) needs
// little of a plane once it is past it: the code generator cuts it into three stages, each of which reads one plane and
// hands a few values on (Spec::First, Spec::Second).  A wave marches through the planes with one of them in registers; the plane
// that enters ends the results of the plane before, carries on those of its own and begins those of the next.  Every
// element is loaded once per band of rows instead of staged in LDS, products of a tap and a weight are shared by all the results and
// stages that use them, and instead of three planes the wave holds one and 2 * R * V values.
//
// A lane owns V columns of a band of R rows; the bands' lanes are numbered through and dealt to the waves 62 at a
// time (the outermost two lend their columns to the neighbours, which come by wave shifts), so rows of any length fill the
// lanes.  Lanes that end a row are dealt with where they are: a lane whose columns reach beyond the row loads the row's last V
// and moves them.
//
// Measured (smoothing with 27 taps, 401 x 387 x 393 Float32, floor of the traffic 76 us): 110 us; three planes in registers (stencil3d_rows.hpp)
// 162, through LDS 194.  49.5 vector instructions a result (47.2 million), of which 26 are its additions and about ten the planes
// recomputed at the ends of chunks, against 62 and 100; every row is loaded 5 / 3 times (borders of bands) and every plane 8 / 6 times (borders
// of chunks), mostly from the L2.  Float64 210 / 319 / 333 us.
//
// Outside the array a tap is replaced as `bounded` says (Interpreter.hs:797-839): columns in the registers, rows and
// planes by the index that is loaded, or the constant.  Lanes outside the array compute values nobody uses, on taps that no
// element has, so the function must be defined for all of them.

#define ACC_SP_ROWS (Spec::R + 2 * Spec::HY)
#define ACC_SP_E (Spec::V + 2 * Spec::HX)

struct Stencil3dPlanesParams {
  i64 d, h, w;   // extents; h * w elements are fewer than 2^31 bytes, w at least V
  i64 lanes;     // lanes of a band (wrap: with one more at either end)
  i64 bands;     // bands of S::R rows
  i64 groups;    // workgroups that hold them
  i64 planes;    // planes per chunk
};

struct PlaneRow { Spec::E e[ACC_SP_E]; };
struct PlaneWin { PlaneRow r[ACC_SP_ROWS]; };

static constexpr int kEnd = Spec::HX > 0 ? 1 : 0;  // lanes at either end of a wave that only lend their columns
static constexpr int kOwn = ACC_WAVE - 2 * kEnd;

template <bool XE> ACC_DEV PlaneRow acc_plane_row(const Spec::Env& env, const Spec::E (&v)[Spec::V], int gx, int w) {
  typedef Spec S;
  const int V = S::V, HX = S::HX;
  PlaneRow r;
#pragma unroll
  for (int k = 0; k < V; ++k) r.e[HX + k] = v[k];
  if constexpr (XE && S::BOUNDARY != 2) {
    // (columns of the lane itself that lie outside: mirror may need the left neighbour, so neighbours come first)
#pragma unroll
    for (int j = 1; j <= HX; ++j) r.e[HX - j] = acc_neighbour<0x138, S::FOLD>(v[V - j]);
    if constexpr (S::BOUNDARY == 0) {
#pragma unroll
      for (int i = -1; i >= -HX; --i) r.e[HX + i] = gx + i < 0 ? r.e[HX + i + 1] : r.e[HX + i];
#pragma unroll
      for (int j = 1; j <= HX; ++j) r.e[HX + V - 1 + j] = acc_neighbour<0x130, S::FOLD>(v[j - 1]);
      // (its own are right already: acc_planes moves a row's last element along)
#pragma unroll
      for (int i = V; i < V + HX; ++i) r.e[HX + i] = gx + i >= w ? r.e[HX + i - 1] : r.e[HX + i];
    } else if constexpr (S::BOUNDARY == 1) {
#pragma unroll
      for (int j = 1; j <= HX; ++j) r.e[HX + V - 1 + j] = acc_neighbour<0x130, S::FOLD>(v[j - 1]);
#pragma unroll
      for (int j = 1; j <= HX; ++j) r.e[HX - j] = gx == 0 ? r.e[HX + j] : r.e[HX - j];
#pragma unroll
      for (int i = 1; i < V + HX; ++i)
#pragma unroll
        for (int j = 1; j <= HX; ++j)
          if (i - 2 * j >= -HX) r.e[HX + i] = gx + i == w - 1 + j ? r.e[HX + i - 2 * j] : r.e[HX + i];
    } else {
#pragma unroll
      for (int j = 1; j <= HX; ++j) r.e[HX + V - 1 + j] = acc_neighbour<0x130, S::FOLD>(v[j - 1]);
      const S::E c = S::outside(env);
#pragma unroll
      for (int i = -HX; i < V + HX; ++i) r.e[HX + i] = (gx + i < 0 || gx + i >= w) ? c : r.e[HX + i];
    }
  } else {
#pragma unroll
    for (int j = 1; j <= HX; ++j) {
      r.e[HX - j] = acc_neighbour<0x138, S::FOLD>(v[V - j]);
      r.e[HX + V - 1 + j] = acc_neighbour<0x130, S::FOLD>(v[j - 1]);
    }
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

template <bool XE> ACC_DEV void acc_planes(const Spec::Env& env, const Spec::Out& out, const Stencil3dPlanesParams& p, bool own,
                                           int gx, int y0, int z0, int z1) {
  typedef Spec S;
  typedef S::E E;
  const int V = S::V, HY = S::HY, NR = ACC_SP_ROWS;
  const int d = (int)p.d, h = (int)p.h, w = (int)p.w;
  int col = gx, moved = 0;
  u32 each[S::V];  // wrap, rows that are no whole number of lanes: where a lane's columns lie, one by one
  if constexpr (S::BOUNDARY == 2 && XE) {
    col = 0;
#pragma unroll
    for (int k = 0; k < V; ++k) {
      int c = gx + k;
      if (c < 0) c += w;
      if (c >= w) c -= w;
      each[k] = (u32)(c >= w ? w - 1 : c) * (u32)sizeof(E);
    }
  } else if constexpr (S::BOUNDARY == 2) {
    if (col < 0) col += w;
    if (col >= w) col -= w;
  } else if constexpr (XE) {
    moved = gx + V > w ? gx + V - w : 0;
    col = gx - moved;
  }
  u32 at[ACC_SP_ROWS];   // rows y0 - HY .. y0 + R + HY - 1 of a plane, as the boundary condition reads them: bytes
  bool rowOut[ACC_SP_ROWS];  // constant boundary: the whole row is the constant
#pragma unroll
  for (int j = 0; j < NR; ++j) {
    at[j] = (u32)(acc_bounded(y0 - HY + j, h) * w + col) * (u32)sizeof(E);
    rowOut[j] = S::BOUNDARY == 3 && (y0 - HY + j < 0 || y0 - HY + j >= h);
  }
  const bool ragged = XE && S::BOUNDARY != 2 && w % V != 0;
  auto load = [&](int z, E (&v)[ACC_SP_ROWS][S::V]) __attribute__((always_inline)) {
    const char* plane = (const char*)(S::source(env) + (i64)acc_bounded(z, d) * h * w);
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      if constexpr (S::BOUNDARY == 2 && XE) {
#pragma unroll
        for (int k = 0; k < V; ++k) v[j][k] = *(const E*)(plane + (at[j] + each[k]));
      } else {
        const acc_run<E, S::V> r = *(const acc_run<E, S::V>*)(plane + at[j]);
#pragma unroll
        for (int k = 0; k < V; ++k) v[j][k] = r.e[k];
      }
    }
  };
  auto window = [&](E (&v)[ACC_SP_ROWS][S::V], int z) __attribute__((always_inline)) {
    PlaneWin win;
    if (ragged) {
#pragma unroll
      for (int j = 0; j < NR; ++j)
#pragma unroll
        for (int s = 1; s < V; s *= 2)
#pragma unroll
          for (int k = 0; k < V; ++k) v[j][k] = (moved & s) ? v[j][k + s < V ? k + s : V - 1] : v[j][k];
    }
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      win.r[j] = acc_plane_row<XE>(env, v[j], gx, w);
      if constexpr (S::BOUNDARY == 3) {
        if (rowOut[j] || z < 0 || z >= d) {
          const E c = S::outside(env);
#pragma unroll
          for (int e = 0; e < ACC_SP_E; ++e) win.r[j].e[e] = c;
        }
      }
    }
    return win;
  };
  S::First first[S::R][S::V];
  S::Second second[S::R][S::V];
  const bool whole = gx + V <= w;
  const u32 to = (u32)(y0 * w + gx) * (u32)sizeof(S::T);
  // Plane z: the last of three for the results of z - 1 (END), the middle one for its own (MID), the first for z + 1 (FIRST); the next
  // plane is on its way meanwhile (LOAD).
  auto step = [&](auto does, E (&v)[ACC_SP_ROWS][S::V], E (&next)[ACC_SP_ROWS][S::V], int z) __attribute__((always_inline)) {
    constexpr bool END = does.value & 1, MID = does.value & 2, FIRST = does.value & 4, LOAD = does.value & 8;
    if constexpr (LOAD) load(z + 1, next);
    PlaneWin win = window(v, z);
    S::T r[S::R][S::V];
#pragma unroll
    for (int b = 0; b < S::R; ++b) {
      // (what a result shares with the ones beside it is computed once; what it shares with the next row's would have to be kept for
      // too long, and the compiler must not see that it is the same)
      if (b > 0) {
#pragma unroll
        for (int j = b; j < b + 2 * HY; ++j)
#pragma unroll
          for (int e = 0; e < ACC_SP_E; ++e) asm volatile("" : "+v"(win.r[j].e[e]));
      }
#pragma unroll
      for (int k = 0; k < V; ++k) {
        if constexpr (END) r[b][k] = S::third(env, win, second[b][k], b, k).c0;
        if constexpr (MID) second[b][k] = S::second(env, win, first[b][k], b, k);
        if constexpr (FIRST) first[b][k] = S::first(env, win, b, k);
      }
#pragma unroll
      for (int k = 0; k < V; ++k) {
        if constexpr (END) S::pin(r[b][k]);
        if constexpr (MID) S::pin(second[b][k]);
        if constexpr (FIRST) S::pin(first[b][k]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (END) {
      char* plane = (char*)(S::target(out) + (i64)(z - 1) * h * w);
      if (own && whole) {
#pragma unroll
        for (int b = 0; b < S::R; ++b) {
          acc_run<S::T, S::V> o;
#pragma unroll
          for (int k = 0; k < V; ++k) o.e[k] = r[b][k];
          if (y0 + b < h) *(acc_run<S::T, S::V>*)(plane + (i64)b * w * (i64)sizeof(S::T) + to) = o;
        }
      }
      if (XE && own && !whole) {
#pragma unroll
        for (int b = 0; b < S::R; ++b)
#pragma unroll
          for (int k = 0; k < V; ++k)
            if (y0 + b < h && gx + k < w) ((S::T*)(plane + (i64)b * w * (i64)sizeof(S::T) + to))[k] = r[b][k];
      }
    }
  };
  E a[ACC_SP_ROWS][S::V], c[ACC_SP_ROWS][S::V];   // a plane's rows and the next one's, on their way
  load(z0 - 1, a);
  step(AccConst<4 + 8>(), a, c, z0 - 1);
  if (z1 - z0 == 1) {
    step(AccConst<2 + 8>(), c, a, z0);
  } else {
    step(AccConst<2 + 4 + 8>(), c, a, z0);
    int z = z0 + 1;
    for (; z + 1 <= z1 - 2; z += 2) {
      step(AccConst<15>(), a, c, z);
      step(AccConst<15>(), c, a, z + 1);
    }
    if (z <= z1 - 2) {
      step(AccConst<15>(), a, c, z);
#pragma unroll
      for (int j = 0; j < NR; ++j)
#pragma unroll
        for (int k = 0; k < V; ++k) a[j][k] = c[j][k];
    }
    step(AccConst<1 + 2 + 8>(), a, c, z1 - 1);
#pragma unroll
    for (int j = 0; j < NR; ++j)
#pragma unroll
      for (int k = 0; k < V; ++k) a[j][k] = c[j][k];
  }
  step(AccConst<1>(), a, c, z1);
}

extern "C" __global__ void __launch_bounds__(ACC_BLOCK)
acc_stencil3d_planes(Spec::Env env, Spec::Out out, Stencil3dPlanesParams p) {
  typedef Spec S;
  // chunks of planes outermost; neighbouring bands share rows: neighbours run on the same XCD
  const i64 b = acc_xcd_contiguous((i64)blockIdx.x, (i64)gridDim.x);
  const int chunk = (int)(b / p.groups);
  const i64 wave = (b - chunk * p.groups) * ACC_WAVES + __builtin_amdgcn_readfirstlane(acc_wave());
  const int all = (int)(p.lanes * p.bands);
  const i64 t0 = wave * kOwn - kEnd;
  if (t0 + kEnd >= all) return;
  int t = (int)t0 + acc_lane();
  bool own = acc_lane() >= kEnd && acc_lane() < ACC_WAVE - kEnd && t < all;
  t = t < 0 ? 0 : (t >= all ? all - 1 : t);
  const int band = (int)((u32)t / (u32)p.lanes);
  int pos = t - band * (int)p.lanes;
  bool edge = pos == 0 || pos == (int)p.lanes - 1;
  if constexpr (S::BOUNDARY == 2 && S::HX > 0) {
    own = own && !edge;
    --pos;
    // (a row's last lane of its own may reach beyond it, and may be its wave's outermost, with no lending lane in the wave)
    edge = edge || (i64)(pos + 1) * S::V > p.w;
  }
  const i64 z0 = chunk * p.planes, z1 = z0 + p.planes < p.d ? z0 + p.planes : p.d;
  if ((S::BOUNDARY == 2 && p.w % S::V == 0) || __ballot(edge) == 0) acc_planes<false>(env, out, p, own, pos * S::V, band * S::R, (int)z0, (int)z1);
  else acc_planes<true>(env, out, p, own, pos * S::V, band * S::R, (int)z0, (int)z1);
}
