"""Where the lanes of acc_stencil3d_planes read and write, on the CPU: the kernel's own source, compiled for the host with
a counting element type and run lane by lane.  What a lane reads and lends to nobody is in no result, so no comparison of results
can see that it lies outside the operand."""
import os
import subprocess

import pytest

DEVICE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "accelerate_amd", "csrc", "device")

HOST = r"""
#include <csetjmp>
#include <cstdio>
#include <vector>
typedef int i32; typedef long long i64; typedef unsigned u32; typedef unsigned long long u64;
#define ACC_DEV static inline
#define ACC_WAVE 64
#define ACC_BLOCK 256
#define ACC_WAVES 4
#define __global__
#define __launch_bounds__(...)
#define asm
#define volatile(...)
struct Dim { unsigned x; } blockIdx, gridDim, threadIdx;
static int acc_lane() { return threadIdx.x % 64; }
static int acc_wave() { return threadIdx.x / 64; }
static int __builtin_amdgcn_readfirstlane(int v) { return v; }
static void __builtin_amdgcn_sched_barrier(int) {}
static i64 acc_xcd_contiguous(i64 b, i64) { return b; }

// a lane stops at the ballot, if it comes to one, until all lanes of its wave have said what they vote for
static jmp_buf stopped;
static bool voting;
static u64 votes;
static u64 __ballot(bool v) {
  if (!voting) return votes;
  votes |= (u64)v << acc_lane();
  longjmp(stopped, 1);
}

// operand and result lie in the middle of larger blocks: an address beside them is seen, and does no harm
static const i64 kBeside = 1 << 11;
static i64 D, H, W;
template <class T> struct Block {
  std::vector<T> all;
  std::vector<int> times;
  i64 outside = 0, across = 0;
  T* base() { return all.data() + kBeside; }
  void reset() { all.assign(D * H * W + 2 * kBeside, T()); times.assign(D * H * W, 0); }
  bool holds(const void* p) { return !all.empty() && p >= (const void*)all.data() && p < (const void*)(all.data() + all.size()); }
  void touch(const void* p, int run) {
    if (!holds(p)) return;
    const i64 at = (const T*)p - base();
    if (at < 0 || at + run > D * H * W) ++outside;
    else if (at % W + run > W) ++across;
    else for (int k = 0; k < run; ++k) ++times[at + k];
  }
};
struct Elem;
struct Res;
static Block<Elem>& source();
static Block<Res>& result();
struct Elem {
  BASE v = 0;
  Elem() = default;
  Elem(const Elem& o) : v(o.v) { source().touch(&o, 1); }
  Elem& operator=(const Elem& o) { v = o.v; source().touch(&o, 1); return *this; }
};
struct Res {
  BASE v = 0;
  Res() = default;
  Res(const Res& o) = default;
  Res& operator=(const Res& o) { v = o.v; result().touch(this, 1); return *this; }
};
static Block<Elem>& source() { static Block<Elem> b; return b; }
static Block<Res>& result() { static Block<Res> b; return b; }
template <class T, int N> struct acc_run;
template <int N> struct acc_run<Elem, N> {
  Elem e[N];
  acc_run(const acc_run& o) { source().touch(&o, N); }
};
template <int N> struct acc_run<Res, N> {
  Res e[N];
  acc_run() = default;
  acc_run& operator=(const acc_run&) { result().touch(this, N); return *this; }
};

template <int CTRL, bool FOLD, class T> T acc_neighbour(const T&) { return T(); }
template <int N> struct AccConst { static constexpr int value = N; };

struct Spec {
  struct Env {};
  struct Out {};
  struct Elt { Res c0; };
  struct First {};
  struct Second {};
  typedef Elem E;
  typedef Res T;
  static constexpr int V = COLUMNS, R = 3, HZ = 1, HY = 1, HX = HALO, BOUNDARY = KIND;
  static constexpr bool FOLD = false;
  static Elem outside(const Env&) { return Elem(); }
  static const Elem* source(const Env&) { return ::source().base(); }
  static Res* target(const Out&) { return ::result().base(); }
  template <class X> static void pin(X&) {}
  template <class W> static First first(const Env&, const W&, int, int) { return {}; }
  template <class W> static Second second(const Env&, const W&, const First&, int, int) { return {}; }
  template <class W> static Elt third(const Env&, const W&, const Second&, int, int) { return {}; }
};
#include "stencil3d_planes.hpp"

int main() {
  const i64 V = Spec::V, own = HALO ? 62 : 64, depths[] = {1, 2, 5}, heights[] = {1, 2, 3, 4, 7, 20, 64};
  i64 bad = 0;
  for (W = V; W < 510; W += W < 20 || W % 61 < 3 || W % 62 < 3 || W % 124 < 5 ? 1 : 7)
    for (i64 h : heights)
      for (i64 d : depths) {
        if (h * d > 64 && W % 124 > 2) continue;  // (the largest only where waves and rows end together)
        H = h, D = d;
        source().reset(), result().reset();
        source().outside = source().across = result().outside = result().across = 0;
        Stencil3dPlanesParams p;
        p.d = D, p.h = H, p.w = W;
        p.lanes = (W + V - 1) / V + (HALO && KIND == 2 ? 2 : 0);
        p.bands = (H + 2) / 3;
        p.groups = ((p.lanes * p.bands + own - 1) / own + 3) / 4;
        p.planes = d == 5 ? 3 : 2;
        gridDim.x = p.groups * ((D + p.planes - 1) / p.planes);
        for (blockIdx.x = 0; blockIdx.x < gridDim.x; ++blockIdx.x)
          for (unsigned wave = 0; wave < 4; ++wave) {
            votes = 0;
            static bool waits[64];
            for (unsigned lane = 0; lane < 64; ++lane) {
              threadIdx.x = wave * 64 + lane;
              voting = true;
              waits[lane] = setjmp(stopped) != 0;
              if (!waits[lane]) acc_stencil3d_planes(Spec::Env(), Spec::Out(), p);
            }
            voting = false;
            for (unsigned lane = 0; lane < 64; ++lane) {
              threadIdx.x = wave * 64 + lane;
              if (waits[lane]) acc_stencil3d_planes(Spec::Env(), Spec::Out(), p);
            }
          }
        i64 written = 0;
        for (int t : result().times) written += t == 1;
        if (source().outside || source().across || result().outside || result().across || written != D * H * W)
          if (bad++ < 5)
            std::printf("%lld x %lld x %lld: read outside %lld, across rows %lld, wrote outside %lld, across %lld, once %lld of %lld\n", D, H, W,
                        source().outside, source().across, result().outside, result().across, written, D * H * W);
      }
  std::printf("%lld shapes wrong\n", bad);
  return bad != 0;
}
"""

KINDS = {"clamp": 0, "mirror": 1, "wrap": 2, "constant": 3}


@pytest.mark.parametrize("halo", [1, 0])
@pytest.mark.parametrize("kind,base,columns", [("clamp", "float", 4), ("mirror", "float", 4), ("wrap", "float", 2), ("constant", "double", 2),
                                               ("wrap", "double", 1)])
def test_every_access_lies_in_its_row(tmp_path, kind, base, columns, halo):
    src, exe = tmp_path / "planes.cpp", tmp_path / "planes"
    src.write_text(HOST)
    subprocess.run(["g++", "-std=c++17", "-O2", "-w", "-I", DEVICE, "-DBASE=" + base, "-DCOLUMNS=%d" % columns, "-DHALO=%d" % halo,
                    "-DKIND=%d" % KINDS[kind], "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
