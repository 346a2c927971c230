// Entry point of the scan skeleton: one workgroup per tile, tiles numbered by ticket in
// row-major (row, tile-in-row) order; the tile machinery lives in scan.hpp.

template <class S, bool ALL> ACC_DEV void acc_scan_body(const Spec::Env& env, const Spec::Out& out, const Spec::Out& tot, const ScanParams& p) {
  typedef typename S::Elt Elt;
  const int W = AccScanCfg<S>::W;
  // (no counter: the launch holds no more tiles than the device holds workgroups at a time)
  const i64 gtile = p.ticket ? acc_take_ticket(p.ticket, p.ticket_base) : (i64)blockIdx.x;
  // a ticket outside the launch means that the host's count of tickets is off: touch nothing
  if (gtile < 0 || gtile >= p.rows * p.tpr) {
    if (threadIdx.x == 0) __hip_atomic_store(p.err, 3u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return;
  }
  const i64 row = gtile / p.tpr;
  const i64 tile = gtile - row * p.tpr;
  const i64 n = p.n;
  const i64 inBase = row * n;
  const i64 m = S::kKind == 1 ? n + 1 : n;  // entries per output row
  const i64 outBase = row * m;
  u64* rowDesc = p.desc + (u64)row * (u64)p.tpr * W;

  auto load = [&](i64 t) -> Elt { return S::in_linear(env, inBase + (S::kRight ? n - 1 - t : t)); };
  auto store = [&](i64 t, const Elt& y) {
    if (S::kKind == 0) {
      S::store(out, outBase + (S::kRight ? n - 1 - t : t), y);
    } else {
      const i64 u = t + 1;
      if (S::kKind == 2 && u == n) S::store(tot, row, y);
      else S::store(out, outBase + (S::kRight ? m - 1 - u : u), y);
    }
  };
  // the V consecutive values of a lane, moved with one wide request per leaf (a right scan
  // writes them in reverse).  scan' keeps the row's total apart: only the row's last tile can
  // hold it, the others need no test.
  auto storeRun = [&](i64 t0, const Elt* y) {
    const i64 shift = S::kKind == 0 ? 0 : 1;
    if (!S::kRight) {
      S::store_run(out, outBase + t0 + shift, y);
    } else {
      Elt z[S::V];
#pragma unroll
      for (int k = 0; k < S::V; ++k) z[k] = y[S::V - 1 - k];
      S::store_run(out, outBase + (m - 1 - shift) - (t0 + S::V - 1), z);
    }
  };
  acc_scan_tile<S, ALL>(env, rowDesc, p.tpr, tile, n, p.epoch, p.spin_limit, p.err, load, store, storeRun, S::kKind != 2 || tile + 1 < p.tpr,
                   p.rows * p.tpr >= ACC_SCAN_SETTLE_TILES);

  if (S::kKind != 0 && tile == 0 && threadIdx.x == 0) {
    Elt z = S::seed(env);
    if (S::kKind == 2 && n == 0) S::store(tot, row, z);
    else S::store(out, outBase + (S::kRight ? m - 1 : 0), z);
  }
}

#ifdef ACC_SCAN_FILL
// The launch is a chain of round trips with memory idle in between: the buffer of the next node's defaults is written by its
// last instructions instead of by a launch of 3 us (a radix pass of one million keys 23.4 -> 19.6 us, of 1000 keys 12.1 -> 9.1).
ACC_DEV void acc_scan_fill(const ScanFill& f) {
  const i64 step = (i64)gridDim.x * ACC_SCAN_BLOCK * 2;
  for (i64 i = ((i64)blockIdx.x * ACC_SCAN_BLOCK + threadIdx.x) * 2; i < f.n; i += step) {
    typedef u64 Two __attribute__((ext_vector_type(2)));
    const Two w = {f.word, f.word};
    *(Two*)(f.at + i) = w;
  }
}
#define ACC_SCAN_FILL_PARAM , ScanFill f
#else
#define ACC_SCAN_FILL_PARAM
#endif

extern "C" __global__ void __launch_bounds__(ACC_SCAN_BLOCK, ACC_SCAN_MINWAVES)
acc_scan(Spec::Env env, Spec::Out out, Spec::Out tot, ScanParams p) {
  acc_scan_body<Spec, false>(env, out, tot, p);
}

#ifdef ACC_SCAN_ALL_G
// A few hundred tiles that all run at once: what such a launch takes is a chain of round trips, to the
// data, to the predecessors and back, so tiles are a quarter (a half) of the small ones' size, that
// every CU gets one, and each reads the aggregates of all its predecessors itself (acc_lookback_all)
// instead of waiting for prefixes to travel along the row.  2^18 Float32 7.0 -> 4.6 us, 2^20 Int64
// 9.3 -> 7.2, 2^22 Float32 12.7 -> 10.2.
struct AccAllSpec : Spec {
  static constexpr int G = ACC_SCAN_ALL_G;
};
extern "C" __global__ void __launch_bounds__(ACC_SCAN_BLOCK, ACC_SCAN_MINWAVES)
acc_scan_all(Spec::Env env, Spec::Out out, Spec::Out tot, ScanParams p ACC_SCAN_FILL_PARAM) {
#ifdef ACC_SCAN_FILL
  const i64 words = f.n;
  asm volatile("" : : "s"(words));  // (read with the other parameters: a scalar load at the end costs 0.4 us)
#endif
  acc_scan_body<AccAllSpec, true>(env, out, tot, p);
#ifdef ACC_SCAN_FILL
  if (words) acc_scan_fill(f);
#endif
}
struct AccAll2Spec : Spec {
  static constexpr int G = 2 * ACC_SCAN_ALL_G;
};
extern "C" __global__ void __launch_bounds__(ACC_SCAN_BLOCK, ACC_SCAN_MINWAVES)
acc_scan_all2(Spec::Env env, Spec::Out out, Spec::Out tot, ScanParams p ACC_SCAN_FILL_PARAM) {
#ifdef ACC_SCAN_FILL
  const i64 words = f.n;
  asm volatile("" : : "s"(words));  // (read with the other parameters: a scalar load at the end costs 0.4 us)
#endif
  acc_scan_body<AccAll2Spec, true>(env, out, tot, p);
#ifdef ACC_SCAN_FILL
  if (words) acc_scan_fill(f);
#endif
}
#endif

#ifdef ACC_ROWS_G  // the small variant
// Rows of at most half a tile: a workgroup scans rpt whole rows at once (acc_rows_tile).
struct ScanRowsParams {
  i64 rows;
  i64 n;    // 1 <= n, rpt * n <= TILE
  i64 rpt;  // rows per workgroup
};

// the rows kernel's own tile size (values carry a head flag there: half the elements per lane)
struct AccRowsSpec : Spec {
  static constexpr int G = ACC_ROWS_G;
};

extern "C" __global__ void __launch_bounds__(ACC_SCAN_BLOCK, ACC_SCAN_MINWAVES)
acc_scan_rows(Spec::Env env, Spec::Out out, Spec::Out tot, ScanRowsParams p) {
  typedef Spec S;
  typedef S::Elt Elt;
  const i64 row0 = (i64)blockIdx.x * p.rpt;
  const i64 nrows = p.rows - row0 < p.rpt ? p.rows - row0 : p.rpt;
  const int n = (int)p.n;
  const i64 m = S::kKind == 1 ? p.n + 1 : p.n;  // entries per output row
  auto load = [&](int idx, int r, int t) -> Elt {
    Elt v = S::in_linear(env, S::kRight ? (row0 + r) * p.n + (n - 1 - t) : row0 * p.n + idx);
    if (S::kSeeded && t == 0) v = S::combine(env, S::seed(env), v);
    return v;
  };
  auto store = [&](int idx, int r, int t, const Elt& y) {
    const i64 row = row0 + r;
    if (S::kKind == 0) {
      S::store(out, S::kRight ? row * p.n + (n - 1 - t) : row0 * p.n + idx, y);
    } else {
      const i64 outBase = row * m;
      if (t == 0) S::store(out, outBase + (S::kRight ? m - 1 : 0), S::seed(env));
      const i64 u = (i64)t + 1;
      if (S::kKind == 2 && u == p.n) S::store(tot, row, y);
      else S::store(out, outBase + (S::kRight ? m - 1 - u : u), y);
    }
  };
  acc_rows_tile<AccRowsSpec>(env, (int)(nrows * p.n), n, load, store);
}
#endif
