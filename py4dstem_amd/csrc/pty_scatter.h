// Deterministic scatter-add of staged frames into the object, as phases
// between barriers (compiled for the GPU, and for the host emulator that checks
// their LDS accesses and indices).
//
// The sums are those of Gather in pty_core.h, bit for bit: per object pixel
// conj(P_shift) * chi and |P_shift|^2, float32 products rounded separately,
// added in float64 in batch order.  A pixel's sum is one serial chain, so a
// thread per pixel leaves the chip idle wherever the object is small (a
// 256^2 object is one wave per SIMD) while hundreds of windows overlap.  Here
// a work group of four waves owns a tile of TP pixels and deals the tile's
// hit list to its waves: each wave loads and multiplies HPW hits of a chunk
// for the whole tile and leaves the float32 products in LDS, then the
// threads, one (component, pixel) pair each, add the chunk in hit order.
// Loads of the next chunk are in flight meanwhile (two product buffers, one
// barrier per chunk).  Lanes outside a hit's window read beyond the buffer's
// range, which returns zeros without a memory access: their products add
// +0.0.  Tile rows are dealt to the 8 XCDs in turn, so column neighbours,
// which share the cache lines at their common edge, use the same L2.
//
// Bound: HBM/Infinity-Cache reads where the object is large, the load-to-add
// round trip of a tile's hit list where it is small.  Scatter alone, one
// launch, against the one-thread-per-pixel-pair kernel it replaced
// (8 x 64 tiles, 4 hits in flight): 128 px frames, 740 slots on 284x272
// pixels 166 -> 45 us; 400 slots on 284^2 94 -> 26 us; 64 px, 1024 slots on
// 256^2 87 -> 20 us; 32 px, 64 slots on 128^2 18 -> 8 us; 128 px, 1024 slots
// on 720^2 63 -> 56 us (4.8 TB/s of frame bytes).

#pragma once

#include <algorithm>

#include "pty_core.h"

namespace pty {

// Tile of a work group: ROWS lane-rows of C columns, R pixels per lane.
// R = 1 (4 x 16 pixels): most work groups, shortest hit lists.
// R = 4 (8 x 32 pixels): a quarter of the hit tests and list look-ups.
template <int R> struct ScatterTile {
  static constexpr int C = R == 1 ? 16 : 32;
  static constexpr int LR = 64 / C;           // rows of lanes in a wave
  static constexpr int ROWS = LR * R;
  static constexpr int TP = 64 * R;           // pixels
  static constexpr int HPW = R == 1 ? 4 : 1;  // hits per wave and chunk
  static constexpr int CHUNK = 4 * HPW;
};
constexpr int SCATTER_SEG = 1024;  // batch slots per hit list
constexpr int SCATTER_THREADS = 256;

// Beyond this many object pixels the 256-pixel tiles are used: 4096 work
// groups of 64 pixels are about four rounds of the 1024 that fit the chip
// (LDS).  Measured where hundreds of windows overlap, with 128 px frames: 284x272 pixels 45 us against 115 us with 256-pixel
// tiles, 440x416 (256 px frames) 32 against 42, 720^2 74 against 56.
constexpr long long SCATTER_SMALL_PIXELS = 64 * 4096;

// num_tiles: entries of tilemax, at least the launch's own tiles; those beyond
// them are cleared (|P|^2 sums are not negative)
struct ScatterPlan {
  int rows_per_lane, tiles_x, tiles_y, num_tiles;
};

PTY_HD int scatter_rows(int Px, int Py) { return (long long)Px * Py <= SCATTER_SMALL_PIXELS ? 1 : 4; }
// 256-pixel tiles below that, too, where a pixel meets few windows: a quarter
// of the hit tests against longer lists and fewer work groups, for `pixels` of
// all objects that share the launch (the problems of a batched run, the modes
// of a mixed state).  r = pixels / SCATTER_SMALL_PIXELS, h = frame_pixels /
// pixels windows a pixel.  Whole runs with 64-pixel tiles over runs with
// 256-pixel ones: r 0.12, h 2 0.97; r 0.26, h 1.5 1.07, h 4 1.02, h 12 0.96;
// r 0.5, h 2 1.16, h 6 1.07, h 25 0.96; r 0.9, h 14 1.10, h 42 1.01; r 1.1,
// h 5 1.13, h 20 1.01, h 54 0.95, h 167 0.91; r 2.9, h 8 1.20, h 21 1.09, h 84
// 0.99, h 276 0.98; r 6.7, h 24 1.11, h 95 1.01, h 263 1.00; r 11, h 44 1.09.
inline bool scatter_wide(long long pixels, long long frame_pixels) {
  const double r = (double)pixels / (double)SCATTER_SMALL_PIXELS;
  return (double)frame_pixels <= 25.0 * r * std::min(r, 1.0) * (double)pixels;
}
PTY_HD ScatterPlan scatter_plan(int Px, int Py, int rows_per_lane) {
  ScatterPlan s;
  s.rows_per_lane = rows_per_lane;
  const int rows = rows_per_lane == 1 ? ScatterTile<1>::ROWS : ScatterTile<4>::ROWS;
  const int cols = rows_per_lane == 1 ? ScatterTile<1>::C : ScatterTile<4>::C;
  s.tiles_x = (Px + rows - 1) / rows;
  s.tiles_y = (Py + cols - 1) / cols;
  s.num_tiles = s.tiles_x * s.tiles_y;
  return s;
}
PTY_HD int scatter_num_tiles(int Px, int Py) {
  return scatter_plan(Px, Py, scatter_rows(Px, Py)).num_tiles;
}
// work groups of a launch: tile rows rounded up to the 8 XCDs
PTY_HD int scatter_blocks(const ScatterPlan& s) { return (s.tiles_x + 7) / 8 * 8 * s.tiles_y; }
// the frames are read through one buffer resource with a 32-bit byte range
PTY_HD bool scatter_in_range(int B, int S) { return (long long)B * S * S * 8 <= 0x7fffffffll; }

struct ScatterHit {
  int offset;  // byte offset of the slot's frame
  int dr, dc;  // tile origin in window coordinates, in [0, Px) x [0, Py)
};

template <int R> struct ScatterShared {
  using T = ScatterTile<R>;
  ScatterHit list[SCATTER_SEG];
  float prod[2 * 3 * T::CHUNK * T::TP];  // [buffer][component][hit][pixel]
  int count[4];
  float red[4];
};

template <int R> struct ScatterSharedView {
  ScatterShared<R>* s;
  PTY_HD LdsArr<ScatterHit> list() const { return LdsArr<ScatterHit>{s->list}; }
  PTY_HD LdsArr<float> prod() const { return LdsArr<float>{s->prod}; }
  PTY_HD LdsArr<int> count() const { return LdsArr<int>{s->count}; }
  PTY_HD LdsArr<float> red() const { return LdsArr<float>{s->red}; }
};

// Frames read through a buffer resource of `range` bytes.  SCATTER_OUT as a
// lane's offset is beyond every range: zeros, without a memory access.
constexpr unsigned SCATTER_OUT = 0x80000000u;
struct ScatterBuf {
#if defined(__HIP_DEVICE_COMPILE__)
  __amdgpu_buffer_rsrc_t r;
#else
  const cf* p;
  unsigned range;
#endif
};

PTY_HD ScatterBuf scatter_buf(const cf* p, int range) {
  ScatterBuf b;
#if defined(__HIP_DEVICE_COMPILE__)
  b.r = __builtin_amdgcn_make_buffer_rsrc(const_cast<cf*>(p), (short)0, range, 0x00020000);
#else
  b.p = p;
  b.range = (unsigned)range;
#endif
  return b;
}

// vo: the lane's byte offset, so: the wave's
PTY_HD cf scatter_load(const ScatterBuf& b, unsigned vo, int so) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_bit_cast(cf, __builtin_amdgcn_raw_buffer_load_b64(b.r, vo, so, 0));
#else
  if (vo == SCATTER_OUT) return mkcf(0.f, 0.f);
  PTY_CHECK(so >= 0 && vo % 8 == 0 && vo + (unsigned)so + 8u <= b.range, "scatter load out of range");
  return b.p[(vo + (unsigned)so) / 8u];
#endif
}

// set bits of a wave's mask, all and those below a lane
PTY_HD int mask_count(unsigned long long m) { return __builtin_popcountll(m); }
PTY_HD int mask_rank(unsigned long long m, int lane) {
#if defined(__HIP_DEVICE_COMPILE__)
  (void)lane;
  return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
#else
  return __builtin_popcountll(m & ((1ull << lane) - 1ull));
#endif
}

// the tile of a work group
struct ScatterOrigin {
  int tr, tc, R0, C0;
};

template <int R> struct Scatter {
  using T = ScatterTile<R>;
  static constexpr int C = T::C, LR = T::LR, TP = T::TP, HPW = T::HPW, CHUNK = T::CHUNK;
  static constexpr int CAND = SCATTER_SEG / SCATTER_THREADS;  // slots tested per thread
  // (component, pixel) pairs, pair e = THREADS k + tid of a thread: component
  // e / TP of tile pixel e % TP
  static constexpr int PAIRS = 3 * TP, PPT = (PAIRS + SCATTER_THREADS - 1) / SCATTER_THREADS;

  struct Regs {
    double acc[PPT];
    int dr[CAND], dc[CAND], at[CAND];
    bool hit[CAND];
    unsigned long long mask[CAND];  // hit[k] over the wave
    int n, nh;                      // hits of the wave, of the segment
    cf p[HPW][R], c[HPW][R];
    float max;
  };

  static PTY_HD ScatterOrigin origin(const ScatterPlan& plan, int blk) {
    ScatterOrigin t;
    const int j = blk >> 3;
    t.tr = (j / plan.tiles_y) * 8 + (blk & 7);
    t.tc = j % plan.tiles_y;
    t.R0 = t.tr * T::ROWS;
    t.C0 = t.tc * C;
    return t;
  }

  static PTY_HD bool pixel(const GatherArgs& a, const ScatterOrigin& t, int e, int& row, int& col) {
    const int p = e % TP;
    row = t.R0 + (p / 64) * LR + (p % 64) / C;
    col = t.C0 + p % C;
    return (PAIRS % SCATTER_THREADS == 0 || e < PAIRS) && row < a.Px && col < a.Py;
  }

  static PTY_HD int prod_at(int buf, int comp, int hit, int pix) { return ((buf * 3 + comp) * CHUNK + hit) * TP + pix; }

  // running sums: zero, or carried over from the previous stage of the batch
  static PTY_HD void p_init(int tid, const GatherArgs& a, const ScatterOrigin& t, Regs& r) {
#pragma unroll
    for (int k = 0; k < PPT; ++k) {
      const int e = SCATTER_THREADS * k + tid;
      int row, col;
      r.acc[k] = 0.0;
      if (a.run && !a.run_first && pixel(a, t, e, row, col)) r.acc[k] = a.run[((size_t)row * a.Py + col) * 3 + e / TP];
    }
  }

  // hits of a segment in batch order: wave w tests slots [w, w + 1) * 64 CAND
  // of it, the masks give the order inside the wave
  static PTY_HD int slot(int tid, int seg0) { return seg0 + wave_uniform(tid >> 6) * (64 * CAND) + (tid & 63); }

  static PTY_HD void p_test(int tid, const GatherArgs& a, const ScatterOrigin& t, int seg0, Regs& r) {
    const int S = a.S, b0 = slot(tid, seg0);
    const int rows = a.Px - t.R0, cols = a.Py - t.C0;
    const int th = rows < T::ROWS ? rows : T::ROWS, tw = cols < C ? cols : C;
    int idx[CAND];
    float px[CAND], py[CAND];
#pragma unroll
    for (int k = 0; k < CAND; ++k) {
      const int b = b0 + 64 * k;
      idx[k] = a.order[b < a.B ? b : 0];
      idx[k] = ((unsigned)idx[k] < (unsigned)a.N) ? idx[k] : 0;
    }
#pragma unroll
    for (int k = 0; k < CAND; ++k) {
      px[k] = a.positions[2 * idx[k]];
      py[k] = a.positions[2 * idx[k] + 1];
    }
#pragma unroll
    for (int k = 0; k < CAND; ++k) {
      const int x0 = wrapi_fast((int)rintf(px[k]), a.Px), y0 = wrapi_fast((int)rintf(py[k]), a.Py);
      r.dr[k] = wrap1(t.R0 - x0 + S / 2, a.Px);
      r.dc[k] = wrap1(t.C0 - y0 + S / 2, a.Py);
      r.hit[k] = (b0 + 64 * k < a.B) & ((r.dr[k] < S) | (r.dr[k] + th > a.Px)) & ((r.dc[k] < S) | (r.dc[k] + tw > a.Py));
    }
  }

  template <class V> static PTY_HD void p_rank(int tid, Regs& r, V sh) {
    r.n = 0;
#pragma unroll
    for (int k = 0; k < CAND; ++k) {
      r.at[k] = r.n + mask_rank(r.mask[k], tid & 63);
      r.n += mask_count(r.mask[k]);
    }
    if ((tid & 63) == 0) sh.count().st(wave_uniform(tid >> 6), r.n);
  }

  template <class V> static PTY_HD void p_list(int tid, const GatherArgs& a, int seg0, Regs& r, V sh) {
    const int wave = wave_uniform(tid >> 6), b0 = slot(tid, seg0);
    int base = 0, nh = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const int c = sh.count().ld(w);
      base += w < wave ? c : 0;
      nh += c;
    }
    r.nh = wave_uniform(nh);
#pragma unroll
    for (int k = 0; k < CAND; ++k)
      if (r.hit[k]) sh.list().st(base + r.at[k], ScatterHit{(b0 + 64 * k) * (a.S * a.S * 8), r.dr[k], r.dc[k]});
  }

  // this wave's hits of the chunk at h0, requested
  template <class V>
  static PTY_HD void p_load(int tid, const GatherArgs& a, const ScatterBuf& ps, const ScatterBuf& chi, int h0, Regs& r,
                            V sh) {
    const unsigned S = (unsigned)a.S, lr = (tid & 63) / C, lc = (tid & 63) % C;
    const int ls = __builtin_ctz(S);
#pragma unroll
    for (int u = 0; u < HPW; ++u) {
      const int h = h0 + wave_uniform(tid >> 6) * HPW + u;
      const ScatterHit e = sh.list().ld(h < r.nh ? h : 0);  // beyond the list: loaded, not added
      const int so = wave_uniform(e.offset);
      unsigned d = (unsigned)e.dc + lc;
      d = umin(d, d - (unsigned)a.Py);
#pragma unroll
      for (int g = 0; g < R; ++g) {
        unsigned w = (unsigned)e.dr + lr + g * LR;
        w = umin(w, w - (unsigned)a.Px);
        unsigned o = ((w ^ (S / 2)) << (ls + 3)) | ((d ^ (S / 2)) << 3);
        o = (w | d) < S ? o : SCATTER_OUT;  // S a power of two: both below S
        r.p[u][g] = scatter_load(ps, o, so);
        r.c[u][g] = scatter_load(chi, o, so);
      }
    }
  }

  // their products, separately rounded (no fused multiply-add)
  template <class V> static PTY_HD void p_products(int tid, int buf, Regs& r, V sh) {
#if defined(__clang__)
#pragma clang fp contract(off)
#endif
    const int lane = tid & 63, h0 = wave_uniform(tid >> 6) * HPW;
#pragma unroll
    for (int u = 0; u < HPW; ++u)
#pragma unroll
      for (int g = 0; g < R; ++g) {
        const cf t = cconjmul_rn(r.p[u][g], r.c[u][g]);
        sh.prod().st(prod_at(buf, 0, h0 + u, g * 64 + lane), t.x);
        sh.prod().st(prod_at(buf, 1, h0 + u, g * 64 + lane), t.y);
        sh.prod().st(prod_at(buf, 2, h0 + u, g * 64 + lane), cabs2_rn(r.p[u][g]));
      }
  }

  // the chunk's first m products of this thread's pairs, in hit order
  template <class V> static PTY_HD void p_add(int tid, int buf, int m, Regs& r, V sh) {
#pragma unroll
    for (int k = 0; k < PPT; ++k) {
      const int e = SCATTER_THREADS * k + tid;
      if (PAIRS % SCATTER_THREADS == 0 || e < PAIRS) {
        const int f = prod_at(buf, e / TP, 0, e % TP);
        if (m == CHUNK) {
#pragma unroll
          for (int h = 0; h < CHUNK; ++h) r.acc[k] += (double)sh.prod().ld(f + h * TP);
        } else {
          for (int h = 0; h < m; ++h) r.acc[k] += (double)sh.prod().ld(f + h * TP);
        }
      }
    }
  }

  static PTY_HD void p_store(int tid, const GatherArgs& a, const ScatterOrigin& t, Regs& r) {
    r.max = 0.f;
#pragma unroll
    for (int k = 0; k < PPT; ++k) {
      const int e = SCATTER_THREADS * k + tid, comp = e / TP;
      int row, col;
      if (!pixel(a, t, e, row, col)) continue;
      const size_t o = (size_t)row * a.Py + col;
      if (a.acc) {
        if (comp < 2) a.acc[2 * o + comp] += r.acc[k];
      } else if (a.run && !a.run_last) {
        a.run[o * 3 + comp] = r.acc[k];
      } else {
        const float v = (float)r.acc[k];
        if (comp == 0) a.grad[o].x = v;
        else if (comp == 1) a.grad[o].y = v;
        else {
          a.spsum[o] = v;
          r.max = fmaxf(r.max, v);
        }
      }
    }
  }

  template <class V>
  static PTY_HD void p_max(int tid, const GatherArgs& a, const ScatterPlan& plan, const ScatterOrigin& t, V sh) {
    if (tid != 0) return;
    const int own = plan.tiles_x * plan.tiles_y;
    int i = t.tr * plan.tiles_y + t.tc;
    a.tilemax[i] = fmaxf(fmaxf(sh.red().ld(0), sh.red().ld(1)), fmaxf(sh.red().ld(2), sh.red().ld(3)));
    for (i += own; i < plan.num_tiles; i += own) a.tilemax[i] = 0.f;
  }
};

// Work group blk of the scatter; a.S a power of two, scatter_in_range(a.B,
// a.S).  Run: phase(fn) and barrier() as for fused_position; ballot() fills the
// threads' masks from their hits, wave_max() makes `max` the wave's, uniform()
// reads a value that all threads hold.
template <int R, class Run>
PTY_HD void scatter_tile(Run& run, const GatherArgs& a, const ScatterPlan& plan, int blk) {
  using K = Scatter<R>;
  using Regs = typename K::Regs;
  const ScatterOrigin t = K::origin(plan, blk);
  if (t.tr >= plan.tiles_x) return;  // uniform over the work group
  const int range = a.B * (a.S * a.S * 8);
  const ScatterBuf ps = scatter_buf(a.ps, range), chi = scatter_buf(a.chi, range);
  run.phase([&](int tid, Regs& r, auto) { K::p_init(tid, a, t, r); });
  for (int seg0 = 0; seg0 < a.B; seg0 += SCATTER_SEG) {
    run.phase([&](int tid, Regs& r, auto) { K::p_test(tid, a, t, seg0, r); });
    run.ballot();
    run.phase([&](int tid, Regs& r, auto sh) { K::p_rank(tid, r, sh); });
    run.barrier();
    run.phase([&](int tid, Regs& r, auto sh) { K::p_list(tid, a, seg0, r, sh); });
    run.barrier();
    const int nh = run.uniform([](const Regs& r) { return r.nh; });
    if (nh > 0) run.phase([&](int tid, Regs& r, auto sh) { K::p_load(tid, a, ps, chi, 0, r, sh); });
    int buf = 0;
    for (int h0 = 0; h0 < nh; h0 += K::CHUNK, buf ^= 1) {
      run.phase([&](int tid, Regs& r, auto sh) {
        K::p_products(tid, buf, r, sh);
        if (h0 + K::CHUNK < nh) K::p_load(tid, a, ps, chi, h0 + K::CHUNK, r, sh);
      });
      // one barrier per chunk: the buffer written now is read until the
      // chunk after next is written, one barrier later
      run.barrier();
      const int m = nh - h0 < K::CHUNK ? nh - h0 : K::CHUNK;
      run.phase([&](int tid, Regs& r, auto sh) { K::p_add(tid, buf, m, r, sh); });
    }
    run.barrier();  // the list and the buffers are free for the next segment
  }
  run.phase([&](int tid, Regs& r, auto) { K::p_store(tid, a, t, r); });
  if (!a.tilemax || (a.run && !a.run_last)) return;
  run.wave_max();
  run.phase([&](int tid, Regs& r, auto sh) {
    if ((tid & 63) == 0) sh.red().st(wave_uniform(tid >> 6), r.max);
  });
  run.barrier();
  run.phase([&](int tid, Regs&, auto sh) { K::p_max(tid, a, plan, t, sh); });
}

}  // namespace pty
