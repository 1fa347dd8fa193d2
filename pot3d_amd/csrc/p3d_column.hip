// D-ILU triangular solves by columns: one launch per sweep.
//
// A column is 8x8 (r, theta) points and all c phi planes; one wave marches it
// (lane = ii + 8 jj): lane (ii,jj) handles plane k = s - ii - 2 jj at step s.
// What a column needs from its lower neighbours in i and j is passed on while
// both are marching, as words {value, stamp} of 8 bytes that the reader polls
// until the stamp is the sweep's own: a word is its own flag, so no fence, no
// counter and no cache write-back or invalidation is needed, and nothing has
// to be cleared between sweeps.
//
// What bounds it: the chain of columns and of steps, until the grid is large
// enough for memory.  The tile schedule pays one launch (about 9 us: load,
// march, drain) per anti-diagonal of tiles, 74 per sweep at 151x301x601; here
// a column starts about 2 us after its neighbour (two chunks of steps, one
// store and one poll) and the 57 diagonals of columns overlap with the march
// along phi (46 ns a step).  FP64 apply without a cut, tiles and columns: 350
// and 100 us at 51x91x181, 1383 and 410 us at 151x301x601, 4.98 and 1.86 ms
// at 301x601x1201 (3.7 TB/s of its 32 bytes per unknown).
//
// Termination: columns are numbered by anti-diagonal, so a column only waits
// for columns of lower workgroup number.  Workgroups start in that order on
// every XCD, so of one launch the lowest unfinished one is always running or
// next to run and never waits for one that is not.  Launches that do not wait
// end by themselves and give their place back.  Two launches of column sweeps
// side by side could keep each other out: one holds the places of one XCD and
// waits for a column on another, whose places the other launch holds likewise.
// So a call claims room for its columns (columns_claim), and takes the tile
// schedules where the device would not hold all that are under way together.
// What is left are other processes on the same device: every wait is bounded
// (kPolls polls, then a flag that ends all other waits), and the solver starts
// the call over with the tile schedules.  P3D_COLUMN_POLLS in the environment
// sets another bound for the plans built from then on (0: a wait gives up once
// it has polled in vain), so that this path can be tested.
//
// Per-point arithmetic and order are those of p3d_sweep.hip: the same bits.
//
// Stored couplings (the legacy CSR input, any values): the same march on x in
// natural order, the three couplings of a point and its pivot inverse as one
// 16-byte word per step and lane, laid out in marching order for each
// direction (32 bytes per unknown instead of the 12 that the couplings and
// dinv take once in natural order, but one coalesced load of 1 KB per step).
// What bounds it: the chain, as above.  One call of the drop-in interface,
// tiles and columns: 333 and 85 us at 20x31x60, 1429 and 167 us at 51x91x181,
// 3448 and 368 us at 101x181x361, 7.06 and 0.87 ms at 151x301x601.
#include <stdlib.h>

#include <mutex>
#include <type_traits>
#include <vector>

#include "p3d_column.hpp"
#include "p3d_kernels.hpp"

namespace p3d {

namespace {

constexpr int kCU = 8;                   // steps per chunk
constexpr int kCP = 4;                   // chunks of loads in flight
constexpr int kFP = 1;                   // chunks of face words asked for ahead
constexpr int kCS = kCU * kCP;           // steps per round of the march loop
constexpr int kJ = 2;                    // steps by which a lane lags its j neighbour
constexpr int kDelay = 7 + 7 * kJ;       // steps between a column's first and last lane
constexpr int kFront = kCS;              // rows before row 0 of dinv_s and y_s
constexpr int kRing = 64;                // steps whose values a column holds in LDS
constexpr int kThreads = 256;            // four waves: march, in, out, faces
constexpr unsigned kPolls = 1u << 20;    // polls of one wait (about a second)

#define P3D_DPP(v, ctrl) __builtin_amdgcn_mov_dpp((v), (ctrl), 0xf, 0xf, true)

__device__ __forceinline__ float bperm(int src_lane4, float v) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute(src_lane4, __float_as_int(v)));
}

typedef unsigned long long u64;
__device__ __forceinline__ u64 word_load(const u64* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void word_store(u64* p, float v, unsigned stamp) {
  __hip_atomic_store(p, ((u64)stamp << 32) | (u64)__float_as_uint(v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

// Workgroup barrier for LDS alone: the global loads and stores in flight are
// not waited for.  The wait is written out (lgkmcnt 0): an LDS-scope release
// fence lost it at the head of the march loop, where the pending writes come
// over the back edge.
__device__ __forceinline__ void lds_barrier() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// A workgroup is one column in four waves: wave 0 marches, wave 1 brings the
// column's rows from memory to LDS, wave 2 takes the results to memory, wave 3
// waits for the neighbours' faces.  A wave's memory operations retire in
// order, so a wave that polled and streamed would wait, at every poll, for
// the rows it has just asked for; and the march, one instruction after the
// other, is what all columns wait for.  One LDS barrier per chunk of steps.
struct ColLds {
  // per step and lane {right-hand side, pivot inverse}, step s in row s mod
  // 64; the march overwrites the right-hand side by its result
  float2 v[kRing][64];
  // incoming faces of two chunks: entry jj {from i, .}, entry 8 + ii {., from
  // j}, entry 0 both
  float2 f[2][kCU][16];
};

// With stored couplings, those of 32 steps besides: (k, j) and i.  Written two
// chunks and read one chunk ahead, so four chunks of rows do.
struct ColLdsStored : ColLds {
  float2 ckj[kCS][64];
  float ci[kCS][64];
};

// Phi factors of the couplings (ColArgs::mode), or the couplings themselves.
enum { kPhiAny = 0, kPhiCut = 1, kPhiUniform = 2, kStored = 3 };

// Offset of plane k of column col in a tile-major vector (TileMap); 32 bits
// hold it (build_column_plan).
__device__ __forceinline__ uint32_t tm_row(const ColArgs& ca, int col, int k) {
  const uint32_t tile = (uint32_t)col + (uint32_t)(ca.NI * ca.NJ) * (uint32_t)(k >> ca.tk_log2);
  return ((tile << ca.tk_log2) + (uint32_t)(k & ((1 << ca.tk_log2) - 1))) * 64u;
}

__device__ __forceinline__ float neg_fma(float a, float b, float c) {
  return __builtin_fmaf(-a, b, c);
}
__device__ __forceinline__ double neg_fma(double a, double b, double c) {
  return __builtin_fma(-a, b, c);
}

template <int P>
using Phase = std::integral_constant<int, P>;

template <typename F>
__device__ __forceinline__ void rounds(int n, F&& f) {
#pragma unroll 1
  for (int it = 0; it < n; it++) {
    f(Phase<0>{}, it * kCP);
    f(Phase<1>{}, it * kCP + 1);
    f(Phase<2>{}, it * kCP + 2);
    f(Phase<3>{}, it * kCP + 3);
  }
}

// What the waves of a column share.
struct ColCtx {
  int lane, ii, jj, dl, wave, col, I, J;
  SweepCoup cp;
  bool act;
  unsigned stamp;
  size_t fbase, sk;  // this column's faces; its row kFront of dinv_s and y_s
};

template <bool kFwd, bool kSt = false>
__device__ __forceinline__ ColCtx col_ctx(const Metric& m, const Grid3& g, const ColArgs& ca) {
  ColCtx x;
  x.lane = threadIdx.x & 63;
  x.ii = x.lane & 7;
  x.jj = x.lane >> 3;
  x.dl = x.ii + kJ * x.jj;
  x.wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  x.col = ca.order[kFwd ? (int)blockIdx.x : (int)gridDim.x - 1 - (int)blockIdx.x];
  x.I = x.col % ca.NI;
  x.J = x.col / ca.NI;
  const int i = x.I * 8 + x.ii, j = x.J * 8 + x.jj;
  x.act = i < g.a && j < g.b;
  if constexpr (kSt)
    x.cp = SweepCoup{};
  else
    x.cp = kFwd ? sweep_coup_lower(m, x.act ? i : 0, x.act ? j : 0)
                : sweep_coup_upper(m, x.act ? i : 0, x.act ? j : 0);
  x.stamp = __hip_atomic_load(ca.ctr + (kFwd ? 0 : 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  x.fbase = (size_t)x.col * ca.face_rows * 8;
  x.sk = ((size_t)x.col * ca.rows_alloc + kFront) * 64;
  return x;
}

// Wave 0, both directions.  Forward (kFwd):
//   y = rhs - aw t_w - ak t_(k-1) - aj t_(j-1) - ai t_(i-1), t = dinv y
// backward, with the mirrored lane and plane order:
//   z = (rhs - bi z_(i+1) - bj z_(j+1) - bk z_(k+1) - bw z_w) dinv
// A lane lags its neighbour in i by one step (handed over by DPP) and the one
// in j by two, so that the hand-over through the LDS crossbar is not on the
// chain of steps.  The inputs of the next chunk are read during this one.
template <bool kFwd, int kMode>
__device__ __forceinline__ void march(const Metric& m, const ColArgs& ca, const ColCtx& x,
                                      ColLds& sh, const float2* pf) {
  constexpr bool kTable = kMode == kPhiAny || kMode == kPhiCut;
  const ColLdsStored& st = (const ColLdsStored&)sh;  // (with kStored only)
  const int lane = x.lane, dly = kFwd ? x.dl : kDelay - x.dl;
  const int nbr = (kFwd ? (lane - 8) & 63 : (lane + 8) & 63) << 2;
  const bool edge_i = x.ii == (kFwd ? 0 : 7), edge_j = x.jj == (kFwd ? 0 : 7);
  // the lane's face entry: its row's for i, its column's for j, the lane on
  // both edges entry 0 (the j faces are numbered from that lane)
  const int fe = edge_i ? (kFwd ? x.jj : 7 - x.jj) : 8 + (kFwd ? x.ii : 7 - x.ii);
  // coupling of the phi wrap
  float wc = 0.f;
  if constexpr (kMode == kStored) {
    if (x.act && ca.bl.wrap)
      wc = (kFwd ? ca.wrap_lo : ca.wrap_up)[x.I * 8 + x.ii + m.a * (x.J * 8 + x.jj)];
  } else {
    if (ca.bl.wrap) wc = x.cp.k * (kFwd ? m.FDPU[m.c - 1] : m.FDPL[0]);
  }
  // first and last plane of the grid, counted in marching order
  const int q_first = kFwd ? 0 : ca.skip, q_last = q_first + ca.c - 1;
  const float2* pfl = pf + (kDelay - dly);
  const float ck0 = x.cp.k * ca.u_k, cj0 = x.cp.j * ca.u_d, ci0 = x.cp.i * ca.u_d;
  float t = 0.f, t_w = 0.f, nj[kJ] = {};  // nj: from the j neighbour, oldest first
  float2 rd[2][kCU], cf[2][kCU];
  float cg[2][kCU];
  lds_barrier();
#pragma unroll
  for (int u = 0; u < kCU; u++) {
    rd[0][u] = sh.v[u][lane];
    if constexpr (kTable) cf[0][u] = pfl[u];
    if constexpr (kMode == kStored) {
      cf[0][u] = st.ckj[u][lane];
      cg[0][u] = st.ci[u][lane];
    }
  }
  rounds(ca.rounds, [&](auto pc, int n) {
    constexpr int p = decltype(pc)::value, q = p & 1;
    const int s0 = n * kCU;
    float2* v = &sh.v[(n & 7) * kCU][lane];
    const float2* vn = &sh.v[((n + 1) & 7) * kCU][lane];
    const float2* pn = pfl + s0 + kCU;
    float2 fc[kCU];
#pragma unroll
    for (int u = 0; u < kCU; u++) fc[u] = sh.f[q][u][fe];
    auto steps = [&](auto ec) {
      constexpr bool kEdge = decltype(ec)::value;
#pragma unroll
      for (int u = 0; u < kCU; u++) {
        const int s = s0 + u;
        const float from_i = __int_as_float(
            kFwd ? P3D_DPP(__float_as_int(t), 0x111) : P3D_DPP(__float_as_int(t), 0x101));
        const float tj = edge_j ? fc[u].y : nj[0], ti = edge_i ? fc[u].x : from_i;
        float ck = ck0, cj = cj0, ci = ci0;
        if constexpr (kMode == kPhiAny) {
          ck = x.cp.k * cf[q][u].y;
          cj = x.cp.j * cf[q][u].x;
          ci = x.cp.i * cf[q][u].x;
        } else if constexpr (kMode == kStored) {
          ck = cf[q][u].x;
          cj = cf[q][u].y;
          ci = cg[q][u];
        } else if constexpr (kMode == kPhiCut) {
          ck = cf[q][u].y == 0.f ? 0.f : ck0;
        }
        const float w = kEdge && s - dly == q_last ? wc : 0.f;
        float y = rd[q][u].x;
        if constexpr (kFwd) {
          if constexpr (kEdge) y = sub_prod(y, w, t_w);
          y = sub_prod(y, ck, t);
          y = sub_prod(y, cj, tj);
          y = sub_prod(y, ci, ti);
          t = rd[q][u].y * y;
        } else {
          y = sub_prod(y, ci, ti);
          y = sub_prod(y, cj, tj);
          y = sub_prod(y, ck, t);
          if constexpr (kEdge) y = sub_prod(y, w, t_w);
          t = y = y * rd[q][u].y;
        }
        if constexpr (kEdge) t_w = s - dly == q_first ? t : t_w;
#pragma unroll
        for (int h = 0; h + 1 < kJ; h++) nj[h] = nj[h + 1];
        nj[kJ - 1] = bperm(nbr, t);
        v[u * 64].x = y;
        rd[1 - q][u] = vn[u * 64];
        if constexpr (kTable) cf[1 - q][u] = pn[u];
        if constexpr (kMode == kStored) {
          cf[1 - q][u] = st.ckj[((p + 1) % kCP) * kCU + u][lane];
          cg[1 - q][u] = st.ci[((p + 1) % kCP) * kCU + u][lane];
        }
      }
    };
    if (s0 <= kDelay + q_first || s0 + kCU >= q_last)
      steps(std::true_type{});
    else
      steps(std::false_type{});
    lds_barrier();
  });
}

// Wave 3: the neighbours' face words, chunk by chunk, 8 rows x 8 words of
// each face (lane = 8 row + entry), asked for kFP chunks ahead.  One is best:
// two or three let the march run through when a poll takes longer than a
// chunk, but a column then starts that many chunks later, and the start of
// 57 columns one after the other weighs more (151x301x601, FP64 apply: 410,
// 456 and 492 us for 1, 2 and 3).
template <bool kFwd>
__device__ __forceinline__ void faces(const ColArgs& ca, const ColCtx& x, ColLds& sh) {
  const bool has_i = kFwd ? x.I > 0 && ca.bl.lo_i(x.I * 8)
                          : x.I + 1 < ca.NI && ca.bl.lo_i((x.I + 1) * 8);
  const bool has_j = kFwd ? x.J > 0 && ca.bl.lo_j(x.J * 8)
                          : x.J + 1 < ca.NJ && ca.bl.lo_j((x.J + 1) * 8);
  const int row = x.lane >> 3, e = x.lane & 7;
  float* fi = &sh.f[0][row][kFwd ? e : 7 - e].x;
  float* fj = &sh.f[0][row][e == (kFwd ? 0 : 7) ? 0 : 8 + (kFwd ? e : 7 - e)].y;
  constexpr int kBuf = kCU * 16 * 2;  // floats of one chunk's faces
  fi[0] = fi[kBuf] = fj[0] = fj[kBuf] = 0.f;
  if (!has_i && !has_j) {
    lds_barrier();
    rounds(ca.rounds, [&](auto, int) { lds_barrier(); });
    return;
  }
  // step s takes the i words of the neighbour's step s + 7, the j words of
  // its step s + 14; an absent face reads (and drops) this column's own
  const size_t fs = (size_t)ca.face_rows * 8;
  const int d = kFwd ? -1 : 1;
  const u64* pi = ca.face_i + (has_i ? x.col + d : x.col) * fs + (kCU + 7) * 8 + x.lane;
  const u64* pj = ca.face_j + (has_j ? x.col + d * ca.NI : x.col) * fs + (kCU + 7 * kJ) * 8 + x.lane;
  const unsigned mi = has_i ? ~0u : 0u, mj = has_j ? ~0u : 0u, stamp = x.stamp;
  unsigned* abort = ca.failed;
  bool dead = false;
  u64 wi[kCP], wj[kCP];
  auto load = [&](int p, int n) {
    wi[p] = word_load(pi + (size_t)n * (kCU * 8));
    wj[p] = word_load(pj + (size_t)n * (kCU * 8));
  };
  auto missing = [&](int p) {
    return ((((unsigned)(wi[p] >> 32) ^ stamp) & mi) | (((unsigned)(wj[p] >> 32) ^ stamp) & mj)) !=
           0u;
  };
  auto get = [&](auto pc, int n) {
    constexpr int p = decltype(pc)::value;
    if (__any(missing(p)) && !dead) {
      unsigned spins = 0;
      do {
        // this chunk and the next ones, which were asked for even earlier
#pragma unroll
        for (int q = 0; q < kFP; q++) load((p + q) % kCP, n + q);
        const bool stop = ++spins >= ca.polls;
        if (stop || (spins & 1023u) == 0) {
          if (stop && x.lane == 0)
            __hip_atomic_store(abort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          if (stop || __hip_atomic_load(abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            dead = true;
        }
      } while (__any(missing(p)) && !dead);
    }
    fi[(p & 1) * kBuf] = __uint_as_float((unsigned)wi[p] & mi);
    fj[(p & 1) * kBuf] = __uint_as_float((unsigned)wj[p] & mj);
    load((p + kFP) % kCP, n + kFP);
  };
#pragma unroll
  for (int p = 0; p < kFP; p++) load(p, p);
  get(Phase<0>{}, 0);
  lds_barrier();
  rounds(ca.rounds, [&](auto pc, int n) {
    if (n + 1 < ca.rounds * kCP) get(Phase<(decltype(pc)::value + 1) % kCP>{}, n + 1);
    lds_barrier();
  });
}

// Wave 1, start: zero right-hand sides, phi factors.
__device__ __forceinline__ void col_lds_init(const ColArgs& ca, ColLds& sh, float2* pf,
                                             const float2* src, int lane) {
#pragma unroll
  for (int t = 0; t < kRing; t++) sh.v[t][lane] = make_float2(0.f, 0.f);
  if (ca.mode == kPhiAny || ca.mode == kPhiCut)
    for (int q = lane; q < ca.pf_n; q += 64) pf[q] = src[q];
}

// Wave 2, forward: the march's results, to the next columns and to y_s.
__device__ __forceinline__ void forward_out(const ColArgs& ca, const ColCtx& x, ColLds& sh) {
  const int lane = x.lane;
  u64* oi = ca.face_i + x.fbase + lane;
  u64* oj = ca.face_j + x.fbase + lane;
  float* ys = ca.y_s + x.sk;
  const int fu = lane >> 3, fe = lane & 7;  // this lane's face row and entry
  // chunk n - 1's results: the faces first, then the rows
  auto out = [&](int n) {
    const int b = ((n - 1) & 7) * kCU;
    const float2 vi = sh.v[b + fu][7 + 8 * fe], vj = sh.v[b + fu][56 + fe];
    float y[kCU];
#pragma unroll
    for (int u = 0; u < kCU; u++) y[u] = sh.v[b + u][lane].x;
    word_store(oi + (size_t)n * (kCU * 8), vi.y * vi.x, x.stamp);
    word_store(oj + (size_t)n * (kCU * 8), vj.y * vj.x, x.stamp);
    float* yo = ys + (ptrdiff_t)(n - 1) * (kCU * 64);
#pragma unroll
    for (int u = 0; u < kCU; u++) yo[u * 64 + lane] = y[u];
  };
  lds_barrier();
  rounds(ca.rounds, [&](auto, int n) {
    out(n);
    lds_barrier();
  });
  const int end = ca.rounds * kCP;
  out(end);
  // the rows that a reader's last steps ask for lie behind the grid
  for (int n = end + 1; n <= end + (7 * kJ + kCU - 1) / kCU; n++) {
    word_store(oi + (size_t)n * (kCU * 8), 0.f, x.stamp);
    word_store(oj + (size_t)n * (kCU * 8), 0.f, x.stamp);
  }
}

// ---------------------------------------------------------------------------
// Forward sweep, y = L^-1 r.  With kUpd r -= alpha ap first, r written back
// (the same fused multiply-add as k_r_update and k_cg_update).
template <typename T, bool kUpd, int kMode>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(3)))
    k_col_fwd(Metric m, Grid3 g, ColArgs ca, T* __restrict__ r, const CgState* guard,
              const T* __restrict__ ap) {
  extern __shared__ char lds[];
  ColLds& sh = *(ColLds*)lds;
  float2* pf = (float2*)(lds + sizeof(ColLds));
  const ColCtx x = col_ctx<true>(m, g, ca);
  const int lane = x.lane;
  if (x.wave == 1) {
    const int kmax = ca.planes;  // planes of the tile-major vectors
    const int last = ca.rounds * kCP - 1;
    // ap in FP64 comes two chunks ahead only: registers for three waves per SIMD
    constexpr int kAP = !kUpd ? 1 : (sizeof(T) == 8 ? 2 : kCP);
    T rv[kCP][kCU], av[kAP][kCU];
    float dv[kCP][kCU];
    // past the vector's planes: its last ones (pivot 0 there, not used)
    auto row = [&](int n) { return tm_row(ca, x.col, min(n * kCU, kmax - kCU)); };
    auto load = [&](int p, int n) {
      const T* rb = r + row(n);
      const float* d = ca.dinv_s + x.sk + (size_t)min(n, last) * (kCU * 64);
#pragma unroll
      for (int u = 0; u < kCU; u++) {
        rv[p][u] = rb[u * 64 + lane];
        dv[p][u] = d[u * 64 + lane];
      }
    };
    auto load_a = [&](int p, int n) {
      const T* ab = ap + row(n);
#pragma unroll
      for (int u = 0; u < kCU; u++) av[p][u] = ab[u * 64 + lane];
    };
#pragma unroll
    for (int p = 0; p < kCP; p++) load(p, p);
    if constexpr (kUpd) {
#pragma unroll
      for (int p = 0; p < kAP; p++) load_a(p, p);
    }
    const T alpha = kUpd ? (T)st_load(&guard->alpha) : (T)0;
    col_lds_init(ca, sh, pf, ca.pf_lo, lane);
    if (guard && st_done(guard)) return;
    // chunk n's inputs to LDS (n = phase p mod kCP): row q of r to step q + dl
    auto put = [&](auto pc, int n) {
      constexpr int p = decltype(pc)::value;
      T v[kCU];
      float2* d = &sh.v[(n & 7) * kCU][lane];
      const int o = (n & 7) * kCU + x.dl;
#pragma unroll
      for (int u = 0; u < kCU; u++) {
        v[u] = rv[p][u];
        if constexpr (kUpd) v[u] = neg_fma(alpha, av[p % kAP][u], v[u]);
        sh.v[(o + u) & (kRing - 1)][lane].x = (float)v[u];
        d[u * 64].y = dv[p][u];
      }
      if constexpr (kUpd) {
        const bool in = n * kCU < kmax;
        T* ro = (in ? r : (T*)ca.dummy) + (in ? tm_row(ca, x.col, n * kCU) : 0u);
#pragma unroll
        for (int u = 0; u < kCU; u++) ro[u * 64 + lane] = v[u];
        load_a(p % kAP, n + kAP);
      }
      load(p, n + kCP);
    };
    put(Phase<0>{}, 0);
    put(Phase<1>{}, 1);
    lds_barrier();
    rounds(ca.rounds, [&](auto pc, int n) {
      put(Phase<(decltype(pc)::value + 2) % kCP>{}, n + 2);
      lds_barrier();
    });
    return;
  }
  if (guard && st_done(guard)) return;
  if (x.wave == 0) {
    // the backward sweep's stamp (no workgroup of this launch reads it)
    if (blockIdx.x == 0 && lane == 0)
      __hip_atomic_store(ca.ctr + 1, x.stamp + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    march<true, kMode>(m, ca, x, sh, pf);
  } else if (x.wave == 3) {
    faces<true>(ca, x, sh);
  } else {
    forward_out(ca, x, sh);
  }
}

// Wave 2, backward: the march's results to the next columns, and the planes
// that a chunk completes, k downwards (lane dl finished plane top - s at step
// s - dl), to store(k, values); what lies outside the grid stays zero.
template <typename F>
__device__ __forceinline__ void backward_out(const ColArgs& ca, const ColCtx& x, ColLds& sh,
                                             F&& store) {
  const int lane = x.lane, top = ca.c + ca.skip + kDelay - 1;
  u64* oi = ca.face_i + x.fbase + lane;
  u64* oj = ca.face_j + x.fbase + lane;
  const int fu = lane >> 3, fe = lane & 7;
  auto out = [&](int n) {
    const int b = ((n - 1) & 7) * kCU;
    const float ti = sh.v[b + fu][8 * fe].x, tj = sh.v[b + fu][fe].x;
    float y[kCU];
#pragma unroll
    for (int u = 0; u < kCU; u++) y[u] = sh.v[(b + u - x.dl) & (kRing - 1)][lane].x;
    word_store(oi + (size_t)n * (kCU * 8), ti, x.stamp);
    word_store(oj + (size_t)n * (kCU * 8), tj, x.stamp);
    store(top - (n - 1) * kCU, y);
  };
  lds_barrier();
  rounds(ca.rounds, [&](auto, int n) {
    out(n);
    lds_barrier();
  });
  const int end = ca.rounds * kCP;
  out(end);
  for (int n = end + 1; n <= end + (7 * kJ + kCU - 1) / kCU; n++) {
    word_store(oi + (size_t)n * (kCU * 8), 0.f, x.stamp);
    word_store(oj + (size_t)n * (kCU * 8), 0.f, x.stamp);
  }
}

// ---------------------------------------------------------------------------
// Backward sweep, z = U^-1 y: the forward sweep mirrored.  At step s lane
// (ii,jj) handles the plane s - (21 - ii - 2 jj) counted from plane c + skip
// - 1 downwards, row c + skip + 20 - s of dinv_s and y_s; skip makes a chunk's
// finished planes 8 planes of one tile.
template <typename T, int kMode>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(3)))
    k_col_bwd(Metric m, Grid3 g, ColArgs ca, T* __restrict__ z, const CgState* guard) {
  extern __shared__ char lds[];
  ColLds& sh = *(ColLds*)lds;
  float2* pf = (float2*)(lds + sizeof(ColLds));
  const ColCtx x = col_ctx<false>(m, g, ca);
  const int lane = x.lane, top = ca.c + ca.skip + kDelay - 1;  // row of step 0
  if (x.wave == 1) {
    float yv[kCP][kCU], dv[kCP][kCU];
    const int last = ca.rounds * kCP - 1;
    const size_t s0 = x.sk + (size_t)top * 64;
    auto load = [&](int p, int n) {
      const size_t o = s0 - (size_t)min(n, last) * (kCU * 64);
      const float* y = ca.y_s + o;
      const float* d = ca.dinv_s + o;
#pragma unroll
      for (int u = 0; u < kCU; u++) {
        yv[p][u] = y[-u * 64 + lane];
        dv[p][u] = d[-u * 64 + lane];
      }
    };
#pragma unroll
    for (int p = 0; p < kCP; p++) load(p, p);
    col_lds_init(ca, sh, pf, ca.pf_up, lane);
    if (guard && st_done(guard)) return;
    auto put = [&](auto pc, int n) {
      constexpr int p = decltype(pc)::value;
      float2* d = &sh.v[(n & 7) * kCU][lane];
      // y_s outside the grid is whatever the march made of what it met there
      // (a NaN, next to an overflow)
      const int k0 = top - n * kCU - x.dl;
#pragma unroll
      for (int u = 0; u < kCU; u++)
        d[u * 64] = make_float2(x.act && (unsigned)(k0 - u) < (unsigned)ca.c ? yv[p][u] : 0.f,
                                dv[p][u]);
      load(p, n + kCP);
    };
    put(Phase<0>{}, 0);
    put(Phase<1>{}, 1);
    lds_barrier();
    rounds(ca.rounds, [&](auto pc, int n) {
      put(Phase<(decltype(pc)::value + 2) % kCP>{}, n + 2);
      lds_barrier();
    });
    return;
  }
  if (guard && st_done(guard)) return;
  if (x.wave == 0) {
    // the next forward sweep's stamp
    if (blockIdx.x == 0 && lane == 0)
      __hip_atomic_store(ca.ctr, x.stamp + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    march<false, kMode>(m, ca, x, sh, pf);
  } else if (x.wave == 3) {
    faces<false>(ca, x, sh);
  } else {
    backward_out(ca, x, sh, [&](int k, const float* y) {
      const bool in = k >= 0 && k < ca.planes;
      T* zo = (in ? z : (T*)ca.dummy) + (in ? tm_row(ca, x.col, k - (kCU - 1)) : 0u);
#pragma unroll
      for (int u = 0; u < kCU; u++)
        zo[(kCU - 1 - u) * 64 + lane] = (T)(x.act && k - u < ca.c ? y[u] : 0.f);
    });
  }
}

// ---------------------------------------------------------------------------
// The sweeps with stored couplings: x in natural order, solved in place.
// lo_s and up_s hold {k, j, i coupling, dinv} by step of the direction's own
// march.  The forward sweep keeps the right-hand side as it uses it (FP32,
// natural order): what the tile schedule starts from when a wait runs out.
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
    k_col_fwd_stored(Grid3 g, ColArgs ca, const double* __restrict__ xv, float* __restrict__ r32) {
  extern __shared__ char lds[];
  ColLdsStored& sh = *(ColLdsStored*)lds;
  Metric m{};
  m.a = g.a;
  const ColCtx x = col_ctx<true, true>(m, g, ca);
  if (x.wave == 1) {
    const int lane = x.lane, last = ca.rounds * kCP - 1;
    const size_t base = x.act ? (size_t)(x.I * 8 + x.ii) + (size_t)g.a * (x.J * 8 + x.jj) : 0;
    const float4* cs = ca.lo_s + (size_t)x.col * ca.rounds * (kCS * 64) + lane;
    constexpr int kAP = 2;  // chunks of couplings in flight: registers
    double rv[kCP][kCU];
    float4 cv[kAP][kCU];
    auto load = [&](int p, int n) {
#pragma unroll
      for (int u = 0; u < kCU; u++)
        rv[p][u] = xv[base + (size_t)g.ab * (size_t)min(n * kCU + u, ca.c - 1)];
    };
    auto load_c = [&](int p, int n) {
      const float4* c = cs + (size_t)min(n, last) * (kCU * 64);
#pragma unroll
      for (int u = 0; u < kCU; u++) cv[p][u] = c[u * 64];
    };
#pragma unroll
    for (int p = 0; p < kCP; p++) load(p, p);
#pragma unroll
    for (int p = 0; p < kAP; p++) load_c(p, p);
    col_lds_init(ca, sh, nullptr, nullptr, lane);
    auto put = [&](auto pc, int n) {
      constexpr int p = decltype(pc)::value;
      const int o = (n & 7) * kCU + x.dl;
#pragma unroll
      for (int u = 0; u < kCU; u++) {
        const int k = n * kCU + u;
        const bool in = x.act && k < ca.c;
        const float v = in ? (float)rv[p][u] : 0.f;
        sh.v[(o + u) & (kRing - 1)][lane].x = v;
        if (in) r32[base + (size_t)g.ab * k] = v;
        const float4 c = cv[p % kAP][u];
        sh.v[(n & 7) * kCU + u][lane].y = c.w;
        sh.ckj[p * kCU + u][lane] = make_float2(c.x, c.y);
        sh.ci[p * kCU + u][lane] = c.z;
      }
      load_c(p % kAP, n + kAP);
      load(p, n + kCP);
    };
    put(Phase<0>{}, 0);
    put(Phase<1>{}, 1);
    lds_barrier();
    rounds(ca.rounds, [&](auto pc, int n) {
      put(Phase<(decltype(pc)::value + 2) % kCP>{}, n + 2);
      lds_barrier();
    });
  } else if (x.wave == 0) {
    // the backward sweep's stamp (no workgroup of this launch reads it)
    if (blockIdx.x == 0 && x.lane == 0)
      __hip_atomic_store(ca.ctr + 1, x.stamp + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    march<true, kStored>(m, ca, x, sh, nullptr);
  } else if (x.wave == 3) {
    faces<true>(ca, x, sh);
  } else {
    forward_out(ca, x, sh);
  }
}

__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
    k_col_bwd_stored(Grid3 g, ColArgs ca, double* __restrict__ xv) {
  extern __shared__ char lds[];
  ColLdsStored& sh = *(ColLdsStored*)lds;
  Metric m{};
  m.a = g.a;
  const ColCtx x = col_ctx<false, true>(m, g, ca);
  const int top = ca.c + ca.skip + kDelay - 1;  // row of step 0
  if (x.wave == 1) {
    const int lane = x.lane, last = ca.rounds * kCP - 1;
    const float4* cs = ca.up_s + (size_t)x.col * ca.rounds * (kCS * 64) + lane;
    const float* ys = ca.y_s + x.sk + (size_t)top * 64 + lane;
    constexpr int kAP = 2;
    float yv[kCP][kCU];
    float4 cv[kAP][kCU];
    auto load = [&](int p, int n) {
      const float* y = ys - (ptrdiff_t)min(n, last) * (kCU * 64);
#pragma unroll
      for (int u = 0; u < kCU; u++) yv[p][u] = y[-u * 64];
    };
    auto load_c = [&](int p, int n) {
      const float4* c = cs + (size_t)min(n, last) * (kCU * 64);
#pragma unroll
      for (int u = 0; u < kCU; u++) cv[p][u] = c[u * 64];
    };
#pragma unroll
    for (int p = 0; p < kCP; p++) load(p, p);
#pragma unroll
    for (int p = 0; p < kAP; p++) load_c(p, p);
    col_lds_init(ca, sh, nullptr, nullptr, lane);
    auto put = [&](auto pc, int n) {
      constexpr int p = decltype(pc)::value;
      const int k0 = top - n * kCU - x.dl;
#pragma unroll
      for (int u = 0; u < kCU; u++) {
        const bool in = x.act && (unsigned)(k0 - u) < (unsigned)ca.c;
        const float4 c = cv[p % kAP][u];
        sh.v[(n & 7) * kCU + u][lane] = make_float2(in ? yv[p][u] : 0.f, c.w);
        sh.ckj[p * kCU + u][lane] = make_float2(c.x, c.y);
        sh.ci[p * kCU + u][lane] = c.z;
      }
      load_c(p % kAP, n + kAP);
      load(p, n + kCP);
    };
    put(Phase<0>{}, 0);
    put(Phase<1>{}, 1);
    lds_barrier();
    rounds(ca.rounds, [&](auto pc, int n) {
      put(Phase<(decltype(pc)::value + 2) % kCP>{}, n + 2);
      lds_barrier();
    });
  } else if (x.wave == 0) {
    // the next forward sweep's stamp
    if (blockIdx.x == 0 && x.lane == 0)
      __hip_atomic_store(ca.ctr, x.stamp + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    march<false, kStored>(m, ca, x, sh, nullptr);
  } else if (x.wave == 3) {
    faces<false>(ca, x, sh);
  } else {
    const size_t base = x.act ? (size_t)(x.I * 8 + x.ii) + (size_t)g.a * (x.J * 8 + x.jj) : 0;
    backward_out(ca, x, sh, [&](int k, const float* y) {
#pragma unroll
      for (int u = 0; u < kCU; u++)
        if (x.act && (unsigned)(k - u) < (unsigned)ca.c)
          xv[base + (size_t)g.ab * (size_t)(k - u)] = (double)y[u];
    });
  }
}

// dinv (natural order) -> skewed columns: row kFront + k + ii + 2 jj of column
// (I, J), zero where no point of the grid lies.
__global__ void k_col_gather(Grid3 g, int NI, int rows_alloc, size_t n,
                             const float* __restrict__ src, float* __restrict__ dst) {
  const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= n) return;
  const int lane = (int)(t & 63);
  const size_t cr = t >> 6;
  const int row = (int)(cr % (size_t)rows_alloc), col = (int)(cr / (size_t)rows_alloc);
  const int i = (col % NI) * 8 + (lane & 7), j = (col / NI) * 8 + (lane >> 3);
  const int k = row - kFront - (lane & 7) - kJ * (lane >> 3);
  dst[t] = (i < g.a && j < g.b && k >= 0 && k < g.c)
               ? src[(size_t)i + (size_t)g.a * j + (size_t)g.ab * k]
               : 0.f;
}

// The couplings and dinv of one direction by step of its march: entry s of
// column (I, J) belongs to the plane that lane (ii, jj) handles at step s,
// zero where no point of the grid lies (and for what the point does not have).
__global__ void k_col_gather_stored(Grid3 g, int NI, int steps, int top, size_t n,
                                    const float* __restrict__ ck, const float* __restrict__ cj,
                                    const float* __restrict__ ci, const float* __restrict__ dinv,
                                    int fwd, float4* __restrict__ dst) {
  const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= n) return;
  const int lane = (int)(t & 63);
  const size_t cr = t >> 6;
  const int s = (int)(cr % (size_t)steps), col = (int)(cr / (size_t)steps);
  const int i = (col % NI) * 8 + (lane & 7), j = (col / NI) * 8 + (lane >> 3);
  const int dl = (lane & 7) + kJ * (lane >> 3), k = fwd ? s - dl : top - s - dl;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  if (i < g.a && j < g.b && k >= 0 && k < g.c) {
    const size_t q = (size_t)i + (size_t)g.a * j + (size_t)g.ab * k;
    v = make_float4((fwd ? k > 0 : k < g.c - 1) ? ck[q] : 0.f,
                    (fwd ? j > 0 : j < g.b - 1) ? cj[q] : 0.f,
                    (fwd ? i > 0 : i < g.a - 1) ? ci[q] : 0.f, dinv[q]);
  }
  dst[t] = v;
}

// Room taken by the column sweeps under way, by device.
constexpr int kDevices = 64;
std::mutex room_mutex;
long room_used[kDevices] = {};

// Places that a launch of n columns may need: it goes round the 8 XCDs, so one
// XCD gets (n + 7) / 8 of them at most.
long room_of(int n) { return (long)n + 7; }

size_t col_lds(const ColArgs& ca) {
  if (ca.mode == kStored) return sizeof(ColLdsStored);
  return sizeof(ColLds) + (ca.mode == kPhiUniform ? 0 : ca.pf_n * sizeof(float2));
}

template <typename T, int kMode>
void launch_columns(const ColArgs& ca, const Metric& m, const Grid3& g, T* r, T* z,
                    const CgState* guard, const T* ap, hipStream_t s) {
  const size_t lds = col_lds(ca);
  const int nb = ca.NI * ca.NJ;
  if (ap)
    k_col_fwd<T, true, kMode><<<nb, kThreads, lds, s>>>(m, g, ca, r, guard, ap);
  else
    k_col_fwd<T, false, kMode><<<nb, kThreads, lds, s>>>(m, g, ca, r, guard, nullptr);
  k_col_bwd<T, kMode><<<nb, kThreads, lds, s>>>(m, g, ca, z, guard);
}

}  // namespace

namespace {

// What both kinds of plan share: the columns and steps of the grid, and the
// device memory that does not depend on where the couplings come from.
// Returns 0, or 1 when a buffer cannot be had (the caller frees the plan).
int plan_columns(ColumnPlan& plan, const Grid3& g, const IluBlocks& bl, int planes,
                 unsigned* failed) {
  ColArgs& ca = plan.a;
  if (hipGetDevice(&plan.dev) != hipSuccess ||
      hipDeviceGetAttribute(&plan.ncu, hipDeviceAttributeMultiprocessorCount, plan.dev) !=
          hipSuccess)
    return 1;
  const char* polls = getenv("P3D_COLUMN_POLLS");
  ca.polls = polls && *polls ? (unsigned)strtoul(polls, nullptr, 10) : kPolls;
  ca.NI = (g.a + 7) / 8;
  ca.NJ = (g.b + 7) / 8;
  ca.c = g.c;
  ca.planes = planes;
  ca.bl = bl;
  ca.skip = (kCU - 1 - (g.c + kDelay - 1)) & (kCU - 1);
  ca.rounds = (g.c + ca.skip + kDelay + kCS - 1) / kCS;
  ca.rows_alloc = kFront + ca.rounds * kCS;
  ca.face_rows = (ca.rounds * kCP + kCP + 6) * kCU;  // from chunk -1 on
  ca.pf_n = ca.rounds * kCS + kCU + kDelay;
  const int ncol = ca.NI * ca.NJ;
  const size_t nsk = (size_t)ncol * ca.rows_alloc * 64, nf = (size_t)ncol * ca.face_rows * 8;
  // columns by anti-diagonal inside their block (blocks are independent)
  const int bI = bl.bi < g.a ? bl.bi / 8 : ca.NI, bJ = bl.bj < g.b ? bl.bj / 8 : ca.NJ;
  std::vector<int> order;
  order.reserve(ncol);
  for (int L = 0; L <= bI + bJ - 2; L++)
    for (int J = 0; J < ca.NJ; J++)
      for (int I = 0; I < ca.NI; I++)
        if (I % bI + J % bJ == L) order.push_back(I + ca.NI * J);
  const unsigned ctr[4] = {1u, 2u, 0u, 0u};
  const bool ok =
      hipMalloc((void**)&plan.order, ncol * sizeof(int)) == hipSuccess &&
      hipMalloc((void**)&plan.y_s, nsk * sizeof(float)) == hipSuccess &&
      hipMalloc((void**)&plan.face, 2 * nf * sizeof(u64)) == hipSuccess &&
      hipMalloc((void**)&plan.ctr, sizeof ctr) == hipSuccess &&
      hipMalloc((void**)&plan.dummy, kCU * 64 * sizeof(double)) == hipSuccess &&
      hipMemset(plan.y_s, 0, nsk * sizeof(float)) == hipSuccess &&
      hipMemset(plan.face, 0, 2 * nf * sizeof(u64)) == hipSuccess &&
      hipMemcpy(plan.order, order.data(), ncol * sizeof(int), hipMemcpyHostToDevice) ==
          hipSuccess &&
      hipMemcpy(plan.ctr, ctr, sizeof ctr, hipMemcpyHostToDevice) == hipSuccess;
  ca.order = plan.order;
  ca.y_s = plan.y_s;
  ca.face_i = plan.face;
  ca.face_j = plan.face + nf;
  ca.ctr = plan.ctr;
  ca.failed = failed ? failed : plan.ctr + 2;
  ca.dummy = plan.dummy;
  return ok ? 0 : 1;
}

int no_plan(ColumnPlan& plan) {
  free_column_plan(plan);
  (void)hipGetLastError();  // a failed allocation: the tile schedules run
  return 1;
}

}  // namespace

// A single launch needs no room of its own (see the head of this file).  Beside
// others it has to fit at two columns per CU: two fit whatever their kernels
// (kColLdsMax of 160 KB of LDS each, 256 registers at most, one wave per SIMD),
// so a column that finds no place finds at least that many resident on every CU
// of its XCD.
extern "C" int p3d_columns_claim(int dev, int ncol, int ncu) {
  if (dev < 0 || dev >= kDevices) return 0;
  std::lock_guard<std::mutex> lock(room_mutex);
  long& used = room_used[dev];
  if (used > 0 && used + room_of(ncol) > 2L * ncu) return 0;
  used += room_of(ncol);
  return 1;
}

extern "C" void p3d_columns_release(int dev, int ncol) {
  std::lock_guard<std::mutex> lock(room_mutex);
  room_used[dev] -= room_of(ncol);
}

bool ColumnUse::claim(const ColumnPlan& plan) {
  release();
  if (!plan.ready || !p3d_columns_claim(plan.dev, plan.a.NI * plan.a.NJ, plan.ncu)) return false;
  dev = plan.dev;
  ncol = plan.a.NI * plan.a.NJ;
  return true;
}

void ColumnUse::release() {
  if (ncol) p3d_columns_release(dev, ncol);
  ncol = 0;
}

int build_column_plan(ColumnPlan& plan, const Metric& m, const Grid3& g, const IluBlocks& bl,
                      int tk_log2, const float* dinv, unsigned* failed) {
  free_column_plan(plan);
  ColArgs& ca = plan.a;
  ca.tk_log2 = tk_log2;
  const int TK = 1 << tk_log2, planes = (g.c + TK - 1) / TK * TK;
  if ((uint64_t)((g.a + 7) / 8) * ((g.b + 7) / 8) * planes * 64 >= (1ull << 32)) return 1;
  if ((bl.bi < g.a && bl.bi % 8) || (bl.bj < g.b && bl.bj % 8)) return 2;
  // phi factors by plane, zero outside the grid; a coupling that the
  // block-Jacobi cut drops has a zero factor
  std::vector<float> dph(g.c), dpl(g.c), dpu(g.c);
  if (hipMemcpy(dph.data(), m.FDPH, g.c * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess ||
      hipMemcpy(dpl.data(), m.FDPL, g.c * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess ||
      hipMemcpy(dpu.data(), m.FDPU, g.c * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess)
    return 1;
  // phi factors that are all equal need no table (the usual, uniform mesh),
  // or only the planes where the cut drops the coupling in k
  bool uniform = true;
  for (int k = 0; k < g.c; k++)
    uniform = uniform && dph[k] == dph[0] && dpl[k] == dpl[0] && dpu[k] == dpl[0];
  ca.mode = !uniform ? kPhiAny : (bl.bk < g.c ? kPhiCut : kPhiUniform);
  ca.u_d = dph[0];
  ca.u_k = dpl[0];
  if (plan_columns(plan, g, bl, planes, failed) != 0) return no_plan(plan);
  if (col_lds(ca) > kColLdsMax) return no_plan(plan);
  std::vector<float2> lo(ca.pf_n, make_float2(0.f, 0.f)), up(lo);
  for (int k = 0; k < g.c; k++) {
    lo[kDelay + k] = make_float2(dph[k], k > 0 && k % bl.bk ? dpl[k] : 0.f);
    up[kDelay + ca.skip + g.c - 1 - k] =
        make_float2(dph[k], k < g.c - 1 && (k + 1) % bl.bk ? dpu[k] : 0.f);
  }
  const size_t nsk = (size_t)ca.NI * ca.NJ * ca.rows_alloc * 64;
  if (hipMalloc((void**)&plan.dinv_s, nsk * sizeof(float)) != hipSuccess ||
      hipMalloc((void**)&plan.pf, 2 * ca.pf_n * sizeof(float2)) != hipSuccess)
    return no_plan(plan);
  k_col_gather<<<(unsigned)((nsk + 255) / 256), 256>>>(g, ca.NI, ca.rows_alloc, nsk, dinv,
                                                       plan.dinv_s);
  if (hipGetLastError() != hipSuccess ||
      hipMemcpy(plan.pf, lo.data(), ca.pf_n * sizeof(float2), hipMemcpyHostToDevice) !=
          hipSuccess ||
      hipMemcpy(plan.pf + ca.pf_n, up.data(), ca.pf_n * sizeof(float2), hipMemcpyHostToDevice) !=
          hipSuccess ||
      hipDeviceSynchronize() != hipSuccess)
    return no_plan(plan);
  ca.dinv_s = plan.dinv_s;
  ca.pf_lo = plan.pf;
  ca.pf_up = plan.pf + ca.pf_n;
  plan.ready = 1;
  return 0;
}

int build_column_plan_stored(ColumnPlan& plan, const Grid3& g, const CoefArrays& co, bool wrap,
                             const float* dinv) {
  free_column_plan(plan);
  ColArgs& ca = plan.a;
  ca.mode = kStored;
  if (plan_columns(plan, g, IluBlocks{g.a, g.b, g.c, wrap ? 1 : 0}, g.c, nullptr) != 0)
    return no_plan(plan);
  const int steps = ca.rounds * kCS;
  const size_t n = (size_t)ca.NI * ca.NJ * steps * 64;
  if (hipMalloc((void**)&plan.cs, 2 * n * sizeof(float4)) != hipSuccess) return no_plan(plan);
  const int top = ca.c + ca.skip + kDelay - 1;
  const unsigned nb = (unsigned)((n + 255) / 256);
  k_col_gather_stored<<<nb, 256>>>(g, ca.NI, steps, top, n, co.lo_k, co.lo_j, co.lo_i, dinv, 1,
                                   plan.cs);
  k_col_gather_stored<<<nb, 256>>>(g, ca.NI, steps, top, n, co.up_k, co.up_j, co.up_i, dinv, 0,
                                   plan.cs + n);
  if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess)
    return no_plan(plan);
  ca.lo_s = plan.cs;
  ca.up_s = plan.cs + n;
  ca.wrap_lo = co.wrap_lo;
  ca.wrap_up = co.wrap_up;
  plan.ready = 1;
  return 0;
}

void free_column_plan(ColumnPlan& plan) {
  void* bufs[] = {plan.order, plan.dinv_s, plan.y_s, plan.face, plan.pf, plan.ctr, plan.dummy, plan.cs};
  for (void* b : bufs)
    if (b) hipFree(b);
  plan = ColumnPlan();
}

template <typename T>
void launch_dilu_columns(const ColumnPlan& plan, const Metric& m, const Grid3& g, T* r, T* z,
                         const CgState* guard, const T* ap, hipStream_t s) {
  const ColArgs& ca = plan.a;
  if (ca.mode == kPhiUniform)
    launch_columns<T, kPhiUniform>(ca, m, g, r, z, guard, ap, s);
  else if (ca.mode == kPhiCut)
    launch_columns<T, kPhiCut>(ca, m, g, r, z, guard, ap, s);
  else
    launch_columns<T, kPhiAny>(ca, m, g, r, z, guard, ap, s);
}

void launch_dilu_columns_stored(const ColumnPlan& plan, const Grid3& g, double* x, float* r32,
                                hipStream_t s) {
  const ColArgs& ca = plan.a;
  const int nb = ca.NI * ca.NJ;
  k_col_fwd_stored<<<nb, kThreads, sizeof(ColLdsStored), s>>>(g, ca, x, r32);
  k_col_bwd_stored<<<nb, kThreads, sizeof(ColLdsStored), s>>>(g, ca, x);
}

const unsigned* column_failure_flag(const ColumnPlan& plan) { return plan.ctr + 2; }

template void launch_dilu_columns<double>(const ColumnPlan&, const Metric&, const Grid3&, double*,
                                          double*, const CgState*, const double*, hipStream_t);
template void launch_dilu_columns<float>(const ColumnPlan&, const Metric&, const Grid3&, float*,
                                         float*, const CgState*, const float*, hipStream_t);

}  // namespace p3d
