// chain.hip - the Omega weight-update chain of one parameter in one pass each way (gfx950): the loop
// body of atlas_pytorch/omega.py:254-322 over [BH, n, P] surprises, per column of P
//     m_0,t = a_0,t m_0,t-1 + s_t ;  m_o,t = a_o,t m_o,t-1 + m_o-1,t        (momentum orders)
//     x_t   = gate_t m_last,t ;      u_t = sum_{j<e} x_{t-j} (x_{-1-j}: the carried buffer)
//     c_t   = (1 - decay_t) c_{t-1} + u_t ,  c_{-1} = last_update           (update = [c_{-1}; c_0 ..])
// with update = 0 when every gate of the batch is below 1e-3 (the sums above are then still formed for
// the carried momentum and buffer).
//
// Bound: HBM. The separate scans, products, window sums and copies moved about 30 tensors of [BH, n, P]
// per forward + backward in 32 launches; here the forward reads the surprises and writes the updates
// (and, when a backward follows, the momenta and a second copy of the updates), the backward reads dupdate,
// that copy and the momenta and writes dsurprise. One wave owns 64 * V columns of one row and walks n with every
// recurrence in registers. The operands of the kU = 8 steps ahead are in flight: per wave 4 KB (fp32, V = 2; bf16
// half) in the forward, 12 KB (order 2: 16) in the backward.
// What the walk leaves out of a step, since one wave to a SIMD issues it alone where BH * P is small: no load whose
// value outlives a branch and no store under a condition (the wave would wait there for every access in flight),
// addresses are a wave-uniform pointer and a fixed lane offset, and eight steps' sums over the lanes are formed
// together (sums8). 16 x 64 x 8192 fp32, order 1: backward 48 -> 26.4 us, 5.1 TB/s, forward 24.6, 5.4 TB/s; 1 x 4096 x 64
// of order 0 without gate or window, where the separate scans took 1012 us forward and backward: 1428 -> 831.
// The scalars' gradients are dot products over P: each wave leaves its columns' sums as a partial and a second launch
// adds the partials in a fixed order (no atomics: bitwise reproducible).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/atlas_mem.h"
#include "mem_common.h"

namespace atlas {
namespace chain {

constexpr int kMaxOrder = 2;
constexpr int kMaxWin = 16;
constexpr int kU = 8;               // steps per load group
constexpr float kGateOff = 1e-3f;   // omega.py:311

template <typename T>
struct Args {
  int n, bh, e;
  int64_t p;
  const T *s, *decay, *last, *am, *lm0, *gate, *buf;   // am [O, bh, n], lm0 [O, bh, p], buf [bh, e-1, p]
  T *update, *moms, *lm1, *buf1;                       // forward outputs (moms null: no backward follows)
  T *kept, *kdecay;                                    // copies of update and decay for the backward (null: none)
  const T *dup, *dlm1, *dbuf1;                         // backward: gradients of the outputs (null: zero)
  const T *upd;                                        // backward: the forward's update
  const T *msrc;                                       // backward: the momenta (order 0: unused)
  T *ds, *dlast, *dlm0, *dbuf;                         // dbuf null: not wanted
  float *part;                                         // [bh, nblk, K, n], K = 1 (decay) + O + 1 (gate)
};

// V elements at a wave-uniform address plus the lane's byte offset.
template <typename T, int V>
__device__ __forceinline__ void ldv(const T* p, uint32_t lo, float* v) {
  typedef T vt __attribute__((ext_vector_type(V)));
  const char* q = reinterpret_cast<const char*>(p) + lo;
  if constexpr (V == 1) {
    v[0] = to_f32(*reinterpret_cast<const T*>(q));
  } else {
    const vt u = *reinterpret_cast<const vt*>(q);
#pragma unroll
    for (int i = 0; i < V; ++i) v[i] = to_f32(u[i]);
  }
}
template <typename T, int V>
__device__ __forceinline__ void stv(T* p, uint32_t lo, const float* v) {
  typedef T vt __attribute__((ext_vector_type(V)));
  char* q = reinterpret_cast<char*>(p) + lo;
  if constexpr (V == 1) {
    *reinterpret_cast<T*>(q) = from_f32<T>(v[0]);
  } else {
    vt u;
#pragma unroll
    for (int i = 0; i < V; ++i) u[i] = from_f32<T>(v[i]);
    *reinterpret_cast<vt*>(q) = u;
  }
}
__device__ __forceinline__ float lane_of(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
// The sums over the 64 lanes of eight values: lanes exchange halves of them (quad permutations), add up within their
// row (rotations) and across the rows (the swaps of 32 and of 16 lanes), 27 instructions instead of the 6 dependent
// ones of a sum each. Lane l returns the sum of value 4 (l & 1) + (l & 2) + (l >> 5).
__device__ __forceinline__ float sums8(const float (&v)[8]) {
  const int l = lane_id();
  const bool b0 = l & 1, b1 = l & 2;
  float w[4], x[2];
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = (b0 ? v[i + 4] : v[i]) + dpp<0xb1>(b0 ? v[i] : v[i + 4]);
#pragma unroll
  for (int i = 0; i < 2; ++i) x[i] = (b1 ? w[i + 2] : w[i]) + dpp<0x4e>(b1 ? w[i] : w[i + 2]);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    x[i] += dpp<0x128>(x[i]);   // row_ror 8, 4
    x[i] += dpp<0x124>(x[i]);
  }
  const auto h = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, x[0]), __builtin_bit_cast(unsigned, x[1]), false, false);
  const float y = __builtin_bit_cast(float, (unsigned)h[0]) + __builtin_bit_cast(float, (unsigned)h[1]);
  const auto q = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, y), __builtin_bit_cast(unsigned, y), false, false);
  return __builtin_bit_cast(float, (unsigned)q[0]) + __builtin_bit_cast(float, (unsigned)q[1]);
}
__device__ __forceinline__ int sums8_value(int l) { return 4 * (l & 1) + (l & 2) + (l >> 5); }

// Every gate of the batch below the threshold (a NaN is not). The first 64 gates settle it for any
// memory that is in use; all of them are read only when the chunk is really switched off.
template <typename T>
__device__ __forceinline__ bool gates_off(const T* gate, int64_t count) {
  if (!gate) return false;
  for (int64_t i0 = 0; i0 < count; i0 += 64) {
    const int64_t i = i0 + lane_id();
    const bool on = i < count && !(to_f32(gate[i]) < kGateOff);
    if (__ballot(on)) return false;
  }
  return true;
}

// The wave's columns: lanes past the row's end stand in for lane 0, whose values they compute and store a second time
// (a wave's stores are then the same for every wave, under no condition).
template <typename T, int V>
struct Cols {
  bool act;
  uint32_t lo;        // the lane's byte offset
  int64_t first;      // the wave's first column
  __device__ __forceinline__ Cols(int64_t p) {
    first = (int64_t)blockIdx.x * (64 * V);
    act = first + lane_id() * V < p;
    lo = act ? (uint32_t)(lane_id() * V * (int)sizeof(T)) : 0u;
  }
};

// E: window capacity (e <= E), O: momentum order, V: columns per lane
template <typename T, int V, int E, int O>
__global__ __launch_bounds__(64) void k_chain_fwd(Args<T> a) {
  const int row = blockIdx.y, lane = lane_id();
  const Cols<T, V> col(a.p);
  const uint32_t lo = col.lo;
  const int n = a.n, e = a.e;
  const int64_t p = a.p, rp = (int64_t)row * p;
  const bool off = gates_off(a.gate, (int64_t)a.bh * n);
  const T* sp = a.s + rp * n + col.first;
  T* up = a.update + rp * (n + 1) + col.first;
  T* kp = a.kept ? a.kept + rp * (n + 1) + col.first : nullptr;
  const T* gate = (a.gate ? a.gate : a.decay) + (int64_t)row * n;   // (loaded without a branch)
  const T* decay = a.decay + (int64_t)row * n;

  float m[O > 0 ? O : 1][V], c[V], hist[E > 1 ? E - 1 : 1][V];
  ldv<T, V>(a.last + rp + col.first, lo, c);
#pragma unroll
  for (int o = 0; o < O; ++o) ldv<T, V>(a.lm0 + ((int64_t)o * a.bh + row) * p + col.first, lo, m[o]);
  if constexpr (E > 1) {
#pragma unroll
    for (int j = 0; j < E - 1; ++j) {
#pragma unroll
      for (int i = 0; i < V; ++i) hist[j][i] = 0.f;
      if (j < e - 1 && a.buf) ldv<T, V>(a.buf + ((int64_t)row * (e - 1) + (e - 2 - j)) * p + col.first, lo, hist[j]);
    }
    // the buffer's slots that stay in the window (fewer tokens than slots)
    for (int i = n; i < e - 1; ++i) {
      float b[V] = {};
      if (a.buf) ldv<T, V>(a.buf + ((int64_t)row * (e - 1) + i) * p + col.first, lo, b);
      stv<T, V>(a.buf1 + ((int64_t)row * (e - 1) + (i - n)) * p + col.first, lo, b);
    }
  }
  float zero[V] = {};
  stv<T, V>(up, lo, off ? zero : c);
  if (kp) stv<T, V>(kp, lo, off ? zero : c);

  // step u of a group of kU: the surprises of the step kU later take its registers as it is done, the scalars of
  // the next group are in flight (lane u: step u's)
  float x[kU][V], sc[2 + O], scn[2 + O];
  auto load_scalars = [&](int t0) {
    const int tl = min(t0 + (lane & (kU - 1)), n - 1);
    scn[0] = to_f32(decay[tl]);
    scn[1] = to_f32(gate[tl]);
#pragma unroll
    for (int o = 0; o < O; ++o) scn[2 + o] = to_f32(a.am[((int64_t)o * a.bh + row) * n + tl]);
  };
  load_scalars(0);
#pragma unroll
  for (int u = 0; u < kU; ++u) ldv<T, V>(sp + (int64_t)min(u, n - 1) * p, lo, x[u]);
  auto group = [&](auto whole, int t0) {
#pragma unroll
    for (int k = 0; k < 2 + O; ++k) sc[k] = scn[k];
    load_scalars(t0 + kU);
    if (a.kdecay && blockIdx.x == 0 && lane < kU && t0 + lane < n) a.kdecay[(int64_t)row * n + t0 + lane] = from_f32<T>(sc[0]);
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int t = t0 + u;
      if (decltype(whole)::value || t < n) {
        const float keep = 1.f - lane_of(sc[0], u), g = lane_of(sc[1], u);
        float y[V], w[V];
#pragma unroll
        for (int i = 0; i < V; ++i) y[i] = x[u][i];
        ldv<T, V>(sp + (int64_t)min(t + kU, n - 1) * p, lo, x[u]);
#pragma unroll
        for (int o = 0; o < O; ++o) {
          const float am = lane_of(sc[2 + o], u);
#pragma unroll
          for (int i = 0; i < V; ++i) y[i] = m[o][i] = am * m[o][i] + y[i];
          if (a.moms) stv<T, V>(a.moms + (((int64_t)o * a.bh + row) * n + t) * p + col.first, lo, y);
        }
        if (a.gate) {
#pragma unroll
          for (int i = 0; i < V; ++i) y[i] *= g;
        }
#pragma unroll
        for (int i = 0; i < V; ++i) w[i] = E > 1 ? 0.f : y[i];
        if constexpr (E > 1) {
          if (t + e - 1 >= n) stv<T, V>(a.buf1 + ((int64_t)row * (e - 1) + (t + e - 1 - n)) * p + col.first, lo, y);
#pragma unroll
          for (int j = E - 2; j >= 0; --j)   // oldest first, as atlas_window_sum adds
            if (j < e - 1) {
#pragma unroll
              for (int i = 0; i < V; ++i) w[i] += hist[j][i];
            }
#pragma unroll
          for (int i = 0; i < V; ++i) w[i] += y[i];
#pragma unroll
          for (int j = E - 2; j > 0; --j)
#pragma unroll
            for (int i = 0; i < V; ++i) hist[j][i] = hist[j - 1][i];
#pragma unroll
          for (int i = 0; i < V; ++i) hist[0][i] = y[i];
        }
#pragma unroll
        for (int i = 0; i < V; ++i) c[i] = keep * c[i] + w[i];
        stv<T, V>(up + (int64_t)(t + 1) * p, lo, off ? zero : c);
        if (kp) stv<T, V>(kp + (int64_t)(t + 1) * p, lo, off ? zero : c);
      }
    }
  };
  int t0 = 0;
  for (; t0 + kU <= n; t0 += kU) group(std::true_type{}, t0);
  if (t0 < n) group(std::false_type{}, t0);
#pragma unroll
  for (int o = 0; o < O; ++o) stv<T, V>(a.lm1 + ((int64_t)o * a.bh + row) * p + col.first, lo, m[o]);
}

// The reverse walk: lc the adjoint of c, lm[o] of m_o; hist[j] = du_{t+1+j}.
template <typename T, int V, int E, int O>
__global__ __launch_bounds__(64) void k_chain_bwd(Args<T> a) {
  constexpr int K = 2 + O, B = O > 0 ? O : 1;
  const int row = blockIdx.y, lane = lane_id();
  const Cols<T, V> col(a.p);
  const uint32_t lo = col.lo;
  const int n = a.n, e = a.e;
  const int64_t p = a.p, rp = (int64_t)row * p;
  const bool off = gates_off(a.gate, (int64_t)a.bh * n);
  const bool live = !off && a.dup;            // dupdate reaches the columns
  const T* cp = a.upd + rp * (n + 1) + col.first;   // row t: c_{t-1}
  const T* dp = a.dup ? a.dup + rp * (n + 1) + col.first : cp;   // (absent: readable rows, not used)
  const T* gate = (a.gate ? a.gate : a.decay) + (int64_t)row * n;
  const T* decay = a.decay + (int64_t)row * n;
  const T *bp[B], *b0[B];                     // momenta of order o and the one before the first step (order 0: the
                                              // surprises, which only the gate's gradient needs: readable rows where
                                              // they are absent, and before the first step)
  if constexpr (O > 0) {
#pragma unroll
    for (int o = 0; o < O; ++o) {
      bp[o] = a.msrc + ((int64_t)o * a.bh + row) * n * p + col.first;
      b0[o] = a.lm0 + ((int64_t)o * a.bh + row) * p + col.first;
    }
  } else {
    bp[0] = b0[0] = a.s ? a.s + rp * n + col.first : cp;
  }
  T* ds = a.ds + rp * n + col.first;
  float* part = a.part + ((int64_t)row * gridDim.x + blockIdx.x) * K * n;

  float lc[V] = {}, lm[B][V] = {}, hist[E > 1 ? E - 1 : 1][V] = {};
  float base[B][V];                           // m_o at the step (order 0: the surprise)
#pragma unroll
  for (int o = 0; o < B; ++o) ldv<T, V>(bp[o] + (int64_t)(n - 1) * p, lo, base[o]);

  // groups [t1 - kU, t1) walked from their end, step u at t = t1 - 1 - u; the operands of the step kU further take a
  // step's registers as it is done. No load whose value outlives a branch is in the walk: at the join the wave would
  // wait for every access in flight, its own stores included.
  float dn[kU][V], cn[kU][V], bn[B][kU][V], sn[K], sc[K];
  auto load = [&](int u, int t) {             // t may lie before the first step (read from it, not used)
    const int64_t r = (int64_t)max(t, 0) * p;
    ldv<T, V>(dp + r + p, lo, dn[u]);
    ldv<T, V>(cp + r, lo, cn[u]);
#pragma unroll
    for (int o = 0; o < B; ++o) ldv<T, V>(t > 0 ? bp[o] + r - p : b0[o], lo, bn[o][u]);   // the step before
  };
  auto load_scalars = [&](int t1) {
    const int tl = max(t1 - 1 - (lane & (kU - 1)), 0);
    sn[0] = to_f32(decay[tl]);
    sn[1] = to_f32(gate[tl]);
#pragma unroll
    for (int o = 0; o < O; ++o) sn[2 + o] = to_f32(a.am[((int64_t)o * a.bh + row) * n + tl]);
  };
  load_scalars(n);
#pragma unroll
  for (int u = 0; u < kU; ++u) load(u, n - 1 - u);
  float keep_next = 0.f, am_next[B] = {};
  auto group = [&](auto whole, int t1) {
    float acc[K][kU] = {};
#pragma unroll
    for (int k = 0; k < K; ++k) sc[k] = sn[k];
    load_scalars(t1 - kU);
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int t = t1 - 1 - u;
      if (decltype(whole)::value || t >= 0) {
        const float keep = 1.f - lane_of(sc[0], u), g = lane_of(sc[1], u);
        float dx[V], prev[B][V];
#pragma unroll
        for (int i = 0; i < V; ++i) {
          lc[i] = (live ? dn[u][i] : 0.f) + keep_next * lc[i];
          dx[i] = lc[i];
          acc[0][u] -= lc[i] * cn[u][i];
#pragma unroll
          for (int o = 0; o < B; ++o) prev[o][i] = bn[o][u][i];
        }
        load(u, t - kU);
        if constexpr (E > 1) {
#pragma unroll
          for (int j = 0; j < E - 1; ++j)
            if (j < e - 1) {
#pragma unroll
              for (int i = 0; i < V; ++i) dx[i] += hist[j][i];
            }
#pragma unroll
          for (int j = E - 2; j > 0; --j)
#pragma unroll
            for (int i = 0; i < V; ++i) hist[j][i] = hist[j - 1][i];
#pragma unroll
          for (int i = 0; i < V; ++i) hist[0][i] = lc[i];
          if (a.dbuf1 && t + e - 1 >= n) {
            float b[V];
            ldv<T, V>(a.dbuf1 + ((int64_t)row * (e - 1) + (t + e - 1 - n)) * p + col.first, lo, b);
#pragma unroll
            for (int i = 0; i < V; ++i) dx[i] += b[i];
          }
        }
        if (a.gate) {
#pragma unroll
          for (int i = 0; i < V; ++i) {
            acc[1][u] += dx[i] * base[B - 1][i];
            dx[i] *= g;
          }
        }
#pragma unroll
        for (int o = O - 1; o >= 0; --o) {
          if (a.dlm1 && t == n - 1) {
            float b[V];
            ldv<T, V>(a.dlm1 + ((int64_t)o * a.bh + row) * p + col.first, lo, b);
#pragma unroll
            for (int i = 0; i < V; ++i) dx[i] += b[i];
          }
#pragma unroll
          for (int i = 0; i < V; ++i) {
            lm[o][i] = dx[i] + am_next[o] * lm[o][i];
            dx[i] = lm[o][i];
            acc[2 + o][u] += lm[o][i] * prev[o][i];
          }
          am_next[o] = lane_of(sc[2 + o], u);
        }
#pragma unroll
        for (int o = 0; o < B; ++o)
#pragma unroll
          for (int i = 0; i < V; ++i) base[o][i] = prev[o][i];
        keep_next = keep;
        stv<T, V>(ds + (int64_t)t * p, lo, dx);
      }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (k == 1 && !a.gate) continue;
      float v[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) v[u] = col.act ? acc[k][u] : 0.f;
      const float s = sums8(v);
      const int t = t1 - 1 - sums8_value(lane);
      if ((lane & 28) == 0 && t >= 0) part[(int64_t)k * n + t] = s;
    }
  };
  int t1 = n;
  for (; t1 >= kU; t1 -= kU) group(std::true_type{}, t1);
  if (t1 > 0) group(std::false_type{}, t1);
  float d0[V] = {};
  if (live) ldv<T, V>(dp, lo, d0);
#pragma unroll
  for (int i = 0; i < V; ++i) d0[i] += keep_next * lc[i];
  stv<T, V>(a.dlast + rp + col.first, lo, d0);
#pragma unroll
  for (int o = 0; o < O; ++o) {
#pragma unroll
    for (int i = 0; i < V; ++i) lm[o][i] *= am_next[o];
    stv<T, V>(a.dlm0 + ((int64_t)o * a.bh + row) * p + col.first, lo, lm[o]);
  }
  if constexpr (E > 1) {
    if (a.dbuf) {   // slot i: du_0 .. du_min(n - 1, i) (hist[t] = du_t now, zero past n) and its copy in the next buffer
      float run[V] = {};
#pragma unroll
      for (int j = 0; j < E - 1; ++j) {
        if (j < e - 1) {
          float b[V] = {}, o[V];
          if (a.dbuf1 && j >= n) ldv<T, V>(a.dbuf1 + ((int64_t)row * (e - 1) + (j - n)) * p + col.first, lo, b);
#pragma unroll
          for (int i = 0; i < V; ++i) {
            run[i] += hist[j][i];
            o[i] = run[i] + b[i];
          }
          stv<T, V>(a.dbuf + ((int64_t)row * (e - 1) + j) * p + col.first, lo, o);
        }
      }
    }
  }
}

// ddecay [bh, n], dgate [bh, n], dam [O, bh, n] from the waves' partials [bh, nblk, K, n].
template <typename T>
__global__ __launch_bounds__(256) void k_chain_sum(int bh, int n, int nblk, int O, const float* part, T* ddecay, T* dgate,
                                                   T* dam) {
  const int K = 2 + O;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, per = (int64_t)K * n;
  if (i >= per * bh) return;
  const int64_t row = i / per, kt = i - row * per;
  const int k = (int)(kt / n), t = (int)(kt - (int64_t)k * n);
  T* out = k == 0 ? ddecay + row * n : k == 1 ? (dgate ? dgate + row * n : nullptr)
                                              : dam + ((int64_t)(k - 2) * bh + row) * n;
  if (!out) return;
  const float* q = part + row * nblk * per + kt;
  float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
  int b = 0;
  for (; b + 3 < nblk; b += 4) {
    s0 += q[(int64_t)b * per];
    s1 += q[(int64_t)(b + 1) * per];
    s2 += q[(int64_t)(b + 2) * per];
    s3 += q[(int64_t)(b + 3) * per];
  }
  for (; b < nblk; ++b) s0 += q[(int64_t)b * per];
  out[t] = from_f32<T>((s0 + s1) + (s2 + s3));
}

template <typename T, int V, int E, int O>
hipError_t launch(const Args<T>& a, bool bwd, hipStream_t s) {
  const dim3 grid((unsigned)((a.p + 64 * V - 1) / (64 * V)), (unsigned)a.bh);
  if (bwd) hipLaunchKernelGGL((k_chain_bwd<T, V, E, O>), grid, dim3(64), 0, s, a);
  else hipLaunchKernelGGL((k_chain_fwd<T, V, E, O>), grid, dim3(64), 0, s, a);
  return hipGetLastError();
}
template <typename T, int V, int E>
hipError_t by_order(const Args<T>& a, int order, bool bwd, hipStream_t s) {
  return order == 0 ? launch<T, V, E, 0>(a, bwd, s) : order == 1 ? launch<T, V, E, 1>(a, bwd, s)
                                                                 : launch<T, V, E, 2>(a, bwd, s);
}
template <typename T, int V>
hipError_t by_window(const Args<T>& a, int order, bool bwd, hipStream_t s) {
  if (a.e == 1) return by_order<T, V, 1>(a, order, bwd, s);
  if (a.e <= 4) return by_order<T, V, 4>(a, order, bwd, s);
  return by_order<T, V, kMaxWin>(a, order, bwd, s);
}
template <typename T>
hipError_t run(const Args<T>& a, int order, bool bwd, hipStream_t s) {
  // two columns per lane (8-byte fp32 accesses) where the rows stay aligned to it
  return a.p % 2 == 0 ? by_window<T, 2>(a, order, bwd, s) : by_window<T, 1>(a, order, bwd, s);
}
int waves_per_row(int64_t p) { return (int)((p + (p % 2 == 0 ? 127 : 63)) / (p % 2 == 0 ? 128 : 64)); }

bool bad(int64_t bh, int64_t n, int64_t p, int order, int window) {
  return bh < 1 || bh > 65535 || n < 1 || n > (1 << 24) || p < 1 || p > ((int64_t)1 << 31) || order < 0 ||
         order > kMaxOrder || window < 1 || window > kMaxWin;
}
bool off16(const void* q) { return q && (reinterpret_cast<uintptr_t>(q) & 15) != 0; }

}  // namespace chain
}  // namespace atlas

using namespace atlas;
using namespace atlas::chain;

extern "C" {

int64_t atlas_omega_chain_workspace_bytes(int64_t bh, int64_t n, int64_t p, int order) {
  if (bad(bh, n, p, order, 1)) return 0;
  return bh * waves_per_row(p) * (2 + order) * n * (int64_t)sizeof(float);
}

int atlas_omega_chain_fwd_keep(int dtype, int64_t bh, int64_t n, int64_t p, int order, int window, const void* surprise,
                               const void* decay, const void* last_update, const void* momentum, const void* last_momentum,
                               const void* gate, const void* buffer, void* update, void* moments, void* next_momentum,
                               void* next_buffer, void* kept_update, void* kept_decay, void* stream) {
  if (bad(bh, n, p, order, window)) return ATLAS_MEM_ERR_SHAPE;
  if (!surprise || !decay || !last_update || !update || (order > 0 && (!momentum || !last_momentum || !next_momentum)) ||
      (window > 1 && !next_buffer))
    return ATLAS_MEM_ERR_NULL;
  for (const void* q : {surprise, last_update, last_momentum, buffer, (const void*)update, (const void*)moments,
                        (const void*)next_momentum, (const void*)next_buffer, (const void*)kept_update})
    if (off16(q)) return ATLAS_MEM_ERR_ALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto go = [&](auto tag) {
    using T = decltype(tag);
    Args<T> a{};
    a.n = (int)n; a.bh = (int)bh; a.e = window; a.p = p;
    a.s = (const T*)surprise; a.decay = (const T*)decay; a.last = (const T*)last_update; a.am = (const T*)momentum;
    a.lm0 = (const T*)last_momentum; a.gate = (const T*)gate; a.buf = (const T*)buffer;
    a.update = (T*)update; a.moms = (T*)moments; a.lm1 = (T*)next_momentum; a.buf1 = (T*)next_buffer;
    a.kept = (T*)kept_update; a.kdecay = (T*)kept_decay;
    return run<T>(a, order, false, s);
  };
  if (dtype != ATLAS_DT_BF16 && dtype != ATLAS_DT_F32) return ATLAS_MEM_ERR_DTYPE;
  const hipError_t err = dtype == ATLAS_DT_BF16 ? go(bf16{}) : go(float{});
  return err == hipSuccess ? ATLAS_MEM_OK : ATLAS_MEM_ERR_LAUNCH;
}

int atlas_omega_chain_fwd(int dtype, int64_t bh, int64_t n, int64_t p, int order, int window, const void* surprise,
                          const void* decay, const void* last_update, const void* momentum, const void* last_momentum,
                          const void* gate, const void* buffer, void* update, void* moments, void* next_momentum,
                          void* next_buffer, void* stream) {
  return atlas_omega_chain_fwd_keep(dtype, bh, n, p, order, window, surprise, decay, last_update, momentum, last_momentum,
                                    gate, buffer, update, moments, next_momentum, next_buffer, nullptr, nullptr, stream);
}

int atlas_omega_chain_bwd(int dtype, int64_t bh, int64_t n, int64_t p, int order, int window, const void* surprise,
                          const void* decay, const void* momentum, const void* last_momentum, const void* gate,
                          const void* update, const void* moments, const void* dupdate, const void* dnext_momentum,
                          const void* dnext_buffer, void* dsurprise, void* ddecay, void* dlast_update, void* dmomentum,
                          void* dlast_momentum, void* dgate, void* dbuffer, void* workspace, int64_t workspace_bytes,
                          void* stream) {
  if (bad(bh, n, p, order, window)) return ATLAS_MEM_ERR_SHAPE;
  if (!decay || !update || !dsurprise || !ddecay || !dlast_update || !workspace || (dgate && !gate) ||
      (order == 0 && dgate && !surprise) ||
      (order > 0 && (!momentum || !last_momentum || !moments || !dmomentum || !dlast_momentum)))
    return ATLAS_MEM_ERR_NULL;
  for (const void* q : {surprise, update, last_momentum, moments, dupdate, dnext_momentum, dnext_buffer,
                        (const void*)dsurprise, (const void*)dlast_update, (const void*)dlast_momentum,
                        (const void*)dbuffer, (const void*)workspace})
    if (off16(q)) return ATLAS_MEM_ERR_ALIGN;
  if (workspace_bytes < atlas_omega_chain_workspace_bytes(bh, n, p, order)) return ATLAS_MEM_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto go = [&](auto tag) {
    using T = decltype(tag);
    Args<T> a{};
    a.n = (int)n; a.bh = (int)bh; a.e = window; a.p = p;
    a.s = (const T*)surprise; a.decay = (const T*)decay; a.am = (const T*)momentum; a.lm0 = (const T*)last_momentum;
    a.gate = (const T*)gate; a.upd = (const T*)update; a.msrc = (const T*)moments;
    a.dup = (const T*)dupdate; a.dlm1 = (const T*)dnext_momentum; a.dbuf1 = window > 1 ? (const T*)dnext_buffer : nullptr;
    a.ds = (T*)dsurprise; a.dlast = (T*)dlast_update; a.dlm0 = (T*)dlast_momentum;
    a.dbuf = window > 1 ? (T*)dbuffer : nullptr; a.part = (float*)workspace;
    hipError_t err = run<T>(a, order, true, s);
    if (err != hipSuccess) return err;
    const int64_t outs = bh * (2 + order) * n;
    hipLaunchKernelGGL(k_chain_sum<T>, dim3((unsigned)((outs + 255) / 256)), dim3(256), 0, s, (int)bh, (int)n,
                       waves_per_row(p), order, a.part, (T*)ddecay, (T*)dgate, (T*)dmomentum);
    return hipGetLastError();
  };
  if (dtype != ATLAS_DT_BF16 && dtype != ATLAS_DT_F32) return ATLAS_MEM_ERR_DTYPE;
  const hipError_t err = dtype == ATLAS_DT_BF16 ? go(bf16{}) : go(float{});
  return err == hipSuccess ? ATLAS_MEM_OK : ATLAS_MEM_ERR_LAUNCH;
}

}  // extern "C"
