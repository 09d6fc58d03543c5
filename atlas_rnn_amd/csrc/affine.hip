// affine.hip - right-affine scan H_t = H_{t-1} A_t + B_t (atlas_pytorch/affine_scan.py:36-158) on the fp32
// matrix cores (v_mfma_f32_16x16x4_f32), in one pass over the steps or in chunks.
//
// A: [N][T][D][D], B: [N][T][R][D], prev = H_0: [N][R][D] (zero when absent); out = H_1 .. H_T as
// [N][T][R][D]; fp32, D, R <= 64 (zero-padded to 64 x 64 operands inside LDS).
//
// One kernel walks steps: k_aff_scan, a workgroup per 16 rows of one state (32 or 64 where D is 32 or
// 16), H in LDS and registers, the matrices streaming through LDS. A single chunk moves every operand once,
// but its T steps are serial and occupy N ceil(R / 16) workgroups; where that leaves the card idle the steps are
// cut into nc chunks, each of which composes to one affine map X -> X P_c + Q_c (Geo, affine_geo):
//   kCompose : per (n, chunk): P_c = the product of the chunk's matrices (from the identity, D more rows)
//              and Q_c = its scan from zero; chunk 0 starts from prev and writes its states at once
//   kChain   : per n: the chunk-start states X_{c+1} = X_c P_c + Q_c, chunks as steps
//   kApply   : per (n, chunk > 0): the chunk's states from X_c
// A step is a product of 512 cycles in the matrix cores (D = 64) and takes about 790, 0.33 us, where the operands
// come from the infinity cache, and 0.45 to 0.5 from HBM. Before (three passes of 64-step chunks with every
// wave on its own rows and 2 products a step), forward and backward together: 32 x 1024 steps of 64 x 64 1760 -> 1340
// us, 16 x 1024 974 -> 819, 8 x 1024 888 -> 492, 2 x 1024 829 -> 142, 8 x 300 of 32 x 64 547 -> 78, 20 x 400 of 16 x 16
// 697 -> 99. The largest moves 9 x 537 MB, its scans at 3.1 TB/s: 128 workgroups' pull on three streams.
//
// Backward: with the adjoint G_t = dL/dH_t,  G_T = dout_T,  G_t = dout_t + G_{t+1} A_{t+1}^T, so G is the
// same scan run backwards in time over the transposed matrices (REV, written straight into dB = G). Then k_aff_grad_a forms dA_t = H_{t-1}^T G_t for every (n, t) and
// dprev = G_1 A_1^T (one extra workgroup per n).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/atlas_mem.h"
#include "mem_common.h"
#include "walk_common.h"

namespace atlas {

namespace aff {
constexpr int kThreads = 256;   // 4 waves
constexpr int kMax = 64;        // D, R <= 64; every operand is zero-padded to 64 x 64 in LDS
constexpr int P = kMax + 1;     // LDS pitch (fp32)
constexpr int NE = kMax * kMax / kThreads;   // elements of a 64 x 64 operand per thread (16)
typedef MM<float> M;

struct Geo {
  int N, T, R, D, L, nc;
  int rev;   // 0: forward scan over A; 1: adjoint scan over A^T, backwards in time
};

// A product C = X S on the matrix cores. Wave w owns the output rows 16 w .. 16 w + 15, all four
// 16-column tiles: acc[nt][r] = C[16 w + 4 kq + r][16 nt + tl] (tl = lane & 15, kq = lane >> 4). The
// k order is free as long as both operands follow it; lane group kq takes k = 16 kq + j at step j.
// XT / ST: X(m, k) = X[k][m] / S(k, n) = S[n][k] (the operand is stored transposed). With the pitch
// 65 every one of these scalar reads is free of bank conflicts in either orientation (the lanes of a
// read differ by tl + 16 kq + const modulo 64).
template <bool XT, bool ST>
__device__ __forceinline__ void prod(f32x4 (&acc)[4], const float (*X)[P], const float (*S)[P]) {
  const int l = lane_id(), w = wave_id(), tl = l & 15, kq = l >> 4;
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) acc[nt] = zero4();
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int k = 16 * kq + j;
    const float a = XT ? X[k][16 * w + tl] : X[16 * w + tl][k];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      const float b = ST ? S[16 * nt + tl][k] : S[k][16 * nt + tl];
      acc[nt] = M::mma(a, b, acc[nt]);
    }
  }
}

// A rows x cols row-major matrix in memory (null: zeros) through registers into a zero-padded 64 x 64 LDS
// operand. Thread t holds
// the 4-element groups t + 256 u (row (t + 256 u) / 16): coalesced loads (16-byte loads for a full
// 64 x 64 matrix), conflict-free LDS writes.
struct Pre {
  float v[NE];
};
__device__ __forceinline__ void pre_load(Pre& p, const float* src, int rows, int cols) {
  const bool full = src && rows == kMax && cols == kMax;
#pragma unroll
  for (int u = 0; u < NE / 4; ++u) {
    const int v = threadIdx.x + kThreads * u, r = v / (kMax / 4), c = 4 * (v % (kMax / 4));
    if (full) {
      const float4 x = *reinterpret_cast<const float4*>(src + r * kMax + c);
      p.v[4 * u] = x.x; p.v[4 * u + 1] = x.y; p.v[4 * u + 2] = x.z; p.v[4 * u + 3] = x.w;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float x = 0.f;
        if (src && r < rows && c + i < cols) x = src[r * cols + c + i];
        p.v[4 * u + i] = x;
      }
    }
  }
}
__device__ __forceinline__ void pre_store(const Pre& p, float (*s)[P]) {
#pragma unroll
  for (int u = 0; u < NE / 4; ++u) {
    const int v = threadIdx.x + kThreads * u, r = v / (kMax / 4), c = 4 * (v % (kMax / 4));
#pragma unroll
    for (int i = 0; i < 4; ++i) s[r][c + i] = p.v[4 * u + i];
  }
}

// acc -> memory (rows x cols).
__device__ __forceinline__ void acc_store(const f32x4 (&acc)[4], float* out, int rows, int cols) {
  const int l = lane_id(), w = wave_id(), tl = l & 15, kq = l >> 4;
  const bool full = rows == kMax && cols == kMax;
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * w + 4 * kq + r, col = 16 * nt + tl;
      if (full || (row < rows && col < cols)) out[row * cols + col] = acc[nt][r];
    }
}

// ---- the scan kernel ----
constexpr int kDepth = 4;
constexpr int kAny = 0, kTiny = -1;   // D that the kernel is not built for
constexpr int threads(int d) { return d == 48 ? 192 : 256; }   // of a scan workgroup

struct ScanArgs {
  Geo g;
  const float* A;      // step matrices [N][T][D][D]
  const float* C;      // step additions [N][T][R][D]
  const float* prev;   // start of chunk 0 [N][R][D] or null (zero)
  float* out;          // states by array position [N][T][R][D]
  float* Pc;           // [N][nc][D][D]
  float* Qc;           // [N][nc][R][D]
  float* Xc;           // chunk starts [N][nc][R][D]
  int pass;            // kDirect, kCompose, kApply, kChain
  int parts;           // workgroups per unit
  int units;
};
enum { kDirect, kCompose, kApply, kChain };

__device__ __forceinline__ uint32_t bld4(rsrc_t r, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
}
__device__ __forceinline__ void bst4(rsrc_t r, uint32_t off, uint32_t v) {
  __builtin_amdgcn_raw_buffer_store_b32(v, r, (int)off, 0, 0);
}

}  // namespace aff

using aff::Geo;

// One unit = the steps of one chunk of one n; KD waves = 16 rows of its state, each wave 16 columns.
// DC: D, or kAny / kTiny for a D of 4 .. 63 / 1 .. 3 that is not a multiple of 16. The rows of a kAny matrix are not
// aligned to the lanes' groups of four: the group that crosses the end of a row is loaded as the row's last four
// elements and shifted where it is used, so that a group is one 16-byte load as elsewhere. Element by element it
// was four times the loads (16 x 512 steps of 64 x 63, forward and backward: 1140 -> 620 us, three passes of 64-step
// chunks 932); a shift where it is loaded waits for every load (1520).
template <bool REV, int DC>
__global__ __launch_bounds__(aff::threads(DC), 2) void k_aff_scan(aff::ScanArgs a) {
  using namespace aff;
  constexpr int KD = DC > 0 ? DC / 16 : 4;
  constexpr int TH = threads(DC);
  constexpr int RB = TH / (64 * KD);                  // row blocks of a workgroup
  constexpr int NG = 64 * KD * KD;                    // 4-element groups of a matrix
  constexpr int NU = (NG + TH - 1) / TH;              // of them a thread's
  constexpr int DEPTH = DC != kTiny ? kDepth : 2;   // steps whose operands are in flight in registers (4, 6 and 8 take the same time)
  constexpr int SP = REV ? 64 : 68;
  static_assert(DEPTH % 2 == 0, "the LDS buffers alternate");
  __shared__ __align__(16) float S[2][16 * KD][SP];
  __shared__ __align__(16) float X[2][RB][16][64];
  const Geo& g = a.g;
  const int id = blockIdx.x, unit = (id & 7) + 8 * (id / (8 * a.parts)), part = (id >> 3) % a.parts;
  if (unit >= a.units) return;
  const int l = lane_id(), w = __builtin_amdgcn_readfirstlane(wave_id()), tl = l & 15, kq = l >> 4;
  const int rb = w / KD, cw = w % KD;
  const int D = DC > 0 ? DC : g.D, R = g.R;
  const size_t cs = (size_t)R * D, ds = (size_t)D * D;

  // the unit's steps and operands
  int n, c, k0, k1;
  const float *A = a.A, *C = a.C, *start = nullptr;
  float *out = nullptr, *fin = nullptr;
  int grp = part * RB + rb;
  bool ident = false;
  if (a.pass == kDirect) {
    n = unit; c = 0; k0 = 0; k1 = g.T;
    start = a.prev ? a.prev + n * cs : nullptr;
    out = a.out;
  } else if (a.pass == kChain) {   // chunks 1 .. nc - 2 as steps: X_2 .. X_{nc-1}
    n = unit; c = 0; k0 = 1; k1 = g.nc - 1;
    start = a.Xc + ((size_t)n * g.nc + 1) * cs;
    out = a.Xc + cs;               // step k writes X_{k+1}
    A = a.Pc; C = a.Qc;
  } else {
    const int nch = g.nc - 1;      // compose: chunks 0 .. nc - 2; apply: 1 .. nc - 1
    n = unit / nch; c = unit % nch + (a.pass == kApply ? 1 : 0);
    k0 = c * g.L; k1 = min(g.T, k0 + g.L);
    if (a.pass == kApply) {
      start = a.Xc + ((size_t)n * g.nc + c) * cs;
      out = a.out;
    } else if (c == 0) {           // the start is known: states and X_1
      start = a.prev ? a.prev + n * cs : nullptr;
      out = a.out;
      fin = a.Xc + ((size_t)n * g.nc + 1) * cs;
    } else {
      const int gp = (D + 15) / 16;
      if (grp < gp) {
        ident = true;
        fin = a.Pc + ((size_t)n * g.nc + c) * ds;
      } else {
        grp -= gp;
        fin = a.Qc + ((size_t)n * g.nc + c) * cs;
      }
    }
  }
  const int rows = ident ? D : R;
  const int Tn = a.pass == kChain ? g.nc : g.T;   // positions per n in A, C and out
  A += (size_t)n * Tn * ds;
  C += (size_t)n * Tn * cs;
  if (out) out += (size_t)n * Tn * cs;
  const uint32_t cb = (uint32_t)cs * 4u, db = (uint32_t)ds * 4u;
  // the lane's state elements: row xr, columns xc .. xc + 3 (the accumulator's layout: the products are
  // formed transposed); rows and columns past the last are out of range
  const int xr = 16 * grp + tl, xc = 16 * cw + 4 * kq;
  const uint32_t xo = xr < rows && xc < D ? (uint32_t)(xr * D + xc) * 4u : kOob;
  // the lane's elements of the states written: whole rows, a wave's 1 KB in one piece
  const int wi = 64 * cw + l, wr = wi / (4 * KD), wc = 4 * (wi % (4 * KD));
  const uint32_t wo = 16 * grp + wr < rows && wc < D ? (uint32_t)((16 * grp + wr) * D + wc) * 4u : kOob;

  // The positions of steps k .. k + DEPTH - 1 that lie before k1 as one buffer: step k + u is at u st
  // forward, at o - u st backwards in time; the others are out of range (loads give zero).
  struct Blk {
    rsrc_t r;
    uint32_t o;
  };
  auto blk = [&](const float* base, size_t elems, int k, int shift, bool on) {
    const int nv = __builtin_amdgcn_readfirstlane(min(max(k1 - k, 0), DEPTH));
    const int p = REV ? g.T - shift - k - (nv - 1) : k;
    const uint32_t st = (uint32_t)elems * 4u;
    return Blk{make_rsrc(base + (nv > 0 ? (int64_t)p * (int64_t)elems : 0), nv > 0 && on ? (uint32_t)nv * st : 0u),
               REV ? (uint32_t)(nv - 1) * st : 0u};
  };
  // the states written during steps kk ..: those of the steps before them
  auto blk_out = [&](int kk) {
    Blk b = blk(out, cs, max(kk - 1, k0), 1, out != nullptr);
    if (kk == k0) b.o = REV ? b.o + cb : 0u - cb;
    return b;
  };
  auto at = [&](const Blk& b, uint32_t st, int u) { return REV ? b.o - (uint32_t)u * st : b.o + (uint32_t)u * st; };
  const int rem = D & 3;   // kAny: elements of the crossing group
  auto ld4 = [&](rsrc_t r, uint32_t off, int col) {
    if constexpr (DC > 0) {
      return __builtin_bit_cast(f32x4, bld16(r, off));
    } else if constexpr (DC == kAny) {
      return __builtin_bit_cast(f32x4, bld16(r, col < D && col + 4 > D ? off - 4u * (uint32_t)(4 - rem) : off));
    } else {
      f32x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = __builtin_bit_cast(float, bld4(r, col + i < D ? off + 4u * i : kOob));
      return v;
    }
  };
  // what ld4 loaded, in place: where it is used, so that the loads stay in flight
  auto placed = [&](f32x4 v, int col) {
    if constexpr (DC == kAny) {   // (rem is the same in every lane)
      if (col < D && col + 4 > D) {
        const float a = rem == 3 ? v[1] : rem == 2 ? v[2] : v[3], b = rem == 3 ? v[2] : v[3];
        v = f32x4{a, rem > 1 ? b : 0.f, rem == 3 ? v[3] : 0.f, 0.f};
      }
    }
    return v;
  };
  auto st4 = [&](f32x4 v, rsrc_t r, uint32_t off, int col) {
    if constexpr (DC > 0) {
      bst16(r, off, __builtin_bit_cast(u32x4v, v));
    } else if constexpr (DC == kAny) {
      const bool cross = col < D && col + 4 > D;
      bst16(r, cross ? kOob : off, __builtin_bit_cast(u32x4v, v));
#pragma unroll
      for (int i = 0; i < 3; ++i) bst4(r, cross && i < rem ? off + 4u * i : kOob, __builtin_bit_cast(uint32_t, (float)v[i]));
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) bst4(r, col + i < D ? off + 4u * i : kOob, __builtin_bit_cast(uint32_t, (float)v[i]));
    }
  };
  f32x4 ps[DEPTH][NU], cv[DEPTH];
  auto load_a = [&](int u, int v, const Blk& b) {
    const int i = threadIdx.x + TH * v, r = i / (4 * KD), q = i % (4 * KD);
    ps[u][v] = ld4(b.r, (NG % TH == 0 || i < NG) && r < D && 4 * q < D ? at(b, db, u) + (uint32_t)(r * D + 4 * q) * 4u : kOob, 4 * q);
  };
  auto load_c = [&](int u, const Blk& b) { cv[u] = ld4(b.r, xo + at(b, cb, u), xc); };
  auto stage = [&](int u, int v, int b) {   // slot u's matrix into LDS buffer b
    const int i = threadIdx.x + TH * v, r = i / (4 * KD), q = i % (4 * KD);
    if (NG % TH == 0 || i < NG) *reinterpret_cast<f32x4*>(&S[b][r][4 * (REV ? q ^ (r & 15) : q)]) = placed(ps[u][v], 4 * q);
  };
  // A step's matrix as operands: s[4 i + e] = S(16 ((cw + i) % KD) + 4 kq + e, 16 cw + tl). The wave's own
  // 16 columns of the state come first: their products need no exchange.
  float s[2][4 * KD];
  int ki[KD];
#pragma unroll
  for (int i = 0; i < KD; ++i) ki[i] = cw + i < KD ? cw + i : cw + i - KD;
  auto read_s = [&](int t, int i, int b) {
    if constexpr (REV) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(&S[b][16 * cw + tl][4 * ((4 * ki[i] + kq) ^ tl)]);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[t][4 * i + e] = v[e];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) s[t][4 * i + e] = S[b][16 * ki[i] + 4 * kq + e][16 * cw + tl];
    }
  };
  f32x4 xv[KD];
  auto read_x = [&](int b) {
#pragma unroll
    for (int i = 1; i < KD; ++i) xv[i] = *reinterpret_cast<const f32x4*>(&X[b][rb][tl][4 * ((4 * ki[i] + kq) ^ tl)]);
  };
  auto write_x = [&](int b, f32x4 v) { *reinterpret_cast<f32x4*>(&X[b][rb][tl][4 * ((4 * cw + kq) ^ tl)]) = v; };

  f32x4 x = placed(ld4(make_rsrc(start, start ? cb : 0u), xo, xc), xc);
  if (ident) {
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = xr < D && xr == xc + i ? 1.f : 0.f;
  }
  write_x(0, x);
  // Step k's matrix is A[k] forward and A[T - k] (transposed) in reverse, where step 0 has none: the
  // state before it is zero, and so is the matrix.
  {
    const float* a0 = A + (REV ? (k0 > 0 ? (size_t)(g.T - k0) * ds : 0) : (size_t)k0 * ds);
    const Blk b0{make_rsrc(a0, REV && k0 == 0 ? 0u : db), 0u}, b1 = blk(A, ds, k0 + 1, 0, true);
#pragma unroll
    for (int v = 0; v < NU; ++v) {
      load_a(0, v, b0);
      stage(0, v, 0);
      load_a(0, v, b1);
      stage(0, v, 1);
    }
    const Blk ba = blk(A, ds, k0 + 2, 0, true), bc = blk(C, cs, k0, 1, !ident);
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) {
      __builtin_amdgcn_sched_barrier(0);   // in the loop's order, which its waits count on
#pragma unroll
      for (int v = 0; v < NU; ++v) load_a(u, v, ba);
      load_c(u, bc);
    }
  }
  lds_barrier();
#pragma unroll
  for (int i = 0; i < KD; ++i) read_s(0, i, 0);
  // Step k: s[u & 1] holds S_k, LDS buffer (u + 1) & 1 S_{k+1}, x and X[u & 1] the state before it. One
  // LDS or memory instruction behind each matrix instruction: in a row they would hold up the next one
  // (889 -> 705 cycles a step of 512 in the matrix cores).
  auto step = [&](int u, const Blk& ba, const Blk& bc, const Blk& bo) {
    f32x4 own[2] = {zero4(), zero4()}, acc[2] = {zero4(), zero4()};
#pragma unroll
    for (int e = 0; e < 4; ++e) own[e & 1] = M::mma(s[u & 1][e], x[e], own[e & 1]);
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    read_x(u & 1);
    const f32x4 y = *reinterpret_cast<const f32x4*>(&X[u & 1][rb][wr][4 * ((wc / 4) ^ wr)]);
    __builtin_amdgcn_sched_barrier(0);
    constexpr int NM = KD > 1 ? 4 * (KD - 1) : 1, NO = KD + 2 * NU;   // (KD = 1: all behind the own products)
    auto other = [&](int o) {
      if (o < KD) {
        read_s((u + 1) & 1, o, (u + 1) & 1);                    // S_{k+1}
      } else if ((o - KD) % 2 == 0) {
        stage(u, (o - KD) / 2, u & 1);                          // S_{k+2}: the buffer's S_k was read a step ago
      } else {
        load_a(u, (o - KD) / 2, ba);
      }
    };
#pragma unroll
    for (int j = 0; j < NM; ++j) {
      if constexpr (KD > 1) acc[j & 1] = M::mma(s[u & 1][4 + j], xv[1 + j / 4][j % 4], acc[j & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int o = j * NO / NM; o < (j + 1) * NO / NM; ++o) other(o);
      __builtin_amdgcn_sched_barrier(0);
    }
    const f32x4 c = placed(cv[u], xc);
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = (acc[0][i] + acc[1][i]) + (own[0][i] + own[1][i]) + c[i];
    write_x((u + 1) & 1, x);
    st4(y, bo.r, wo + at(bo, cb, u), wc);   // the state before step k
    load_c(u, bc);
  };
  int kk = k0;
  for (; kk + DEPTH <= k1; kk += DEPTH) {
    const Blk ba = blk(A, ds, kk + 2 + DEPTH, 0, true), bc = blk(C, cs, kk + DEPTH, 1, !ident),
              bo = blk_out(kk);
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) step(u, ba, bc, bo);
  }
  if (kk < k1) {   // the last, partial block: nothing is left to load
    const Blk none{make_rsrc(A, 0u), 0u}, bo = blk_out(kk);
#pragma unroll
    for (int u = 0; u < DEPTH - 1; ++u)
      if (kk + u < k1) step(u, none, none, bo);
  }
  st4(x, blk(out, cs, k1 - 1, 1, out != nullptr).r, xo, xc);
  st4(x, make_rsrc(fin, fin ? (ident ? db : cb) : 0u), xo, xc);
}

// dA_t = H_{t-1}^T G_t  (D x D, k over R) for every (t, n); workgroup t = T of each n forms
// dprev = G_1 A_1^T (R x D, k over D) when dprev is requested.
__global__ __launch_bounds__(aff::kThreads) void k_aff_grad_a(Geo g, const float* __restrict__ A,
                                                              const float* __restrict__ H,
                                                              const float* __restrict__ prev,
                                                              const float* __restrict__ G, float* __restrict__ dA,
                                                              float* __restrict__ dprev) {
  __shared__ float Xs[aff::kMax][aff::P];
  __shared__ float Ss[aff::kMax][aff::P];
  const int t = blockIdx.x, n = blockIdx.y;
  const size_t cs = (size_t)g.R * g.D;
  aff::Pre ps;
  f32x4 acc[4];
  if (t == g.T) {   // workgroup-uniform
    if (!dprev) return;
    // C[r][d] = sum_e G_1[r][e] A_1[d][e]: X = G_1 as stored, S(e, d) = A_1[d][e] (transposed)
    aff::pre_load(ps, G + (size_t)n * g.T * cs, g.R, g.D);
    aff::pre_store(ps, Xs);
    aff::pre_load(ps, A + (size_t)n * g.T * g.D * g.D, g.D, g.D);
    aff::pre_store(ps, Ss);
    __syncthreads();
    aff::prod<false, true>(acc, Xs, Ss);
    aff::acc_store(acc, dprev + (size_t)n * cs, g.R, g.D);
    return;
  }
  // C[d][e] = sum_r H_{t-1}[r][d] G_t[r][e]: X(d, r) = H[r][d] (transposed), S(r, e) = G[r][e]
  const float* Hp = t > 0 ? H + ((size_t)n * g.T + t - 1) * cs : (prev ? prev + (size_t)n * cs : nullptr);
  aff::pre_load(ps, Hp, g.R, g.D);
  aff::pre_store(ps, Xs);
  aff::pre_load(ps, G + ((size_t)n * g.T + t) * cs, g.R, g.D);
  aff::pre_store(ps, Ss);
  __syncthreads();
  aff::prod<true, false>(acc, Xs, Ss);
  aff::acc_store(acc, dA + ((size_t)n * g.T + t) * g.D * g.D, g.D, g.D);
}

}  // namespace atlas

using namespace atlas;

namespace {

int affine_check(int n, int t, int r, int d) {
  if (n < 1 || t < 1 || r < 1 || d < 1 || r > aff::kMax || d > aff::kMax) return ATLAS_MEM_ERR_SHAPE;
  return ATLAS_MEM_OK;
}

// Chunks: the count with the shortest schedule, in steps. A workgroup more than the 256 CUs costs 0.75 of its
// steps (two share a CU, a step's matrix instructions take 512 of its 790 cycles), a pass more about 12
// steps. Not where a single chunk already fills half the card: the additional passes over A and C would cost more
// than the idle half (32 x 1024 of 64 x 64: 1 chunk 523 + 833 us forward and backward, 3 chunks 554 + 853; 24 x 600:
// 1 chunk 275 + 411, 4 chunks 205 + 330). Whole blocks of kDepth steps per chunk: a partial block at the end of each
// waits for its loads one by one (8 x 1024: 8 chunks of 128 steps 190 us, 10 of 103 218).
Geo affine_geo(int n, int t, int r, int d, int rev) {
  Geo g{};
  g.N = n; g.T = t; g.R = r; g.D = d;
  g.rev = rev;
  constexpr double kCUs = 256., kPass = 12.;
  const int rb = d == 16 ? 4 : d == 32 ? 2 : 1;   // 16-row blocks of a workgroup
  const int gr = (r + 15) / 16, gp = (d + 15) / 16;
  const double wd = (double)n * ((gr + rb - 1) / rb), wc = (double)n * ((gr + gp + rb - 1) / rb);
  auto steps = [&](double wgs, int len) { return len * (wgs <= kCUs ? 1. : std::max(1., 0.75 * wgs / kCUs)); };
  double best = steps(wd, t);
  g.L = t;
  for (int want = 2; want <= 256 && wd < kCUs / 2; ++want) {
    const int len = ((t + want - 1) / want + aff::kDepth - 1) / aff::kDepth * aff::kDepth, nc = (t + len - 1) / len;
    if (nc < 2) break;
    const double cost = steps(wc * (nc - 1), len) + steps(wd * (nc - 1), len) + (nc - 2) + 2. * kPass;
    if (cost < best) {
      best = cost;
      g.L = len;
    }
  }
  g.nc = (t + g.L - 1) / g.L;
  return g;
}

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// workspace: P_c [N][nc][D][D], Q_c and X_c [N][nc][R][D]
size_t affine_ws_bytes(const Geo& g) {
  const size_t nc = (size_t)g.N * g.nc;
  return align256(nc * g.D * g.D * 4) + 2 * align256(nc * g.R * g.D * 4);
}

template <bool REV, int DC>
void launch_scan_d(aff::ScanArgs& a, int blocks, hipStream_t s) {
  const int rb = DC > 0 ? aff::threads(DC) / (4 * DC) : 1;   // 16-row blocks of a workgroup
  a.parts = (blocks + rb - 1) / rb;
  hipLaunchKernelGGL((k_aff_scan<REV, DC>), dim3((unsigned)((a.units + 7) / 8 * 8 * a.parts)), dim3(aff::threads(DC)),
                     0, s, a);
}
template <bool REV>
void launch_scan(aff::ScanArgs& a, int blocks, hipStream_t s) {
  switch (a.g.D) {
    case 64: return launch_scan_d<REV, 64>(a, blocks, s);
    case 48: return launch_scan_d<REV, 48>(a, blocks, s);
    case 32: return launch_scan_d<REV, 32>(a, blocks, s);
    case 16: return launch_scan_d<REV, 16>(a, blocks, s);
    default:
      if (a.g.D < 4) return launch_scan_d<REV, aff::kTiny>(a, blocks, s);
      return launch_scan_d<REV, aff::kAny>(a, blocks, s);
  }
}

int affine_scan(const Geo& g, const float* A, const float* C, const float* prev, float* out, void* ws,
                hipStream_t s) {
  unsigned char* w = static_cast<unsigned char*>(ws);
  const size_t nc = (size_t)g.N * g.nc;
  aff::ScanArgs a{};
  a.g = g;
  a.A = A; a.C = C; a.prev = prev; a.out = out;
  a.Pc = reinterpret_cast<float*>(w);
  a.Qc = reinterpret_cast<float*>(w + align256(nc * g.D * g.D * 4));
  a.Xc = reinterpret_cast<float*>(w + align256(nc * g.D * g.D * 4) + align256(nc * g.R * g.D * 4));
  const int gr = (g.R + 15) / 16, gp = (g.D + 15) / 16;
  auto pass = [&](int kind, int units, int groups, bool rev) {
    a.pass = kind;
    a.units = units;
    if (rev) launch_scan<true>(a, groups, s);
    else launch_scan<false>(a, groups, s);
  };
  if (g.nc == 1) {
    pass(aff::kDirect, g.N, gr, g.rev);
  } else {
    pass(aff::kCompose, g.N * (g.nc - 1), gr + gp, g.rev);
    if (g.nc > 2) pass(aff::kChain, g.N, gr, false);
    pass(aff::kApply, g.N * (g.nc - 1), gr, g.rev);
  }
  return hipGetLastError() == hipSuccess ? ATLAS_MEM_OK : ATLAS_MEM_ERR_LAUNCH;
}

bool aff_misaligned(const void* p) { return p && (reinterpret_cast<uintptr_t>(p) & 3) != 0; }

}  // namespace

extern "C" {

size_t atlas_affine_scan_workspace_bytes(int n, int t, int r, int d) {
  if (affine_check(n, t, r, d) != ATLAS_MEM_OK) return 0;
  return affine_ws_bytes(affine_geo(n, t, r, d, 0));
}

int atlas_affine_scan_fwd(int n, int t, int r, int d, const float* A, const float* B, const float* prev, float* out,
                          void* workspace, size_t workspace_bytes, void* stream) {
  const int st = affine_check(n, t, r, d);
  if (st != ATLAS_MEM_OK) return st;
  if (!A || !B || !out || !workspace) return ATLAS_MEM_ERR_NULL;
  if (aff_misaligned(A) || aff_misaligned(B) || aff_misaligned(prev) || aff_misaligned(out) ||
      aff_misaligned(workspace))
    return ATLAS_MEM_ERR_ALIGN;
  const Geo g = affine_geo(n, t, r, d, 0);
  if (workspace_bytes < affine_ws_bytes(g)) return ATLAS_MEM_ERR_WORKSPACE;
  return affine_scan(g, A, B, prev, out, workspace, static_cast<hipStream_t>(stream));
}

int atlas_affine_scan_bwd(int n, int t, int r, int d, const float* A, const float* H, const float* prev,
                          const float* dout, float* dA, float* dB, float* dprev, void* workspace,
                          size_t workspace_bytes, void* stream) {
  const int st = affine_check(n, t, r, d);
  if (st != ATLAS_MEM_OK) return st;
  if (!A || !H || !dout || !dA || !dB || !workspace) return ATLAS_MEM_ERR_NULL;
  if (aff_misaligned(A) || aff_misaligned(H) || aff_misaligned(prev) || aff_misaligned(dout) || aff_misaligned(dA) ||
      aff_misaligned(dB) || aff_misaligned(dprev) || aff_misaligned(workspace))
    return ATLAS_MEM_ERR_ALIGN;
  const Geo g = affine_geo(n, t, r, d, 1);
  if (workspace_bytes < affine_ws_bytes(g)) return ATLAS_MEM_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // G (the adjoint of every H_t) is the reverse scan of dout over A^T; dB = G
  const int rc = affine_scan(g, A, dout, nullptr, dB, workspace, s);
  if (rc != ATLAS_MEM_OK) return rc;
  hipLaunchKernelGGL(k_aff_grad_a, dim3(t + 1, n), dim3(aff::kThreads), 0, s, g, A, H, prev, dB, dA, dprev);
  return hipGetLastError() == hipSuccess ? ATLAS_MEM_OK : ATLAS_MEM_ERR_LAUNCH;
}

}  // extern "C"
