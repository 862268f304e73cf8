// The path layout: a wave64 as four rows of 16 lanes, one root-to-leaf dof path of the tree per row (left leg, right leg,
// left arm, right arm), lane p of a row holding the path's dof p: the root's 6 dofs first (in every row), then the
// leg's 6 hinges (lanes 12..15 of the leg rows hold none) or the waist's 3 (in both arm rows) and the arm's 7. Two dofs
// couple in a matrix with the tree's sparsity only when they share a path, so such a matrix is four 16 x 16 blocks, a
// column per lane in registers, and every broadcast along a path stays inside a row of lanes: it is the row_newbcast
// modifier of the multiply-add that consumes it (v_fmac_f32_dpp), one instruction for all four paths at once, where a
// dof-per-lane layout takes a v_readlane and a multiply-add per pair of dofs.
//
// What bounds the dof-per-lane form is instruction issue (4 clocks a wave64 instruction, 35 of 64 lanes used) and the
// solves' serial chain. Factorizations, solves and Hessian rows in this layout took the forward from 828 to 718 us at
// 4096 worlds, forward + VJP from 3542 to 3074 us at 16384, one world's step from 277 to 226 us.
//
// Every result is bitwise that of the dof-per-lane elimination and solves (each entry's updates are the same products
// in the same order; where the limbs meet, at the waist and the root, the rows of lanes take their turns): the
// factor's and the solver's rounding, and with it Newton's iteration counts, do not depend on the layout. Compared: the
// solves with a replay one dof at a time; states, info and tapes (both factors of every substep) of 24 batches of 1 to
// 4096 worlds with the dof-per-lane build's.
#pragma once
#include "g1_device.h"

namespace g1k {

constexpr int PP = 16;  // lanes, and dofs at most, of a path

// row g's lane p: its dof, or -1
constexpr int path_dof(int g, int p) {
  return p < 6 ? p : g == 0 ? (p < 12 ? p : -1) : g == 1 ? (p < 12 ? p + 6 : -1) : (g == 2 || p < 9) ? p + 12 : p + 19;
}
// the one lane of a dof from which its value is taken: the root's in row 0, the waist's in row 2
constexpr bool path_owner(int g, int p) {
  return path_dof(g, p) >= 0 && (p >= 6 || g == 0) && (g != 3 || p >= 9);
}
constexpr int owner_lane_of(int i) { return i + (i < 12 ? 0 : i < 18 ? 10 : i < 28 ? 20 : 29); }
constexpr bool check_path_layout() {  // every dof owned once; a dof's ancestors are the lanes up to its own, in order
  int owned[NV] = {};
  for (int g = 0; g < 4; g++)
    for (int p = 0; p < PP; p++) {
      const int d = path_dof(g, p);
      if (d < 0) continue;
      if (d >= NV) return false;
      if (path_owner(g, p)) owned[d]++;
      uint64_t anc = 0;
      for (int q = 0; q <= p; q++) anc |= (uint64_t)1 << path_dof(g, q);
      if (TREE.dofanc[d] != anc) return false;
    }
  for (int d = 0; d < NV; d++) {
    const int l = owner_lane_of(d);
    if (owned[d] != 1 || !path_owner(l >> 4, l & 15) || path_dof(l >> 4, l & 15) != d) return false;
  }
  return true;
}
static_assert(check_path_layout(), "the four dof paths: legs 6..11 / 12..17, waist 18..20 with arms 21..27 / 28..34");

// lane masks (bit l: lane l) as 32-bit halves, rows 0-1 and rows 2-3
struct LaneMask { unsigned lo, hi; };
template <class F>
constexpr LaneMask lane_mask(F f) {
  LaneMask m{0u, 0u};
  for (int l = 0; l < 64; l++)
    if (f(l >> 4, l & 15)) (l < 32 ? m.lo : m.hi) |= 1u << (l & 31);
  return m;
}
constexpr LaneMask PATH_VALID = lane_mask([](int g, int p) { return path_dof(g, p) >= 0; });
constexpr LaneMask PATH_ROOT = lane_mask([](int, int p) { return p < 6; });
constexpr LaneMask PATH_ARMS = lane_mask([](int g, int) { return g >= 2; });
constexpr LaneMask PATH_SHARED2 = lane_mask([](int g, int p) { return g == 2 && p < 9; });  // row 2's root and waist
constexpr LaneMask PATH_WAIST3 = lane_mask([](int g, int p) { return g == 3 && p >= 6 && p < 9; });
template <int K>
struct PathLt { static constexpr LaneMask m = lane_mask([](int, int p) { return p < K; }); };
template <int K>
struct PathGt { static constexpr LaneMask m = lane_mask([](int, int p) { return p > K; }); };
template <int K>
struct PathEq { static constexpr LaneMask m = lane_mask([](int, int p) { return p == K; }); };

// the mask as a scalar register pair, built from opaque halves (scalar moves; no vector compare per use)
__device__ __forceinline__ unsigned long long mask_bits(unsigned lo, unsigned hi) {
  asm("" : "+s"(lo));
  asm("" : "+s"(hi));
  return (unsigned long long)hi << 32 | lo;
}
template <const LaneMask& M>
__device__ __forceinline__ float lane_sel(float on, float off) {  // on in the mask's lanes, off in the others
  float r;
  asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(r) : "v"(off), "v"(on), "s"(mask_bits(M.lo, M.hi)));
  return r;
}
template <const LaneMask& M>
__device__ __forceinline__ float lane_sel0(float on) {  // on in the mask's lanes, 0 in the others
  float r;
  asm("v_cndmask_b32_e64 %0, 0, %1, %2" : "=v"(r) : "v"(on), "s"(mask_bits(M.lo, M.hi)));
  return r;
}

// A VALU write followed by a DPP read of the same register needs two wait states, which the compiler does not count
// across inline assembly: every block below that reads by DPP what may have been written just before it opens with
// s_nop 1, and blocks whose results may be read at once by DPP, v_readlane or a lane swap close with one.
#define G1_BC(k) " row_newbcast:" #k " row_mask:0xf bank_mask:0xf\n\t"
#define G1_FMAC_BC(acc, src, mul, k) "v_fmac_f32_dpp " acc ", " src ", " mul G1_BC(k)
#define G1_NOP "s_nop 1\n\t"

// x's even rows and odd rows copied over their pairs: (x0, x0, x2, x2) and (x1, x1, x3, x3)
__device__ __forceinline__ void row_pairs(float x, float* even, float* odd) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  *even = __uint_as_float(r[0]);
  *odd = __uint_as_float(r[1]);
}
// x's rows 0-1 and rows 2-3 copied over the wave: (x0, x1, x0, x1) and (x2, x3, x2, x3)
__device__ __forceinline__ void row_halves(float x, float* low, float* high) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  *low = __uint_as_float(r[0]);
  *high = __uint_as_float(r[1]);
}

// this lane's dof, or NV on the lanes without one
__device__ __forceinline__ int path_lane_dof(int lane) {
  const int p = lane & 15, g = lane >> 4;
  const int off = p < 6 ? 0 : g < 2 ? 6 * g : (g == 3 && p >= 9) ? 19 : 12;
  return g < 2 && p >= 12 ? NV : p + off;
}
__device__ __forceinline__ int owner_lane(int i) { return owner_lane_of(i); }
// a row of dof entries (a matrix row, indexed by dof) seen from a path: entry m's dof is m plus the row's offset, as
// base addresses of the entries 0..5, 6..8, 9..11 and 12..15 (the leg rows have none: zero, at least 16 entries of 0)
struct PathRow { const float *b0, *b6, *b9, *b12; };
__device__ __forceinline__ PathRow path_row(const float* row, const float* zero, int lane) {
  const int g = lane >> 4, o6 = g < 2 ? 6 * g : 12, o9 = g < 3 ? 6 * g : 19;
  return PathRow{row, row + o6, row + o9, g < 2 ? zero : row + o9};
}
template <int M>
__device__ __forceinline__ float path_entry(const PathRow& r) {
  return (M < 6 ? r.b0 : M < 9 ? r.b6 : M < 12 ? r.b9 : r.b12)[M];
}

// c[m] = base[m] + S . F_m for the row's lanes m: S this lane's motion subspace (w, v), F_m = (n, f) lane m's force
// vector; the symmetric products S_p . F_m of a path, one column per lane, 7 instructions an entry
__device__ __forceinline__ void path_products(float (&c)[PP], const float (&base)[PP], const float* w, const float* v,
                                              const float* n, const float* f) {
  // 0 n0, 1 n1, 2 n2, 3 f0, 4 f1, 5 f2; the order of the terms as the compiler contracts the scalar sum
#define G1_C6(acc, k)                                                                                              \
  "v_mul_f32_dpp " acc ", %5, %11" G1_BC(k) G1_FMAC_BC(acc, "%4", "%10", k) G1_FMAC_BC(acc, "%6", "%12", k)        \
  G1_FMAC_BC(acc, "%7", "%13", k) G1_FMAC_BC(acc, "%8", "%14", k) G1_FMAC_BC(acc, "%9", "%15", k)
#define G1_C24(k0, k1, k2, k3)                                                                                     \
  {                                                                                                                \
    float t0, t1, t2, t3;                                                                                          \
    asm(G1_NOP G1_C6("%0", k0) G1_C6("%1", k1) G1_C6("%2", k2) G1_C6("%3", k3)                                     \
        : "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3)                                                               \
        : "v"(n[0]), "v"(n[1]), "v"(n[2]), "v"(f[0]), "v"(f[1]), "v"(f[2]), "v"(w[0]), "v"(w[1]), "v"(w[2]),       \
          "v"(v[0]), "v"(v[1]), "v"(v[2]));                                                                        \
    c[k0] = base[k0] + t0; c[k1] = base[k1] + t1; c[k2] = base[k2] + t2; c[k3] = base[k3] + t3;                    \
  }
  G1_C24(0, 1, 2, 3)
  G1_C24(4, 5, 6, 7)
  G1_C24(8, 9, 10, 11)
  G1_C24(12, 13, 14, 15)
#undef G1_C24
#undef G1_C6
}

// The factor in LDS: row m's entries of lane l at m * PFS + l (PFS odd: this order and the transposed reads of path_solve
// both touch every bank once)
constexpr int PFS = 65;
constexpr int PATH_FACTOR_WORDS = PP * PFS;

// c[m] -= (lane m's u) u for m = M0 .. M0 + N - 1, in one block that opens with the wait states (a block per row behind a
// wait of its own would leave the compiler room for a register copy in between). u passes through it, so what reads u by
// a lane swap next has waited too (N = 0: the wait alone).
template <int M0, int N>
__device__ __forceinline__ void path_update(float (&c)[PP], float& u) {
  static_assert(N >= 0 && N <= 6 && M0 + N <= PP, "path_update's rows");
#define G1_U(acc, u, k) "v_fmac_f32_dpp %" #acc ", %" #u ", -%" #u " row_newbcast:%" #k " row_mask:0xf bank_mask:0xf\n\t"
  float* const r = c + M0;
  if constexpr (N == 0)
    asm("s_nop 1" : "+v"(u));
  else if constexpr (N == 1)
    asm(G1_NOP G1_U(0, 1, 2) : "+v"(r[0]), "+v"(u) : "n"(M0));
  else if constexpr (N == 2)
    asm(G1_NOP G1_U(1, 2, 4) G1_U(0, 2, 3) : "+v"(r[0]), "+v"(r[1]), "+v"(u) : "n"(M0), "n"(M0 + 1));
  else if constexpr (N == 3)
    asm(G1_NOP G1_U(2, 3, 6) G1_U(1, 3, 5) G1_U(0, 3, 4)
        : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(u) : "n"(M0), "n"(M0 + 1), "n"(M0 + 2));
  else if constexpr (N == 4)
    asm(G1_NOP G1_U(3, 4, 8) G1_U(2, 4, 7) G1_U(1, 4, 6) G1_U(0, 4, 5)
        : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(u)
        : "n"(M0), "n"(M0 + 1), "n"(M0 + 2), "n"(M0 + 3));
  else if constexpr (N == 5)
    asm(G1_NOP G1_U(4, 5, 10) G1_U(3, 5, 9) G1_U(2, 5, 8) G1_U(1, 5, 7) G1_U(0, 5, 6)
        : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(r[4]), "+v"(u)
        : "n"(M0), "n"(M0 + 1), "n"(M0 + 2), "n"(M0 + 3), "n"(M0 + 4));
  else if constexpr (N == 6)
    asm(G1_NOP G1_U(5, 6, 12) G1_U(4, 6, 11) G1_U(3, 6, 10) G1_U(2, 6, 9) G1_U(1, 6, 8) G1_U(0, 6, 7)
        : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(r[4]), "+v"(r[5]), "+v"(u)
        : "n"(M0), "n"(M0 + 1), "n"(M0 + 2), "n"(M0 + 3), "n"(M0 + 4), "n"(M0 + 5));
#undef G1_U
}

// A = L' L, eliminated leaf first (the tree's sparsity, no fill): lane p's c[m] (m >= p) is A[m][p] of its path (the
// other entries may hold anything; the lanes and rows without a dof 0). Step k, all four paths at once: the pivot from
// lane k, row k = c[k] / sqrt(pivot), then its outer product off the rows above. Where paths meet:
//  - the waist's rows take the right arm's and the left arm's row in turn at each step, in both arm rows of lanes;
//  - the root's rows take the sum over all 29 hinges' rows as one product on the matrix cores, the Schur complement
//    D = X' X, X[k][r] = L[k][r] (hinge rows k = 6..34, root columns r < 6; 29 rows padded to 32): 8 steps of
//    v_mfma_f32_16x16x4f32, lane l giving A[l % 16][k'] = B[k'][l % 16] = X[6 + k'][l % 16] for k' = 4 t + l / 16
//    (columns past the 6th hold other entries, which reach only D's unused rows and columns), read back from the rows
//    stored in buf; lane l holds D[4 (l / 16) + e][l % 16].
// The factor is stored in buf, each row 0 from its diagonal on; the diagonal L[p][p] is returned. Bitwise the factor of
// the elimination one dof at a time (35 pivots, 132 pairs of a v_readlane and an FMA), on 16 pivots with 81 multiply-adds
// outside the matrix cores.
__device__ __forceinline__ float path_factor(float (&c)[PP], float* buf, int lane_) {
  const int lane = opaque_lane(lane_);
  const float tiny = 1e-30f;
  float diag = 0.f;
  static_for<PP - 1, -1, -1>([&](auto kc) {
    constexpr int k = decltype(kc)::value;
    if constexpr (k == 5) {
      float* st = buf + lane;
#pragma unroll
      for (int m = 6; m < PP; m++) st[m * PFS] = c[m];
      wsync();
      const int r = lane & 15, q = lane >> 4;
      // hinge row 6 + 4 t + q as (path row g, entry m): lane q's address runs on by PFS, from the next path's first
      // entries past the 2nd (t = 1: right leg; t = 5: right arm)
      const float* x = buf + q * PFS + r;
      const float *x1 = x + (q >= 2 ? 16 - 6 * PFS : 0), *x5 = x + (q >= 2 ? 16 - 7 * PFS : 0);
      float xv[8] = {x[6 * PFS], x1[10 * PFS], x[8 * PFS + 16], x[6 * PFS + 32], x[10 * PFS + 32], x5[14 * PFS + 32],
                     x[11 * PFS + 48], (buf + r)[15 * PFS + 48]};
      xv[7] = q == 0 ? xv[7] : 0.f;
      mfma4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < 8; t++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[t], xv[t], acc, 0, 0, 0);
      // D[0..3][p] from row 0's lanes, D[4..5][p] from row 1's
#pragma unroll
      for (int e = 0; e < 4; e++) c[e] -= lane_of(acc[e], r);
      c[4] -= lane_of(acc[0], 16 + r);
      c[5] -= lane_of(acc[1], 16 + r);
    }
    // the pivot floored at 1e-30, and its hardware 1 / sqrt (1 ulp), whose result takes a wait state before its use
    float rs;
    asm(G1_NOP "v_max_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf\n\tv_rsq_f32_e32 %0, %0\n\ts_nop 0"
        : "=&v"(rs) : "v"(c[k]), "v"(tiny), "n"(k));
    const float row = c[k] * rs;
    diag = lane_sel<PathEq<k>::m>(row, diag);
    float u = lane_sel0<PathLt<k>::m>(row);
    if constexpr (k >= 9) path_update<9, k - 9>(c, u);
    else if constexpr (k > 6) path_update<6, k - 6>(c, u);
    else if constexpr (k > 0 && k < 6) path_update<0, k>(c, u);
    c[k] = u;
    if constexpr (k >= 9) {
      float l, r;
      row_pairs(u, &l, &r);
      const float a = lane_sel<PATH_ARMS>(r, u), b = lane_sel0<PATH_ARMS>(l);  // a leg row's own, then nothing
      asm(G1_NOP "v_fmac_f32_dpp %0, %3, -%3" G1_BC(6) "v_fmac_f32_dpp %1, %3, -%3" G1_BC(7)
          "v_fmac_f32_dpp %2, %3, -%3" G1_BC(8) "v_fmac_f32_dpp %0, %4, -%4" G1_BC(6) "v_fmac_f32_dpp %1, %4, -%4" G1_BC(7)
          "v_fmac_f32_dpp %2, %4, -%4" G1_BC(8)
          : "+v"(c[6]), "+v"(c[7]), "+v"(c[8]) : "v"(a), "v"(b));
    }
  });
  float* st = buf + lane;
#pragma unroll
  for (int m = 0; m < 6; m++) st[m * PFS] = c[m];
  wsync();
  return diag;
}
__device__ __forceinline__ void path_load(const float* buf, float (&c)[PP], int lane) {
#pragma unroll
  for (int m = 0; m < PP; m++) c[m] = buf[m * PFS + lane];
}

// x = A^-1 b for N right-hand sides at once, A = L' L with the tree's sparsity: cf[m] = -L[m][p] / L[p][p] on the lanes
// p < m (row m of lane p's path), l[k] = -L[p][k] / L[p][p] on the lanes p > k, 0 on the others; dself = 1 / L[p][p], 0 on
// the lanes without a dof; b on every lane of its dof (0 on the lanes without one), x too. Each lane keeps its running
// value scaled by 1 / L[p][p], so the value broadcast at a step is already the solved entry. L' y = b leaf first: the
// limbs (row 2's arm, row 3's arm and both legs at once); the waist's and the root's dofs then take the right arm's
// terms, the left arm's, the waist's, the right leg's and the left leg's, their running values handed from row to row. L x
// = y root first, lane p along row p of L, each row alone. 49 steps of one multiply-add on the dependency chain, where
// the solve one dof at a time takes 68 steps of four instructions; bitwise its result.
template <int N>
__device__ __forceinline__ void path_solve_scaled(const float (&cf)[PP], const float (&l)[PP], float dself,
                                                  const float* b, float* x) {
  float z[N], acc[N], o0, o1;
#pragma unroll
  for (int i = 0; i < N; i++) z[i] = b[i] * dself;
  // one step z += (lane k's z) n on each chain; between a chain's steps two wait states, one of them the other chain's
#define G1_ONE(k, n) G1_FMAC_BC("%0", "%0", n, k) G1_NOP
#define G1_TWO(k, n) G1_FMAC_BC("%0", "%0", n, k) G1_FMAC_BC("%1", "%1", n, k) "s_nop 0\n\t"
#define G1_ADD1(k, n) G1_FMAC_BC("%0", "%1", n, k)
#define G1_ADD2(k, n) G1_FMAC_BC("%0", "%2", n, k) G1_FMAC_BC("%1", "%3", n, k)
#define G1_BOTH(ONE, TWO, IN)                                                                                      \
  if constexpr (N == 1) asm(G1_NOP ONE : "+v"(z[0]) : IN);                                                         \
  else asm(G1_NOP TWO "s_nop 0" : "+v"(z[0]), "+v"(z[N - 1]) : IN);
#define G1_ACC(ONE, TWO, IN)                                                                                       \
  if constexpr (N == 1) asm(G1_NOP ONE "s_nop 1" : "+v"(acc[0]) : "v"(z[0]), IN);                                  \
  else asm(G1_NOP TWO "s_nop 1" : "+v"(acc[0]), "+v"(acc[N - 1]) : "v"(z[0]), "v"(z[N - 1]), IN);
#define G1_IN(...) __VA_ARGS__
  G1_BOTH(G1_ONE(15, "%1") G1_ONE(14, "%2") G1_ONE(13, "%3") G1_ONE(12, "%4") G1_ONE(11, "%5") G1_ONE(10, "%6")
          G1_ONE(9, "%7"),
          G1_TWO(15, "%2") G1_TWO(14, "%3") G1_TWO(13, "%4") G1_TWO(12, "%5") G1_TWO(11, "%6") G1_TWO(10, "%7")
          G1_TWO(9, "%8"),
          G1_IN("v"(cf[15]), "v"(cf[14]), "v"(cf[13]), "v"(cf[12]), "v"(cf[11]), "v"(cf[10]), "v"(cf[9])))
#pragma unroll
  for (int i = 0; i < N; i++) row_pairs(z[i], &o0, &acc[i]);  // row 2's shared dofs go on from row 3's
  G1_ACC(G1_ADD1(15, "%2") G1_ADD1(14, "%3") G1_ADD1(13, "%4") G1_ADD1(12, "%5") G1_ADD1(11, "%6") G1_ADD1(10, "%7")
         G1_ADD1(9, "%8"),
         G1_ADD2(15, "%4") G1_ADD2(14, "%5") G1_ADD2(13, "%6") G1_ADD2(12, "%7") G1_ADD2(11, "%8") G1_ADD2(10, "%9")
         G1_ADD2(9, "%10"),
         G1_IN("v"(cf[15]), "v"(cf[14]), "v"(cf[13]), "v"(cf[12]), "v"(cf[11]), "v"(cf[10]), "v"(cf[9])))
#pragma unroll
  for (int i = 0; i < N; i++) z[i] = lane_sel<PATH_SHARED2>(acc[i], z[i]);
  G1_BOTH(G1_ONE(8, "%1") G1_ONE(7, "%2") G1_ONE(6, "%3"), G1_TWO(8, "%2") G1_TWO(7, "%3") G1_TWO(6, "%4"),
          G1_IN("v"(cf[8]), "v"(cf[7]), "v"(cf[6])))
#pragma unroll
  for (int i = 0; i < N; i++) {
    row_halves(z[i], &o0, &o1);  // row 2's root on to rows 0 and 1
    row_pairs(o1, &acc[i], &o0);
  }
#define G1_LEGS                                                                                                    \
  G1_ACC(G1_ADD1(11, "%2") G1_ADD1(10, "%3") G1_ADD1(9, "%4") G1_ADD1(8, "%5") G1_ADD1(7, "%6") G1_ADD1(6, "%7"),  \
         G1_ADD2(11, "%4") G1_ADD2(10, "%5") G1_ADD2(9, "%6") G1_ADD2(8, "%7") G1_ADD2(7, "%8") G1_ADD2(6, "%9"),  \
         G1_IN("v"(cf[11]), "v"(cf[10]), "v"(cf[9]), "v"(cf[8]), "v"(cf[7]), "v"(cf[6])))
  G1_LEGS  // the right leg's terms (row 1)
#pragma unroll
  for (int i = 0; i < N; i++) {
    row_pairs(acc[i], &o0, &o1);
    acc[i] = o1;
  }
  G1_LEGS  // the left leg's (row 0)
#undef G1_LEGS
#pragma unroll
  for (int i = 0; i < N; i++) {
    row_pairs(acc[i], &o0, &o1);
    row_halves(o0, &acc[i], &o1);  // row 0's root in every row; row 2's waist also in row 3
    row_pairs(z[i], &o0, &o1);
    z[i] = lane_sel<PATH_WAIST3>(o0, z[i]);
    z[i] = lane_sel<PATH_ROOT>(acc[i], z[i]);
  }
  G1_BOTH(G1_ONE(5, "%1") G1_ONE(4, "%2") G1_ONE(3, "%3") G1_ONE(2, "%4") G1_ONE(1, "%5"),
          G1_TWO(5, "%2") G1_TWO(4, "%3") G1_TWO(3, "%4") G1_TWO(2, "%5") G1_TWO(1, "%6"),
          G1_IN("v"(cf[5]), "v"(cf[4]), "v"(cf[3]), "v"(cf[2]), "v"(cf[1])))
#pragma unroll
  for (int i = 0; i < N; i++) z[i] *= dself;
  G1_BOTH(G1_ONE(0, "%1") G1_ONE(1, "%2") G1_ONE(2, "%3") G1_ONE(3, "%4") G1_ONE(4, "%5") G1_ONE(5, "%6")
          G1_ONE(6, "%7") G1_ONE(7, "%8") G1_ONE(8, "%9") G1_ONE(9, "%10") G1_ONE(10, "%11") G1_ONE(11, "%12")
          G1_ONE(12, "%13") G1_ONE(13, "%14") G1_ONE(14, "%15"),
          G1_TWO(0, "%2") G1_TWO(1, "%3") G1_TWO(2, "%4") G1_TWO(3, "%5") G1_TWO(4, "%6") G1_TWO(5, "%7")
          G1_TWO(6, "%8") G1_TWO(7, "%9") G1_TWO(8, "%10") G1_TWO(9, "%11") G1_TWO(10, "%12") G1_TWO(11, "%13")
          G1_TWO(12, "%14") G1_TWO(13, "%15") G1_TWO(14, "%16"),
          G1_IN("v"(l[0]), "v"(l[1]), "v"(l[2]), "v"(l[3]), "v"(l[4]), "v"(l[5]), "v"(l[6]), "v"(l[7]), "v"(l[8]),
                "v"(l[9]), "v"(l[10]), "v"(l[11]), "v"(l[12]), "v"(l[13]), "v"(l[14])))
#undef G1_IN
#undef G1_ACC
#undef G1_BOTH
#undef G1_ADD2
#undef G1_ADD1
#undef G1_TWO
#undef G1_ONE
#pragma unroll
  for (int i = 0; i < N; i++) x[i] = z[i];
}

// from path_factor's rows (in registers: c, and in buf) and diagonal
__device__ __forceinline__ float path_solve(const float* buf, const float (&c)[PP], float diag, float b, int lane_) {
  const int lane = opaque_lane(lane_);
  float l[PP], cf[PP], x;
  const float* row = buf + (lane & 15) * PFS + (lane & 48);
#pragma unroll
  for (int k = 0; k < PP - 1; k++) l[k] = row[k];
  const float dself = lane_sel0<PATH_VALID>(1.f / diag), ds = -dself;
#pragma unroll
  for (int m = 1; m < PP; m++) cf[m] = c[m] * ds;
#pragma unroll
  for (int k = 0; k < PP - 1; k++) l[k] *= ds;
  path_solve_scaled<1>(cf, l, dself, &b, &x);
  return x;
}

// from a packed factor (lower, TRI layout) of the tree's sparsity; Lp readable up to its word 34 * 35 / 2 + 70 (the
// lanes without a dof read past the factor and drop it)
template <int N>
__device__ __forceinline__ void path_solve_packed(const float* Lp, int pd, int lane_, const float* b, float* x) {
  const int lane = opaque_lane(lane_), g = lane >> 4, o6 = g < 2 ? 6 * g : 12, o9 = g < 3 ? 6 * g : 19;
  // row m's dof is m + o: its packed row starts at tri(m) + m o + o (o + 1) / 2
  const float *col = Lp + pd, *row = Lp + tri(pd, 0);
  const float *c6 = col + o6 * (o6 + 1) / 2, *c9 = col + o9 * (o9 + 1) / 2, *r6 = row + o6, *r9 = row + o9;
  const float dself = lane_sel0<PATH_VALID>(1.f / row[pd]), ds = -dself;
  float cf[PP], l[PP];
#pragma unroll
  for (int m = 1; m < PP; m++) cf[m] = m < 6 ? col[tri(m, 0)] : m < 9 ? c6[m * o6 + tri(m, 0)] : c9[m * o9 + tri(m, 0)];
#pragma unroll
  for (int k = 0; k < PP - 1; k++) l[k] = (k < 6 ? row : k < 9 ? r6 : r9)[k];
  static_for<0, PP, 1>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    if constexpr (m > 0) cf[m] = lane_sel0<PathLt<m>::m>(cf[m] * ds);
    if constexpr (m < PP - 1) l[m] = lane_sel0<PathGt<m>::m>(l[m] * ds);
  });
  path_solve_scaled<N>(cf, l, dself, b, x);
}

}  // namespace g1k
