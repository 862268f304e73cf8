// Kinematics outputs of a state and their VJP (the reference's k_kin / k_kin_vjp, g1_engine/kinematics.py:1-45; MuJoCo
// MJX's kinematics + com_pos + com_vel semantics, mujoco 3.17 smooth.py):
//   qpos_n       qpos with the free joint's quaternion normalized;
//   xpos, xquat  the body frames (world body 0 at the origin, identity); the root from qpos; a hinge body composed
//                from its parent: x_b = x_p + R_p p_b, Q_b = Q_p (x) q_b (x) (axis_b, qpos angle);
//   subtree_com  sum over the subtree of m_c xipos_c / its mass, xipos_c = x_c + R_c ipos_c (the torso's ipos + com);
//                the world body's is body 1's;
//   cvel         [W_b; V_b + W_b x (c - x_b)], c = subtree_com[1]: W_b the body's angular velocity, V_b its origin's
//                velocity (root: R_1 qvel[3:6], qvel[0:3]); body 0 zeros.
// Two worlds per wave64, one in each half: lane b of a half = body b. A body lane forms its own hinge's local transform
// (one sine and cosine), then composes its pose and twist along its chain from the root; the sums over the tree run a
// column per lane (tree_sums).
//
// What bounds both is the dependent chain of a wave up to some thousand worlds (the waves are all resident), then vector
// issue; HBM would allow 4.4 us at 4096 worlds for the pair. A body takes one of a half wave's 32 lanes, so a second
// world costs no further instruction. One world per wave, every body lane rotating each hinge of its chain (ten sines
// and cosines) and summing its subtree in a masked loop over the bodies, took, k_kin / k_kin_vjp: 13.2 / 19.9 us at 1024
// worlds, 17.8 / 26.6 at 4096, 45.1 / 79.5 at 16384; this form 8.1 / 8.8, 10.0 / 12.8 and 17.3 / 24.2 (the twists
// composed down the chain, not from differences of positions: cvel's error against float64 falls too).
//
// VJP (reverse mode of the same map; cotangents of the five outputs -> of qpos and qvel): per body the "own"
// cotangents of its origin (x bar: a world force) and of its rotation (tau bar: a world torque; a quaternion cotangent
// g gives 1/2 vec(g Q*)), with the sums over the tree in closed form:
//   cvel:        V bar_b = g_lin, W bar_b = g_ang + (c - x_b) x g_lin, x bar_b += W_b x g_lin, c bar += g_lin x W_b;
//   subtree_com: S bar_b = g_sc_b / m_sub_b; xipos bar_c = m_c sum of S bar over c's path; x bar_c += it,
//                tau bar_c += (xipos_c - x_c) x it;
//   velocities:  V tot_b = sum_sub V bar, W tot_b = sum_sub (W bar_d + x_d x V bar_d) - x_b x V tot_b; hinge rate bar
//                z_b . W tot_b, tau bar_b += qd_b z_b x W tot_b; x bar_b += V tot_b x W_parent - (V tot_b - V bar_b) x W_b;
//                root: qvel[0:3] bar = V tot_1, qvel[3:6] bar = R_1' W tot_1, tau bar_1 += W_1 x W tot_1;
//   poses:       F_b = sum_sub x bar, N_b = sum_sub (tau bar_d + x_d x x bar_d) - x_b x F_b; hinge angle bar z_b . N_b;
//                root position bar F_1; quaternion: a = 2 [0; N_1] (x) u + g_xquat_1 + g_qpos_n[3:7],
//                raw bar = (a - u (u . a)) / |q| (MJX's normalization).
// The incoming cotangents gq_in / gv_in (nullable) are added to the result last.
#include "g1_device.h"

namespace g1k {

constexpr int HALF = 32;  // lanes of a world
static_assert(NB <= HALF, "a body per lane of a half wave");

struct __align__(16) Kin {
  // a hinge body's local transform: quat (x) hinge rotation (0..3), its offset in its parent's frame (4..6), its
  // joint rate (7), its axis in the parent's frame (8..10); then the columns of the VJP's sums
  float T[NB][12];
  float P[NB][4];  // m xipos, summed over subtrees; then the VJP's S bar (row 0 zero)
};

// Sums over subtrees, a column per lane: lane c < n of a half takes column c of every body (rows of `stride` floats),
// adds each body into its parent, highest id first (a body's id is above its parent's, so each is complete when it is
// added), and stores the sums in place. Lanes past the columns compute a copy of the last and do not store.
template <int stride>
__device__ __forceinline__ void tree_sums(float* rows, int n, int l) {
  float* col = rows + min(l, n - 1);
  float v[NB];
#pragma unroll
  for (int b = 1; b < NB; b++) v[b] = col[b * stride];
  static_for<NB - 1, 1, -1>([&](auto bc) {
    constexpr int b = decltype(bc)::value;
    static_assert(BODY_PARENT[b] >= 1 && BODY_PARENT[b] < b, "bodies numbered parents first");
    v[BODY_PARENT[b]] += v[b];
  });
  if (l < n)
#pragma unroll
    for (int b = 1; b < NB; b++) col[b * stride] = v[b];
  wsync();
}

constexpr Arr<float, NB> make_submass() {  // the subtrees' masses (the world body's row: body 1's)
  Arr<float, NB> r{};
  double m[NB] = {};
  for (int b = NB - 1; b >= 1; b--) {
    m[b] += BODY_MASS[b];
    if (BODY_PARENT[b] >= 1) m[BODY_PARENT[b]] += m[b];
  }
  for (int b = 0; b < NB; b++) r.v[b] = (float)m[b < 1 ? 1 : b];
  return r;
}
__constant__ Arr<float, NB> cSubmass = make_submass();

// the body at step i of the root-to-leaf path that body b lies on (PATHS; bodies ascend along a path)
__device__ __forceinline__ int path_step(int b, int i) {
  static_assert(PATHS.lo[0] == 2 && PATHS.lo[1] == 8 && PATHS.lo[2] == 14 && PATHS.hi[2] == 14 && PATHS.hi[3] == 21,
                "the paths of the walks");
  const int lo = b >= 14 ? 14 : b >= 8 ? 8 : 2, hi = b >= 24 ? 21 : lo;
  return (i < 3 ? lo : hi) + i;
}

// what a lane holds of its body after the forward map
struct Body {
  float Q[4], X[3], Z[3], W[3], V[3], Wp[3];  // pose, world hinge axis, angular velocity, the origin's, the parent's W
  float rip[3], qd, qa, inv;                  // xipos - x, hinge rate and angle, 1 / |root quaternion|
};

// the forward map of a half's world; leaves the subtree sums of m xipos in s.P
__device__ __forceinline__ void kin_forward(Kin& s, int b, int l, const float* __restrict__ q,
                                            const float* __restrict__ v, const float* __restrict__ com, Body& B) {
  const bool hinge = b >= 2;
  float q1[4], wl[3], cm[3];
  for (int k = 0; k < 3; k++) { B.X[k] = q[k]; B.V[k] = v[k]; wl[k] = v[3 + k]; cm[k] = com[k]; }
  for (int k = 0; k < 4; k++) q1[k] = q[3 + k];
  B.qa = hinge ? q[b + 5] : 0.f;
  B.qd = hinge ? v[b + 4] : 0.f;
  const float qb[4] = {cQuat[4 * b], cQuat[4 * b + 1], cQuat[4 * b + 2], cQuat[4 * b + 3]};
  const float ax[3] = {cAxis[3 * b], cAxis[3 * b + 1], cAxis[3 * b + 2]};
  float ip[3] = {cIpos[3 * b], cIpos[3 * b + 1], cIpos[3 * b + 2]};
  const float m = b >= 1 ? cMass[b] : 0.f;
  {
    float sn, cs, ql[4], al[3];
    sincosf(0.5f * B.qa, &sn, &cs);
    const float ha[4] = {cs, sn * ax[0], sn * ax[1], sn * ax[2]};
    qmul(qb, ha, ql);
    qrot(qb, ax, al);  // the hinge rotation keeps its own axis
    if (l < NB) {
      float* h = s.T[b];
      for (int k = 0; k < 4; k++) h[k] = ql[k];
      for (int k = 0; k < 3; k++) { h[4 + k] = cPos[3 * b + k]; h[8 + k] = al[k]; }
      h[7] = B.qd;
    }
  }
  B.inv = 1.f / sqrtf(q1[0] * q1[0] + q1[1] * q1[1] + q1[2] * q1[2] + q1[3] * q1[3]);
  for (int k = 0; k < 4; k++) B.Q[k] = q1[k] * B.inv;
  qrot(B.Q, wl, B.W);
  for (int k = 0; k < 3; k++) B.Z[k] = B.Wp[k] = 0.f;
  wsync();
#pragma unroll
  for (int i = 0; i < PATH_STEPS; i++) {
    const int k = path_step(b, i);
    if (k <= b) {
      const float* h = s.T[k];
      const float ql[4] = {h[0], h[1], h[2], h[3]}, pb[3] = {h[4], h[5], h[6]}, qd = h[7], al[3] = {h[8], h[9], h[10]};
      float t[3], u[3], Qn[4];
      qrot(B.Q, pb, t);
      qrot(B.Q, al, B.Z);
      qmul(B.Q, ql, Qn);
      cross(B.W, t, u);
      for (int e = 0; e < 4; e++) B.Q[e] = Qn[e];
      for (int e = 0; e < 3; e++) {
        B.X[e] += t[e];
        B.V[e] += u[e];
        B.Wp[e] = B.W[e];
        B.W[e] += B.Z[e] * qd;
      }
    }
  }
  if (b == 0)
    for (int k = 0; k < 3; k++) { B.X[k] = 0.f; B.Q[k] = k == 0 ? 1.f : 0.f; B.Q[3] = 0.f; }
  if (b == TORSO_BODY)
    for (int k = 0; k < 3; k++) ip[k] += cm[k];
  qrot(B.Q, ip, B.rip);
  if (l < NB)
    for (int k = 0; k < 3; k++) s.P[b][k] = m * (B.X[k] + B.rip[k]);
  wsync();
  tree_sums<4>(&s.P[0][0], 3, l);
}

__global__ __launch_bounds__(64) void k_kin(int nw, const float* __restrict__ qpos, const float* __restrict__ qvel,
                                            const float* __restrict__ com, float* __restrict__ qn,
                                            float* __restrict__ xpos, float* __restrict__ xquat,
                                            float* __restrict__ cvel, float* __restrict__ osc) {
  __shared__ Kin sh[2];
  const int l = threadIdx.x % HALF, half = threadIdx.x / HALF;
  const int wi = 2 * blockIdx.x + half;
  if (2 * (int)blockIdx.x >= nw) return;
  const int w = min(wi, nw - 1);  // an odd batch's last half repeats the last world and stores nothing
  const int b = min(l, NB - 1);
  Kin& s = sh[half];
  Body B;
  kin_forward(s, b, l, qpos + (size_t)w * NQ, qvel + (size_t)w * NV, com + (size_t)w * 3, B);
  const int sb = max(b, 1);
  float sc[3], r[3], u[3], cv[6];
  for (int k = 0; k < 3; k++) {
    sc[k] = s.P[sb][k] / cSubmass[b];
    r[k] = s.P[1][k] / cSubmass[1] - B.X[k];
  }
  cross(B.W, r, u);
  for (int k = 0; k < 3; k++) {
    cv[k] = b >= 1 ? B.W[k] : 0.f;
    cv[3 + k] = b >= 1 ? B.V[k] + u[k] : 0.f;
  }
  if (wi >= nw || l >= NB) return;
  const size_t o = (size_t)w * NB + b;
  float* qo = qn + (size_t)w * NQ;
  if (b >= 2) qo[b + 5] = B.qa;
  if (b == 1) {
    for (int k = 0; k < 3; k++) qo[k] = B.X[k];
    for (int k = 0; k < 4; k++) qo[3 + k] = B.Q[k];
  }
  for (int k = 0; k < 3; k++) { xpos[3 * o + k] = B.X[k]; osc[3 * o + k] = sc[k]; }
  for (int k = 0; k < 4; k++) xquat[4 * o + k] = B.Q[k];
  for (int k = 0; k < 6; k++) cvel[6 * o + k] = cv[k];
}

__global__ __launch_bounds__(64) void k_kin_vjp(int nw, const float* __restrict__ qpos,
                                                const float* __restrict__ qvel, const float* __restrict__ com,
                                                const float* __restrict__ gqn, const float* __restrict__ gxpos,
                                                const float* __restrict__ gxquat, const float* __restrict__ gcvel,
                                                const float* __restrict__ gsc, const float* __restrict__ gq_in,
                                                const float* __restrict__ gv_in, float* __restrict__ gq,
                                                float* __restrict__ gv) {
  __shared__ Kin sh[2];
  const int l = threadIdx.x % HALF, half = threadIdx.x / HALF;
  const int wi = 2 * blockIdx.x + half;
  if (2 * (int)blockIdx.x >= nw) return;
  const int w = min(wi, nw - 1);  // an odd batch's last half repeats the last world and stores nothing
  const int b = min(l, NB - 1);
  const bool body = b >= 1, hinge = b >= 2;
  Kin& s = sh[half];
  // the cotangents, loaded before the forward map hides their latency
  const size_t o = (size_t)w * NB + b;
  const float* gn = gqn + (size_t)w * NQ;
  const float* iq = gq_in ? gq_in + (size_t)w * NQ : nullptr;
  const float* iv = gv_in ? gv_in + (size_t)w * NV : nullptr;
  float gA[3], gL[3], gX[3], gS[3], gQ[4], g0[3], gN[7], iQ[7], iV[6];
  for (int k = 0; k < 3; k++) {
    gA[k] = gcvel[6 * o + k];
    gL[k] = body ? gcvel[6 * o + 3 + k] : 0.f;
    gX[k] = gxpos[3 * o + k];
    gS[k] = gsc[3 * o + k];
    g0[k] = gsc[(size_t)w * NB * 3 + k];
  }
  for (int k = 0; k < 4; k++) gQ[k] = gxquat[4 * o + k];
  for (int k = 0; k < 7; k++) { gN[k] = gn[hinge ? b + 5 : k]; iQ[k] = iq ? iq[hinge ? b + 5 : k] : 0.f; }
  for (int k = 0; k < 6; k++) iV[k] = iv ? iv[hinge ? b + 4 : k] : 0.f;
  Body B;
  kin_forward(s, b, l, qpos + (size_t)w * NQ, qvel + (size_t)w * NV, com + (size_t)w * 3, B);
  // cvel: own V bar, W bar, x bar; the reference point's cotangent
  float Wbar[3], xb[3], tb[3] = {0.f, 0.f, 0.f}, cc[3], u[3], r[3];
  for (int k = 0; k < 3; k++) r[k] = s.P[1][k] / cSubmass[1] - B.X[k];
  cross(r, gL, u);
  for (int k = 0; k < 3; k++) Wbar[k] = gA[k] + u[k];
  cross(B.W, gL, xb);
  for (int k = 0; k < 3; k++) { cc[k] = -xb[k]; xb[k] += gX[k]; }
  if (hinge) {  // a hinge body's quaternion cotangent as a world torque: 1/2 vec(g Q*)
    const float qc[4] = {B.Q[0], -B.Q[1], -B.Q[2], -B.Q[3]};
    float t[4];
    qmul(gQ, qc, t);
    for (int k = 0; k < 3; k++) tb[k] = 0.5f * t[1 + k];
  }
  // subtree sums of V bar, of W bar + x x V bar, of the reference point's cotangent (the root's row: its sum)
  cross(B.X, gL, u);
  if (l < NB)
    for (int k = 0; k < 3; k++) { s.T[b][k] = gL[k]; s.T[b][3 + k] = Wbar[k] + u[k]; s.T[b][6 + k] = cc[k]; }
  wsync();
  tree_sums<12>(&s.T[0][0], 9, l);
  float Vt[3], Wt[3];
  for (int k = 0; k < 3; k++) { Vt[k] = s.T[b][k]; Wt[k] = s.T[b][3 + k]; }
  // subtree COM cotangents -> S bar_b (body 0's goes to body 1, with the reference point's)
  if (l < NB)
    for (int k = 0; k < 3; k++)
      s.P[b][k] = body ? (b == 1 ? gS[k] + (g0[k] + s.T[1][6 + k]) : gS[k]) / cSubmass[b] : 0.f;
  wsync();
  {  // xipos bar_c = m_c sum of S bar over c's path (root .. c)
    float a[3] = {s.P[1][0], s.P[1][1], s.P[1][2]};
#pragma unroll
    for (int i = 0; i < PATH_STEPS; i++) {
      const int k = path_step(b, i), j = k <= b ? k : 0;
      for (int e = 0; e < 3; e++) a[e] += s.P[j][e];
    }
    const float m = cMass[b];
    for (int k = 0; k < 3; k++) { a[k] *= m; xb[k] += a[k]; }
    cross(B.rip, a, u);
    for (int k = 0; k < 3; k++) tb[k] += u[k];
  }
  // velocities
  cross(B.X, Vt, u);
  for (int k = 0; k < 3; k++) Wt[k] -= u[k];
  float dv[3];
  for (int k = 0; k < 3; k++) dv[k] = Vt[k] - gL[k];
  cross(dv, B.W, u);
  for (int k = 0; k < 3; k++) xb[k] -= u[k];
  const float rate = dot3(B.Z, Wt);  // hinge rate bar
  if (hinge) {
    cross(Vt, B.Wp, u);
    for (int k = 0; k < 3; k++) xb[k] += u[k];
    cross(B.Z, Wt, u);
    for (int k = 0; k < 3; k++) tb[k] += B.qd * u[k];
  } else {
    cross(B.W, Wt, u);
    for (int k = 0; k < 3; k++) tb[k] += u[k];
  }
  // poses: F_b = sum_sub x bar, N_b = sum_sub (tau bar + x x x bar) - x_b x F_b
  cross(B.X, xb, u);
  wsync();
  if (l < NB)
    for (int k = 0; k < 3; k++) { s.T[b][k] = xb[k]; s.T[b][3 + k] = tb[k] + u[k]; }
  wsync();
  tree_sums<12>(&s.T[0][0], 6, l);
  float F[3], N[3];
  for (int k = 0; k < 3; k++) { F[k] = s.T[b][k]; N[k] = s.T[b][3 + k]; }
  cross(B.X, F, u);
  for (int k = 0; k < 3; k++) N[k] -= u[k];
  if (wi >= nw || l >= NB) return;
  // outputs: hinge bodies write their angle's and rate's entries; the root its position, quaternion, velocities
  float* oq = gq + (size_t)w * NQ;
  float* ov = gv + (size_t)w * NV;
  if (hinge) {
    const int qa = b + 5, da = b + 4;
    const float ang = dot3(B.Z, N) + gN[0];
    oq[qa] = iq ? ang + iQ[0] : ang;
    ov[da] = iv ? rate + iV[0] : rate;
  }
  if (b == 1) {
    for (int k = 0; k < 3; k++) {
      const float pq = F[k] + gN[k];
      oq[k] = iq ? pq + iQ[k] : pq;
      ov[k] = iv ? Vt[k] + iV[k] : Vt[k];
    }
    float wl[3];
    qrot_inv(B.Q, Wt, wl);
    for (int k = 0; k < 3; k++) ov[3 + k] = iv ? wl[k] + iV[3 + k] : wl[k];
    const float n4[4] = {0.f, N[0], N[1], N[2]};
    float a[4];
    qmul(n4, B.Q, a);
    for (int k = 0; k < 4; k++) a[k] = 2.f * a[k] + gQ[k] + gN[3 + k];
    const float ua = B.Q[0] * a[0] + B.Q[1] * a[1] + B.Q[2] * a[2] + B.Q[3] * a[3];
    for (int k = 0; k < 4; k++) {
      const float g = (a[k] - B.Q[k] * ua) * B.inv;
      oq[3 + k] = iq ? g + iQ[3 + k] : g;
    }
  }
}

int launch_kinematics(hipStream_t st, int nw, const float* qpos, const float* qvel, const float* com, float* qn,
                      float* xpos, float* xquat, float* cvel, float* sc) {
  if (nw <= 0) return 0;
  hipLaunchKernelGGL(k_kin, dim3((nw + 1) / 2), dim3(64), 0, st, nw, qpos, qvel, com, qn, xpos, xquat, cvel, sc);
  return (int)hipGetLastError();
}

int launch_kinematics_vjp(hipStream_t st, int nw, const float* qpos, const float* qvel, const float* com,
                          const float* gqn, const float* gxpos, const float* gxquat, const float* gcvel,
                          const float* gsc, const float* gq_in, const float* gv_in, float* gq, float* gv) {
  if (nw <= 0) return 0;
  hipLaunchKernelGGL(k_kin_vjp, dim3((nw + 1) / 2), dim3(64), 0, st, nw, qpos, qvel, com, gqn, gxpos, gxquat, gcvel, gsc,
                     gq_in, gv_in, gq, gv);
  return (int)hipGetLastError();
}

}  // namespace g1k
