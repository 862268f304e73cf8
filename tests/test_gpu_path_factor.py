"""The factorizations and solves in the path layout (csrc/g1_path.h) at the places where it can go wrong: no
constraint rows at all; a limit row on every hinge (every diagonal entry), on the waist's three (shared by both arm
paths), on one leg's or one arm's; contacts on one limb; contacts between robot bodies, whose assembly goes through
the packed form, on and off one path, fewer and more than are assembled at once. One substep, from its tape record, against
float64 (the oracle) at the record's own a* and against a float32 replay of the solves one dof at a time."""
import numpy as np
import pytest

import oracle
from nablaengine_amd import synthetic

pytestmark = pytest.mark.gpu
KEYS = ("qpos", "qvel", "warm", "ctrl", "friction", "com")
REC_FLAGS, REC_CLAMP, REC_CZONE, REC_CON, REC_ASTAR, REC_AADV, REC_LH, REC_LQ = 1, 2, 8, 16, 128, 164, 200, 832
FLAG_SINGULAR = 1 << 10
MODEL = synthetic.model()
TREE = np.array([[bool((MODEL["body_ancmask"][MODEL["dof_body"][i]] >> MODEL["dof_body"][j]) & 1) for j in range(35)]
                 for i in range(35)])
HINGES = {"legs_left": (6, 12), "legs_right": (12, 18), "waist": (18, 21), "arm_left": (21, 28), "arm_right": (28, 35),
          "all": (6, 35)}


def _states(kind, n):
    st = synthetic.states(n, config=4 if kind == "tangled" else 1, seed=77)
    rng = np.random.default_rng(78)
    if kind == "tangled":
        return st
    st["qpos"][:, 2] = 2.0  # in the air
    if kind in HINGES:  # past the upper limit of each hinge of the range
        hi = np.asarray(synthetic.model()["dof_range"]).reshape(35, 2)[:, 1]
        a, b = HINGES[kind]
        st["qpos"][:, a + 1:b + 1] = hi[a:b] + rng.uniform(0.01, 0.05, (n, b - a))
    elif kind == "feet":  # the legs rolled inwards until the feet's 7 spheres each overlap: 1 to 28 contacts
        st["qpos"][:, 7:19] = rng.normal(0.0, 0.03, (n, 12))
        st["qpos"][:, 8] -= 0.16
        st["qpos"][:, 14] += 0.16
    elif kind == "one_foot":  # rolled about x until only one foot's spheres touch
        st["qpos"][:, 2] = 0.74
        st["qpos"][:, 3:7] = [np.cos(0.15), np.sin(0.15), 0, 0]
    return {k: np.ascontiguousarray(v, np.float32) for k, v in st.items()}


def _unpack(x):
    L = np.zeros((35, 35))
    L[np.tril_indices(35)] = x[:630]
    return L


def _self_contacts(rec):
    """Per record (float32 words): its contacts between two robot bodies with a row in the quadratic zone."""
    w = rec.view(np.uint32)
    c = np.arange(64)
    zone = (w[:, REC_CZONE + c // 8] >> (4 * (c % 8)).astype(np.uint32)) & 15
    pair = (w[:, REC_CON + c // 2] >> (16 * (c % 2)).astype(np.uint32)) & 511
    body1 = np.asarray(MODEL["geom_body"])[np.asarray(MODEL["pair_g1"] + [0] * 10)[pair]]
    return ((c < (w[:, :1] & 255)) & (zone != 0) & (body1 != 0)).sum(1)


def _centres(s, rec):
    """What the direction between two geom centres (or axis points) a distance nu apart loses by their float32 positions
    (4e-7 m each, FK's error against float64), for a record flagged for a nu below 5 mm; else 0."""
    if not rec[REC_FLAGS:REC_FLAGS + 1].view(np.uint32)[0] & FLAG_SINGULAR:
        return 0.0
    nu = []
    for r in oracle.contacts(s["qpos"], s["qvel"], s["ctrl"], s["com"], float(s["friction"])):
        g1, g2 = MODEL["pair_g1"][int(r[0])], MODEL["pair_g2"][int(r[0])]
        if MODEL["geom_body"][g1] != 0:
            nu.append(r[2] + MODEL["geom_size"][3 * g1] + MODEL["geom_size"][3 * g2])
    return 8e-7 / min(nu)


def _taped(kind, B):
    import torch
    from nablaengine_amd import torch_ffi
    st = _states(kind, B)
    args = [torch.from_numpy(st[k]).cuda() for k in KEYS]
    _, _, _, info, tape = torch_ffi.forward(*args, iterations=50, substeps=1, tape=True)
    rec = tape.cpu().numpy().reshape(B, -1)
    s64 = {k: st[k].astype(np.float64) for k in KEYS}
    s64["warm"] = rec[:, REC_ASTAR:REC_ASTAR + 35].astype(np.float64)  # with 0 iterations: the zones at the record's a*
    return args, info.cpu().numpy(), tape, rec, s64


@pytest.mark.parametrize("kind", ["flight", "all", "waist", "legs_left", "legs_right", "arm_left", "arm_right",
                                  "one_foot", "tangled", "feet"])
def test_path_factors_vs_oracle(kind):
    """L_Q against float64's factor of M + h kv, L_H' L_H against H at the zones of the record's a*, and a_adv's residual
    in (M + h kv) a_adv = M a*. Tolerances: the elimination's backward error is at most about n eps = 35 x 6e-8 = 2e-6 of
    the largest entry, and M and H themselves are sums of some tens of float32 terms (a few 1e-7 each): 1e-5, and what
    the contact normals of nearly coincident centres lose (_centres); the residual is that of the factor times |x|
    (1e-5 |Q| |a_adv|, rows against the largest)."""
    B = 12
    _, info, _, recs, s64 = _taped(kind, B)
    hkv = MODEL["timestep"] * np.diag(np.asarray(MODEL["dof_kv"]))
    for w in range(B):
        s, rec = {k: v[w] for k, v in s64.items()}, recs[w]
        M, H = oracle.substep_hessian(s["qpos"], s["qvel"], s["warm"], s["ctrl"], float(s["friction"]), s["com"],
                                      iterations=0)
        ref = oracle.ltl(M + hkv)
        assert np.abs(_unpack(rec[REC_LQ:]) * TREE - ref).max() <= 1e-5 * np.abs(ref).max(), w
        a, adv = s["warm"], rec[REC_AADV:REC_AADV + 35].astype(np.float64)
        res = (M + hkv) @ adv - M @ a
        assert np.abs(res).max() <= 1e-5 * (np.abs(M + hkv) @ np.abs(adv)).max(), w
        assert not rec[REC_FLAGS:REC_FLAGS + 1].view(np.uint32)[0] & (4 | 16), w
        L = _unpack(rec[REC_LH:])
        assert np.abs(L.T @ L - H).max() <= (1e-5 + _centres(s, rec)) * np.abs(H).max(), w
    if kind in HINGES:
        a, b = HINGES[kind]
        assert (info[:, 2] >= b - a).all(), info  # the limit rows are there
    if kind == "feet":
        n = _self_contacts(recs)  # past one chunk of 8 contacts' edge rows, and batches of 4 that are not full
        assert (n > 8).any() and (n % 4 != 0).any(), n
    if kind == "flight":
        assert (info[:, 2] == 0).sum() >= 4, info  # worlds without any row (a hand may touch the hip in the others)


@pytest.mark.parametrize("kind", ["flight", "all", "waist", "one_foot", "tangled", "feet"])
def test_path_solves_in_the_adjoint(kind):
    """One substep's VJP (exact mode) on the same states, whose tapes hold factors of both kinds (the tree's sparsity,
    solved in the path layout, and with contacts between robot bodies, solved dof by dof), and the same VJPs as pairs of
    cotangent sets. Against the oracle's at the record's a*: the float32 IFT solves with H (condition 1e4 to 1e6) leave
    about 1e-4 at one substep (median over the worlds; the suite's gate for one substep's gradients), and the position
    gradient what the contact normals' derivatives lose (_centres); sets bitwise the single calls."""
    import torch
    from nablaengine_amd import torch_ffi
    B = 12
    args, _, tape, recs, s64 = _taped(kind, B)
    cots = [synthetic.cotangents(B, seed=5 + i) for i in range(3)]
    cq, cv = (torch.from_numpy(np.stack(x)).cuda() for x in zip(*cots))
    sets = torch_ffi._vjp_sets(tape, args[4], args[5], cq, cv, substeps=1, clamp_kv=1, normal=0)
    for i in range(3):
        one = torch_ffi.backward(tape, args[4], args[5], cq[i].contiguous(), cv[i].contiguous(), substeps=1, clamp_kv=1,
                                 normal=0)
        for a, b in zip(one, sets):
            assert torch.equal(a, b[i])
    ref = oracle.vjp(**s64, g_qpos=cots[2][0].astype(np.float64), g_qvel=cots[2][1].astype(np.float64), clamp_kv=1,
                     normal=0, **{**oracle.ENGINE, "iterations": 0}, nsub=1)
    got = [x.cpu().numpy().astype(np.float64) for x in one[:3]]
    near = np.array([_centres({k: v[w] for k, v in s64.items()}, recs[w]) for w in range(B)])
    for name, a, b in zip(("qpos", "qvel", "ctrl"), got, ref):
        if name == "qpos":
            a, b = oracle.qpos_tangent(s64["qpos"], a), oracle.qpos_tangent(s64["qpos"], b)
        e = np.linalg.norm(a - b, axis=1) / np.maximum(np.linalg.norm(b, axis=1), 1e-12)
        tol = 1e-4 + (near if name == "qpos" else 0)
        print(kind, name, f"median {np.median(e):.2g} max {e.max():.2g}, of its bound {np.median(e / tol):.2g}")
        assert np.isfinite(a).all() and np.median(e / tol) <= 1, (name, e)


def _fma(a, b, c):  # float32 a b + c rounded once (a b is exact in the 64-bit mantissa)
    ld = np.longdouble
    return (a.astype(ld) * b.astype(ld) + c.astype(ld)).astype(np.float32)


def _solve(L, b):
    """x = A^-1 b, A = L' L, one dof at a time in float32 as csrc/g1_device.h's ltl_solve: L (B, 35, 35), b (B, 35)."""
    d = np.float32(1) / L[:, range(35), range(35)]
    z = b * d
    for i in range(34, 0, -1):
        z[:, :i] = _fma(-(L[:, i, :i] * d[:, :i]), z[:, i:i + 1], z[:, :i])
    z = z * d
    for k in range(34):
        z[:, k + 1:] = _fma(-(L[:, k + 1:, k] * d[:, k + 1:]), z[:, k:k + 1], z[:, k + 1:])
    return z


@pytest.mark.parametrize("kind,routes", [("flight", "both"), ("all", "dofs"), ("waist", "both"), ("legs_left", "both"),
                                         ("arm_right", "dofs"), ("one_foot", "both"), ("tangled", "both"),
                                         ("feet", "dofs")])
def test_solves_are_bitwise_the_dof_by_dof_ones(kind, routes):
    """With no position cotangent one substep's control gradient is kp lambda (0 where the actuator is at its limit),
    lambda = H^-1 (c - h kv y), y = Q^-1 c, c = h times the velocity cotangent. From the record's own factors, the
    replay of both solves dof by dof gives it to the last bit, whichever route the adjoint takes for L_H: the path layout
    (no contact between robot bodies in its zone) or dof by dof. Solving L_H on the tree's pattern alone would not."""
    import torch
    from nablaengine_amd import torch_ffi
    B = 12
    args, _, tape, rec, _ = _taped(kind, B)
    cv = synthetic.cotangents(B, seed=5)[1]
    gu = torch_ffi.backward(tape, args[4], args[5], torch.zeros((B, 36), device="cuda"), torch.from_numpy(cv).cuda(),
                            substeps=1, clamp_kv=1, normal=0)[2].cpu().numpy()
    LQ, LH = (np.stack([_unpack(r[k:]) for r in rec]).astype(np.float32) for k in (REC_LQ, REC_LH))
    h, kv, kp = np.float32(MODEL["timestep"]), *(np.asarray(MODEL[k], np.float32) for k in ("dof_kv", "dof_kp"))
    c = h * cv
    y = _solve(LQ * TREE, c)
    rhs = _fma(-(h * kv)[None], y, c)
    clamped = (rec.view(np.uint32)[:, REC_CLAMP, None].astype(np.uint64)
               | rec.view(np.uint32)[:, REC_CLAMP + 1, None].astype(np.uint64) << np.uint64(32))
    clamped = (clamped >> np.arange(6, 35).astype(np.uint64)) & np.uint64(1) != 0
    of = lambda lam: np.where(clamped, np.float32(0), kp[6:] * lam[:, 6:])
    assert np.array_equal(gu, of(_solve(LH, rhs)))
    off = _self_contacts(rec) > 0
    assert off.any() and (not off.all() if routes == "both" else off.all()), off
    if kind in ("tangled", "feet"):
        assert not np.array_equal(gu[off], of(_solve(LH * TREE, rhs))[off])
