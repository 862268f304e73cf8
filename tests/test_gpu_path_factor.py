"""The factorizations and solves in the path layout (csrc/g1_path.h) at the places where it can go wrong: no
constraint rows at all; a limit row on every hinge (every diagonal entry), on the waist's three (shared by both arm
paths), on one leg's or one arm's; contacts on one limb; contacts between robot bodies, whose assembly goes through
the packed form, on and off one path, fewer and more than are assembled at once. One substep, from its tape record against float64 (the oracle)."""
import numpy as np
import pytest

import oracle
from nablaengine_amd import synthetic

pytestmark = pytest.mark.gpu
KEYS = ("qpos", "qvel", "warm", "ctrl", "friction", "com")
REC_FLAGS, REC_ASTAR, REC_AADV, REC_LH, REC_LQ = 1, 128, 164, 200, 832
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


@pytest.mark.parametrize("kind", ["flight", "all", "waist", "legs_left", "legs_right", "arm_left", "arm_right",
                                  "one_foot", "tangled", "feet"])
def test_path_factors_vs_oracle(kind):
    """L_Q against float64's factor of M + h kv, L_H' L_H against H at the final zones, and a_adv's residual in
    (M + h kv) a_adv = M a*. Tolerances: the elimination's backward error is at most about n eps = 35 x 6e-8 = 2e-6 of
    the largest entry, and M and H themselves are sums of some tens of float32 terms (a few 1e-7 each): 1e-5; the
    residual is that of the factor times |x| (1e-5 |Q| |a_adv|, rows against the largest)."""
    import torch
    from nablaengine_amd import torch_ffi
    B = 12
    st = _states(kind, B)
    args = [torch.from_numpy(st[k]).cuda() for k in KEYS]
    _, _, _, info, tape = torch_ffi.forward(*args, iterations=50, substeps=1, tape=True)
    tape, info = tape.cpu().numpy(), info.cpu().numpy()
    m = synthetic.model()
    hkv = m["timestep"] * np.diag(np.asarray(m["dof_kv"]))
    tree = np.array([[bool((m["body_ancmask"][m["dof_body"][i]] >> m["dof_body"][j]) & 1) for j in range(35)]
                     for i in range(35)])
    same = []
    for w in range(B):
        s = {k: st[k][w].astype(np.float64) for k in KEYS}
        M, H = oracle.substep_hessian(s["qpos"], s["qvel"], s["warm"], s["ctrl"], float(s["friction"]), s["com"])
        rec = tape[w]
        ref = oracle.ltl(M + hkv)
        assert np.abs(_unpack(rec[REC_LQ:]) * tree - ref).max() <= 1e-5 * np.abs(ref).max(), w
        a, adv = rec[REC_ASTAR:REC_ASTAR + 35].astype(np.float64), rec[REC_AADV:REC_AADV + 35].astype(np.float64)
        res = (M + hkv) @ adv - M @ a
        assert np.abs(res).max() <= 1e-5 * (np.abs(M + hkv) @ np.abs(adv)).max(), w
        if not rec[REC_FLAGS:REC_FLAGS + 1].view(np.uint32)[0] & (4 | 16 | (1 << 9)):
            L = _unpack(rec[REC_LH:])
            if np.abs(L.T @ L - H).max() <= 1e-5 * np.abs(H).max():
                same.append(w)
    # a world whose float32 and float64 solves end in different zones differs by a row's D J J'; with two feet's worth of
    # redundant contacts most do, so there it is enough that worlds past one chunk of edge rows are among the others
    print(kind, "H agrees in", same, "contacts", info[:, 1].tolist())
    assert len(same) >= (3 if kind == "feet" else B - 2), same
    if kind in HINGES:
        a, b = HINGES[kind]
        assert (info[:, 2] >= b - a).all(), info  # the limit rows are there
    if kind == "feet":
        assert info[same, 1].max() > 16 and (info[same, 1] % 4 != 0).any(), info
    if kind == "flight":
        assert (info[:, 2] == 0).sum() >= 4, info  # worlds without any row (a hand may touch the hip in the others)


@pytest.mark.parametrize("kind", ["flight", "all", "waist", "one_foot", "tangled", "feet"])
def test_path_solves_in_the_adjoint(kind):
    """One substep's VJP (exact mode) on the same states, whose tapes hold factors of both kinds (the tree's sparsity,
    solved in the path layout, and with contacts between robot bodies, solved dof by dof), and the same VJPs as pairs of
    cotangent sets. Against the oracle's: the float32 IFT solves with H (condition 1e5 to 1e6) leave about 1e-4 at one
    substep (median over the worlds; the suite's gate for one substep's gradients); sets bitwise the single calls."""
    import torch
    from nablaengine_amd import torch_ffi
    B = 12
    st = _states(kind, B)
    args = [torch.from_numpy(st[k]).cuda() for k in KEYS]
    tape = torch_ffi.forward(*args, iterations=50, substeps=1, tape=True)[4]
    cots = [synthetic.cotangents(B, seed=5 + i) for i in range(3)]
    cq, cv = (torch.from_numpy(np.stack(x)).cuda() for x in zip(*cots))
    sets = torch_ffi._vjp_sets(tape, args[4], args[5], cq, cv, substeps=1, clamp_kv=1, normal=0)
    for i in range(3):
        one = torch_ffi.backward(tape, args[4], args[5], cq[i].contiguous(), cv[i].contiguous(), substeps=1, clamp_kv=1,
                                 normal=0)
        for a, b in zip(one, sets):
            assert torch.equal(a, b[i])
    s64 = {k: st[k].astype(np.float64) for k in KEYS}
    ref = oracle.vjp(**s64, g_qpos=cots[2][0].astype(np.float64), g_qvel=cots[2][1].astype(np.float64), clamp_kv=1,
                     normal=0, **{**oracle.ENGINE, "iterations": 50}, nsub=1)
    got = [x.cpu().numpy().astype(np.float64) for x in one[:3]]
    for name, a, b in zip(("qpos", "qvel", "ctrl"), got, ref):
        if name == "qpos":
            a, b = oracle.qpos_tangent(s64["qpos"], a), oracle.qpos_tangent(s64["qpos"], b)
        e = np.linalg.norm(a - b, axis=1) / np.maximum(np.linalg.norm(b, axis=1), 1e-12)
        print(kind, name, f"median {np.median(e):.2g} max {e.max():.2g}")
        assert np.isfinite(a).all() and (kind == "feet" or np.median(e) <= 1e-4), (name, e)
