"""The many-cotangent adjoint's workgroups (csrc/g1_adjoint.hip sets_per_group) on both sides of each line of the rule: single
sets that fit the resident waves at once and more, pairs in one round and more, even groups of 2, 4 and 6 with a last
shorter one, and launches of 2, 3 and 5 sets. Every set is bitwise its own backward() call."""
import ctypes

import numpy as np
import pytest

from nablaengine_amd import synthetic

pytestmark = pytest.mark.gpu
KEYS = ("qpos", "qvel", "warm", "ctrl", "friction", "com")


@pytest.mark.parametrize("B,K", [(28, 71), (29, 71), (57, 71), (87, 71), (230, 71), (231, 71), (600, 71), (1000, 71),
                                 (1, 2), (300, 3), (9000, 3), (4097, 5), (1100, 2), (1409, 2), (600, 4)])
def test_sets_are_the_backward_calls_at_each_group_size(B, K):
    import torch
    from nablaengine_amd import torch_ffi
    torch_ffi.init(0)
    st = synthetic.states(B, config=1, seed=B)
    args = [torch.from_numpy(np.ascontiguousarray(st[k], np.float32)).cuda() for k in KEYS]
    tape = torch_ffi.forward(*args, substeps=2, tape=True)[4]
    g = torch.Generator(device="cuda").manual_seed(K)
    cq = torch.randn((K, B, 36), device="cuda", generator=g)
    cv = torch.randn((K, B, 35), device="cuda", generator=g)
    sets = torch_ffi._vjp_sets(tape, args[4], args[5], cq, cv, substeps=2)
    for i in sorted({0, 1, K // 2, K - 2, K - 1}):
        one = torch_ffi.backward(tape, args[4], args[5], cq[i], cv[i], substeps=2)
        for a, b in zip(one, sets):
            assert torch.equal(a.view(torch.int32), b[i].view(torch.int32)), i


def test_single_sets_just_past_one_round():
    """The group sizes that the rule gives around one round R of resident waves (8 a CU): single sets while the waves past
    R are all of the last set and at most 3/8 R, then pairs until single sets take 3 rounds."""
    import torch
    from nablaengine_amd import torch_ffi
    torch_ffi.init(0)
    rule = ctypes.CDLL(torch_ffi.library_path())["_ZN3g1k14sets_per_groupEii"]
    R = 8 * torch.cuda.get_device_properties(0).multi_processor_count
    for ncot in (2, 3, 4, 6):
        last = min(R * 11 // 8 // ncot, R // (ncot - 1))  # the most worlds of either bound
        for nw in (R // ncot, R // ncot + 1, last - 1, last):
            assert rule(nw, ncot) == 1, (nw, ncot)
        assert rule(last + 1, ncot) == 2, (last + 1, ncot)
    assert rule(R // 71 + 1, 71) == 1 and rule(R // 71 + 4, 71) == 2
    assert rule(1, 2) == 1 and rule(2 * R, 2) == 2 and rule(8 * R, 2) == 2 and rule(8 * R, 71) == 36
