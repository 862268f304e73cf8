"""k_kin and k_kin_vjp take two worlds per wave: a world's outputs and gradients are the same bits alone, in either half
and in the last wave of an odd batch, whatever the other half holds (non-finite inputs included), and an odd batch's
empty half stores nothing."""
import ctypes

import numpy as np
import pytest

from nablaengine_amd import synthetic

pytestmark = pytest.mark.gpu
OUT = (36, 93, 124, 186, 93)


def _run(n, x, add):
    """The C entries on the first n worlds, into buffers of one more row: (outputs, gradients) with the spare row."""
    import torch
    from nablaengine_amd import torch_ffi
    lib = torch_ffi.load_library()
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    P = [ctypes.c_void_p(t.data_ptr()) for t in x[:3]]
    out = [torch.full((n + 1, k), 7.0, device="cuda") for k in OUT]
    grad = [torch.full((n + 1, k), 7.0, device="cuda") for k in (36, 35)]
    assert lib.dk_fwd_kinematics(st, n, *P, *(ctypes.c_void_p(t.data_ptr()) for t in out)) == 0
    inc = [ctypes.c_void_p(t.data_ptr()) for t in x[8:10]] if add else [None, None]
    cot = [ctypes.c_void_p(t.data_ptr()) for t in x[3:8]]
    assert lib.dk_fwd_kinematics_vjp(st, n, *P, *cot, *inc, *(ctypes.c_void_p(t.data_ptr()) for t in grad)) == 0
    return [t.cpu().numpy() for t in out + grad]


@pytest.mark.parametrize("add", [False, True])
@pytest.mark.parametrize("n", [1, 2, 3, 65])
def test_a_world_is_the_same_in_any_place(n, add):
    import torch
    from nablaengine_amd import torch_ffi
    torch_ffi.init(0)
    st = synthetic.states(n, config=4, seed=9)
    rng = np.random.default_rng(10)
    x = [torch.from_numpy(v).cuda() for v in (st["qpos"], st["qvel"], st["com"], *(
        rng.standard_normal((n, k), dtype=np.float32) for k in (*OUT, 36, 35)))]
    whole = _run(n, x, add)
    for r in whole:
        assert (r[n] == 7.0).all() and np.isfinite(r).all()
    # shifted by one world (the halves swapped) behind a world of NaNs; each world of a few alone
    shifted = [torch.cat([torch.full_like(t[:1], float("nan")), t]) for t in x]
    for a, b in zip(whole, _run(n + 1, shifted, add)):
        assert np.array_equal(a[:n].view(np.uint32), b[1:n + 1].view(np.uint32))
    for w in {0, n // 2, n - 1}:
        for a, b in zip(whole, _run(1, [t[w:w + 1].contiguous() for t in x], add)):
            assert np.array_equal(a[w].view(np.uint32), b[0].view(np.uint32))
