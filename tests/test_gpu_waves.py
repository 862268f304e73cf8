"""The forward's two builds (two waves per SIMD up to 9 worlds a CU, three beyond): the same bits on both sides of the
line, in every output and in the tape, for standing and contact-heavy worlds (contacts between robot bodies included)."""
import numpy as np
import pytest

from nablaengine_amd import synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("config", [1, 4])
def test_both_builds_give_the_same_bits(config):
    import torch
    from nablaengine_amd import torch_ffi
    n = 9 * torch.cuda.get_device_properties(0).multi_processor_count
    st = synthetic.states(n + 1, config=config, seed=31)
    args = [torch.from_numpy(st[k]).cuda() for k in ("qpos", "qvel", "warm", "ctrl", "friction", "com")]
    three = torch_ffi.forward(*args, tape=True)
    two = torch_ffi.forward(*(x[:n] for x in args), tape=True)
    last = torch_ffi.forward(*(x[n:] for x in args), tape=True)
    for a, b, c in zip(three, two, last):
        assert np.array_equal(a[:n].cpu().numpy().view(np.uint8), b.cpu().numpy().view(np.uint8))
        assert np.array_equal(a[n:].cpu().numpy().view(np.uint8), c.cpu().numpy().view(np.uint8))
