"""Deposition onto a small mesh of a set whose particle words pass 2^31 (3 words a
particle): the ones past it, in the mesh, among others that lie far outside,
against a set of these alone, bit for bit."""
import pytest

pytestmark = pytest.mark.gpu


def test_particle_words_beyond_int32():
    import torch
    import pmlib3d_amd as pm
    from pmlib3d_amd import _lib
    few, many = 4096, (1 << 31) // 3 + 5000   # the last ones' words start beyond 2^31
    if torch.cuda.mem_get_info()[0] < 130e9:   # positions 17 GB, keys, ids and records 55 GB
        pytest.skip("not enough free memory on this GPU")
    n, h = 16, 2.0 / 16
    patch = pm.Patch(xmin=(-1.0,) * 3, xmax=(1.0,) * 3, ncell=(n,) * 3, dx=(h,) * 3)
    ops = pm.ParticleOps(patch, interp_order=3, precision=pm.FP32)
    gen = torch.Generator(device="cuda:0").manual_seed(1)
    inside = 1.8 * torch.rand(3 * few, dtype=torch.float64, device="cuda:0", generator=gen) - 0.9
    mesh = [torch.zeros(3 * n ** 3, dtype=torch.float32, device="cuda:0") for _ in range(2)]
    # (the positions serve as strengths too)
    ops.p2m(inside.data_ptr(), inside.data_ptr(), few, mesh[0].data_ptr())
    every = torch.full((3 * many,), 1e3, dtype=torch.float64, device="cuda:0")
    every[-3 * few:] = inside
    ops.p2m(every.data_ptr(), every.data_ptr(), many, mesh[1].data_ptr())
    torch.cuda.synchronize()
    same = bool(torch.equal(mesh[0], mesh[1])) and bool(mesh[0].abs().max() > 0)
    del every
    torch.cuda.empty_cache()
    _lib.check(_lib.load().pmgpu_finalize(), "pmgpu_finalize")   # the workspace of this call
    assert same
