"""pt_md_positions, pt_md_velocities and pt_md_berendsen against the separate calls they
replace (pt_verlet_*, pt_skin_check, pt_permute_state_gated, pt_kinetic_energy,
pt_berendsen_rescale) where their workgroups end: 256 atoms per workgroup of positions and
rescale, 1,024 of velocities, more than 256 workgroups.  The contract is equality bit for bit."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("mass", [True, False])
@pytest.mark.parametrize("n", [1, 3, 255, 257, 1023, 1024, 1025, 70001])
def test_fused_step_equals_separate_calls(n, mass):
    from pantea_amd import _lib

    lib = _lib.load()
    st = _lib.stream_ptr()
    g = torch.Generator().manual_seed(n)
    dev = "cuda"
    L = np.array([20.0, 21.0, 22.0])
    box = (ctypes.c_double * 3)(*L)
    box_p = ctypes.cast(box, ctypes.c_void_p)

    def rnd(*shape):
        return torch.randn(*shape, generator=g, dtype=torch.float64).to(dev)

    pos = torch.rand(n, 4, generator=g, dtype=torch.float64).to(dev) * 20.0
    ref = pos + 0.05 * rnd(n, 4)
    vel, f_old, f_new = rnd(n, 3), rnd(n, 3), rnd(n, 3)
    m = (torch.rand(n, generator=g, dtype=torch.float64) + 0.5).to(dev)
    im = 1.0 / m
    perm = torch.randperm(n, generator=g).to(torch.int32).to(dev)
    ids = torch.arange(n, dtype=torch.int32, device=dev)
    types = (ids % 3 + 1).contiguous()
    imp = im.data_ptr() if mass else None
    dt, tau, t0, kb = 0.3, 2.0, 1.5, 0.7
    scratch = torch.empty(514, dtype=torch.float64, device=dev)

    for skin in (0.2, 100.0, None):
        # separate calls
        p1, ref1 = pos.clone(), ref.clone()
        flag1 = torch.full((1,), 1, dtype=torch.int32, device=dev)
        _lib.check(lib.pt_verlet_positions(n, p1.data_ptr(), vel.data_ptr(), f_old.data_ptr(), imp, dt, box_p, st), "x")
        if skin is not None:
            _lib.check(lib.pt_skin_check(n, p1.data_ptr(), ref1.data_ptr(), box_p, skin, scratch.data_ptr(),
                                         flag1.data_ptr(), st), "skin")
        s1 = [vel.clone(), f_old.clone(), m.clone(), im.clone(), ids.clone(), types.clone()]
        arrays = (_lib.PermuteArray * 6)(*[_lib.PermuteArray(b.data_ptr(), w, wb) for b, w, wb in zip(
            s1, (3, 3, 1, 1, 1, 1), (8, 8, 8, 8, 4, 4))])
        tmp = torch.empty(72 * n, dtype=torch.uint8, device=dev)
        _lib.check(lib.pt_permute_state_gated(n, perm.data_ptr(), 6, arrays, tmp.data_ptr(), tmp.numel(),
                                              flag1.data_ptr(), st), "permute")
        if int(flag1.item()):
            ref1.copy_(p1)
        _lib.check(lib.pt_verlet_velocities(n, s1[0].data_ptr(), s1[1].data_ptr(), f_new.data_ptr(),
                                            s1[3].data_ptr() if mass else None, dt, st), "v")
        ws = torch.empty(lib.pt_reduce_workspace_bytes(n), dtype=torch.uint8, device=dev)
        ke = torch.zeros(1, dtype=torch.float64, device=dev)
        _lib.check(lib.pt_kinetic_energy(n, s1[0].data_ptr(), s1[2].data_ptr(), ke.data_ptr(), ws.data_ptr(),
                                         ws.numel(), st), "ke")
        _lib.check(lib.pt_berendsen_rescale(n, s1[0].data_ptr(), ke.data_ptr(), dt, tau, t0, kb, st), "b")

        # fused
        p2, ref2, pin = pos.clone(), ref.clone(), torch.full_like(pos, float("nan"))
        flag2 = torch.full((1,), 1, dtype=torch.int32, device=dev)
        _lib.check(lib.pt_md_positions(n, p2.data_ptr(), vel.data_ptr(), f_old.data_ptr(), imp, dt, box_p,
                                       pin.data_ptr(), ref2.data_ptr() if skin is not None else None, skin or 0.0,
                                       scratch.data_ptr(), flag2.data_ptr(), st), "md x")
        old = [vel.clone(), m.clone(), im.clone(), ids.clone(), types.clone()]
        new = [torch.empty_like(t) for t in old]
        part = torch.empty(lib.pt_reduce_workspace_bytes(n) // 8, dtype=torch.float64, device=dev)
        _lib.check(lib.pt_md_velocities(n, flag2.data_ptr(), perm.data_ptr(), _lib.MDState(*(t.data_ptr() for t in old)),
                                        _lib.MDState(*(t.data_ptr() for t in new)), f_old.data_ptr(), f_new.data_ptr(),
                                        int(mass), dt, p2.data_ptr(), ref2.data_ptr() if skin is not None else None,
                                        part.data_ptr(), st), "md v")
        _lib.check(lib.pt_md_berendsen(n, new[0].data_ptr(), part.data_ptr(), dt, tau, t0, kb, st), "md b")
        assert int(flag1.item()) == int(flag2.item())
        assert torch.equal(p1, p2) and torch.equal(p2, pin)
        for a, b in zip([s1[0], s1[2], s1[3], s1[4], s1[5]], new):
            assert torch.equal(a, b)
        if skin is not None:
            assert torch.equal(ref1, ref2)
