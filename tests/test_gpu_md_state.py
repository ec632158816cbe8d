"""The one-launch state moves of an MD run (pt_md_start, pt_copy_arrays, pt_scatter_rows3_f64)
against torch indexing, at the ends of their workgroups and at sizes and addresses that do
not allow 16-byte words.  Copies and one division: exactly equal."""

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n", [1, 2, 255, 257, 1023, 5001])
def test_state_moves_equal_indexing(n):
    from pantea_amd import _lib
    from pantea_amd.engine import clone_all

    lib = _lib.load()
    st = _lib.stream_ptr()
    g = torch.Generator().manual_seed(n)
    perm = torch.randperm(n, generator=g).to(torch.int32).cuda()
    vel = torch.randn(n, 3, generator=g, dtype=torch.float64).cuda()
    mass = (torch.rand(n, generator=g, dtype=torch.float64) + 0.5).cuda()
    types = torch.randint(1, 4, (n,), generator=g, dtype=torch.int32).cuda()
    out = [torch.empty_like(vel), torch.empty_like(mass), torch.empty_like(mass), torch.empty_like(perm),
           torch.empty_like(types)]
    _lib.check(lib.pt_md_start(n, perm.data_ptr(), vel.data_ptr(), mass.data_ptr(), types.data_ptr(),
                               _lib.MDState(*(t.data_ptr() for t in out)), st), "start")
    i = perm.long()
    for a, b in zip(out, (vel[i], mass[i], 1.0 / mass[i], perm, types[i])):
        assert torch.equal(a, b)

    # the last one starts 4 bytes past a 16-byte address
    odd = torch.arange(n + 1, dtype=torch.int32, device="cuda")[1:]
    arrays = [vel, mass, types, odd]
    for a, b in zip(arrays, clone_all(arrays)):
        assert torch.equal(a, b)

    pos4 = torch.randn(n, 4, generator=g, dtype=torch.float64).cuda()
    got = torch.full((n, 3), float("nan"), dtype=torch.float64, device="cuda")
    _lib.check(lib.pt_scatter_rows3_f64(n, perm.data_ptr(), pos4.data_ptr(), 4, got.data_ptr(), st), "scatter")
    want = torch.empty_like(got)
    want[i] = pos4[:, :3]
    assert torch.equal(got, want)

    inv = torch.full_like(perm, -1)
    _lib.check(lib.pt_invert_perm(n, perm.data_ptr(), inv.data_ptr(), st), "invert")
    assert torch.equal(inv[i], torch.arange(n, dtype=torch.int32, device="cuda"))
