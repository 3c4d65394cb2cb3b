"""Two calls of one process whose times stand in a known relation, timed in
turn; each bound lies between what the call takes and what the fault it
guards against would make of it, well past the few per cent that timings of
one kernel differ by."""
import pytest

pytestmark = pytest.mark.gpu


def _us(f, reps):
    import torch

    best = float("inf")
    for _ in range(5):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        f()
        a.record()
        for _ in range(reps):
            f()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) / reps * 1e3)
    return best


@pytest.mark.parametrize("n,whole,cin,cout,norm", [
    (81500, 81920, 256, 128, False),    # 255 full 320-row tiles and a partial one
    (32500, 32768, 512, 128, True),     # the conv of the norm row pass, 256 64-column tiles
    (129761, 131072, 256, 128, False),  # two rounds of 256-row tiles
    (32500, 32768, 256, 256, False)])   # two column tiles a row tile
def test_partial_tile_takes_no_round_of_its_own(spc, dev, n, whole, cin, cout, norm):
    """As many tiles as compute units are one round of them, also when the last
    row tile is partial (a round for the one tile added a quarter to a half)."""
    import numpy as np
    import torch

    nat = spc._native
    c = np.concatenate([spc.workloads.ellipsoid_batch(4, seed=s) + [4 * s, 0, 0, 0]
                        for s in range(3)]).astype(np.int32)
    print(f"[case] partial last tile {n} / {whole} rows {cin}->{cout} norm={norm}", flush=True)
    assert c.shape[0] >= whole
    g = torch.Generator(device="cuda").manual_seed(1)
    w = (torch.randn((cout, 27, cin), generator=g, device=dev) * (27 * cin) ** -0.5).bfloat16()
    b = torch.randn(cout, generator=g, device=dev).bfloat16()
    pw, mod, us = nat.pack_weights(w), torch.zeros((12, cout), device=dev), []
    for rows in (n, whole):  # (the mapping's outputs against another geometry's, too)
        coords = torch.from_numpy(np.ascontiguousarray(c[:rows])).to(dev)
        m = nat.map_build(coords, outputs="token")
        p = nat.conv_plan(m.token_major, ntaps=27, n_out=rows)
        x = torch.randn((rows, cin), generator=g, device=dev).bfloat16()
        run = lambda nm=None: nat.sparse_conv(x, pw, b, m.token_major, ntaps=27,  # noqa: E731
                                              n_out=rows, plan=p, norm_mod=nm)
        y = run()
        nat.set_tile_geometry(nat.TILES_SMALL)
        try:
            assert torch.equal(y, run())
        finally:
            nat.set_tile_geometry(nat.TILES_AUTO)
        us.append(_us(lambda: run((mod, mod, coords, 1e-6) if norm else None), 30))
    print(f"[time] {us[0]:.1f} / {us[1]:.1f} us", flush=True)
    assert us[0] <= 1.2 * us[1], us


def test_plan_of_scattered_rows(spc, dev):
    """Tiles past the stage give up early in the setup's hash: the small tiles'
    plan of shuffled rows (every tile past it) takes no longer than of rows in
    order (0.86 times; 1.37 when the hash collected 1,472 rows a tile)."""
    import torch

    nat, n = spc._native, 400000
    par = torch.from_numpy(spc.workloads.ellipsoid_batch(4, seed=1)).to(dev)
    kids = nat.subdivide_map(par)[0][:n]
    assert kids.shape[0] == n
    print(f"[case] plan of {n} rows in order and shuffled", flush=True)
    us = []
    for c in (kids, kids[torch.randperm(n, generator=torch.Generator().manual_seed(1)).to(dev)]):
        m = nat.map_build(c.contiguous(), outputs="token")
        us.append(_us(lambda: nat.conv_plan(m.token_major, ntaps=27, n_out=n,
                                            sections=nat.PLAN_SMALL), 20))
    print(f"[time] {us[0]:.1f} / {us[1]:.1f} us", flush=True)
    assert us[1] <= 1.1 * us[0], us
