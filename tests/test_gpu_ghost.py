"""Ghost-layer flows on the GPU against the oracle's restatement of the
reference's scripts, bit for bit, and against the analytic profiles."""

import numpy as np
import pytest
import torch

from oracle import ghost_ref as g

pytestmark = pytest.mark.gpu

DT = [(torch.float64, np.float64), (torch.float32, np.float32)]


def same(lat, mom, G, omom):
    assert np.array_equal(lat.populations(), G)
    for a, b in zip(mom, omom):
        assert np.array_equal(a.cpu().numpy(), b)


@pytest.mark.parametrize("tdt,ndt", DT)
@pytest.mark.parametrize("steps", [1, 2, 37])
@pytest.mark.parametrize("layout", ["rows", "soa"])
def test_couette_matches_oracle(gpu, tdt, ndt, steps, layout):
    from latticeboltzmann_amd import ghost
    print("couette", tdt, steps, layout, flush=True)
    lat, mom = ghost.couette(20, 12, 0.1, 1.3, steps, dtype=tdt, layout=layout)
    G, omom = g.couette(20, 12, 0.1, 1.3, steps, dtype=ndt)
    same(lat, mom, G, omom)


@pytest.mark.parametrize("tdt,ndt", DT)
@pytest.mark.parametrize("steps", [1, 37])
def test_poiseuille_matches_oracle(gpu, tdt, ndt, steps):
    from latticeboltzmann_amd import ghost
    print("poiseuille", tdt, steps, flush=True)
    lat, mom = ghost.poiseuille(22, 12, 1.001, 0.999, 0.7, steps, uw=0.02, dtype=tdt)
    G, omom = g.poiseuille(22, 12, 1.001, 0.999, 0.7, steps, uw=0.02, dtype=ndt)
    same(lat, mom, G, omom)


@pytest.mark.parametrize("tdt,ndt", DT)
@pytest.mark.parametrize("layout", ["rows", "soa"])
def test_sliding_lid_matches_oracle(gpu, tdt, ndt, layout):
    from latticeboltzmann_amd import ghost
    print("sliding lid", tdt, layout, flush=True)
    lat, mom = ghost.sliding_lid(16, steps=37, uw=0.1, omega=1.7, dtype=tdt, layout=layout)
    G, omom = g.sliding_lid(18, 18, 0.1, 1.7, 37, dtype=ndt)
    same(lat, mom, G, omom)


@pytest.mark.parametrize("tdt,ndt", DT)
@pytest.mark.parametrize("layout", ["rows", "soa"])
def test_obstacle_canal_matches_oracle(gpu, tdt, ndt, layout):
    from latticeboltzmann_amd import ghost
    print("obstacle canal", tdt, layout, flush=True)
    ob = (12, 8, 15, 11)
    lat, mom = ghost.obstacle_canal(30, 20, ob, rho_diff=0.01, omega=0.8, steps=37, dtype=tdt,
                                    layout=layout)
    G, omom = g.obstacle_canal(32, 22, 1 + 0.01, 1 - 0.01, 0.8, 37, ob, dtype=ndt)
    same(lat, mom, G, omom)


@pytest.mark.parametrize("vertical", [True, False])
def test_pulse_kats(gpu, vertical):
    from latticeboltzmann_amd import ghost
    f = np.zeros((9, 9, 9))
    if vertical:
        f[1, 1, 1:8] = 1
    else:
        f[2, 1:8, 1] = 1
    lat = ghost.GhostLattice(9, 9, 1.0, ghost.pulse_walls(9, 9, vertical)).load(f)
    for _ in range(14):
        lat.stream_and_walls()
    got = lat.populations()
    assert np.array_equal(got, g.pulse_walls(f.copy(), 14, vertical))
    assert np.all((got[1, 1, 1:7] if vertical else got[2, 1:7, 1]) == 1)


def test_obstacle_pulses(gpu):
    from latticeboltzmann_amd import ghost
    rng = np.random.default_rng(3)
    f = rng.random((9, 16, 16))
    lat = ghost.GhostLattice(16, 16, 1.0, ghost.obstacle_faces(6, 6, 9, 9)).load(f)
    h = f.copy()
    for _ in range(9):
        lat.stream_and_walls()
        g.stream(h)
        g.apply_obstacle(h, 6, 6, 9, 9)
    assert np.array_equal(lat.populations(), h)


def test_collide_only_and_equilibrium(gpu):
    from latticeboltzmann_amd import ghost
    rng = np.random.default_rng(4)
    rho = 1 + 0.1 * rng.standard_normal((7, 5))
    ux, uy = 0.1 * rng.standard_normal((7, 5)), 0.1 * rng.standard_normal((7, 5))
    lat = ghost.GhostLattice(7, 5, 0.9).init_equilibrium(rho, ux, uy)
    assert np.array_equal(lat.populations(), g.equilibrium(rho, ux, uy))
    f = g.equilibrium(rho, ux, uy) * (1 + 0.05 * rng.standard_normal((9, 7, 5)))
    lat.load(f)
    mom = lat.moment_buffers()
    lat.collide_only(mom)
    h = f.copy()
    om = g.collide(h, 0.9)
    same(lat, mom, h, om)


def test_rule_table_rejections(gpu):
    from latticeboltzmann_amd import ghost, _native as nat
    R = ghost.Rule
    bad = [
        [R(1, 5, 1, 2, 2, 4, 0, -1), R(1, 5, 2, 3, 2, 2, 0, -1)],  # reads what rule 0 wrote
        [R(0, 5, 0, 1, 2, 4, 0, -1)],                              # source outside the grid
        [R(1, 9, 1, 2, 2, 4, 0, -1)],                              # target outside the grid
        [R(1, 5, 1, 2, 9, 4, 0, -1)],                              # channel 9
        [R(1, 5, 8, 9, 7, 5, 0, -1, nat.RULE_LID_RHO, 0.1), R(1, 5, 7, 8, 0, 0, 0, 0)][::-1],
    ]
    for rules in bad:
        lat = ghost.GhostLattice(8, 10, 1.0, rules)
        with pytest.raises(ValueError):
            lat.step()
    with pytest.raises(ValueError):
        ghost.GhostLattice(8, 10, 1.0, [R(1, 2, 1, 2, 0)] * 33)


def test_couette_analytic(gpu):
    from latticeboltzmann_amd import ghost
    lat, (rho, ux, uy) = ghost.couette(100, 52, 0.1, 0.5, 20000)
    prof = ux.cpu().numpy()[50, 1:-1]
    assert np.abs(prof - ghost.couette_profile(50, 0.1)).max() < 3e-4


def test_poiseuille_analytic(gpu):
    from latticeboltzmann_amd import ghost
    lat, (rho, ux, uy) = ghost.poiseuille(102, 52, 1.001, 0.999, 0.5, 15000)
    ana = ghost.poiseuille_profile(100, 50, 0.001, 0.5)
    prof = ux.cpu().numpy()[51, 1:-1]
    assert np.abs(prof - ana).max() / ana.max() < 0.01


def test_sliding_lid_reference_config(gpu):
    # slidingLid.py:20-28: 300 + 2 nodes, Re 1000, lid 0.1, 10000 steps
    from latticeboltzmann_amd import ghost
    lat, (rho, ux, uy) = ghost.sliding_lid()
    u = ux.cpu().numpy()
    assert np.isfinite(lat.populations()).all()
    assert u[151, -2] > 0.05 and u[151, 20:150].min() < 0  # lid-driven primary vortex


@pytest.mark.parametrize("tdt,ndt", DT)
@pytest.mark.parametrize("nx,ny,steps", [(24, 24, 9), (45, 67, 7), (45, 67, 6), (361, 1067, 5),
                                         (352, 1058, 7)])
@pytest.mark.parametrize("flow", ["lid", "couette", "poiseuille", "canal", "sides", "far"])
def test_several_steps_per_launch_match_oracle(gpu, flow, tdt, ndt, nx, ny, steps):
    # small-grid tiles and the two large-grid tiles, every remainder of the
    # four steps a launch takes, wall tiles that are whole, cut, or one node
    # wide; "far" has a rule that reads across many columns (single steps)
    from latticeboltzmann_amd import ghost
    print("multi", flow, tdt, nx, ny, steps, flush=True)
    mx, my = nx // 2, ny // 2
    ob = (mx, my - 2, mx + 3, my + 1)
    rules, pbc, before, after = [], None, None, None
    if flow == "lid":
        rules = ghost.cavity_walls(nx, ny, 0.1)
        after = lambda G: g.bounce_back_cavity(G, 0.1)
    elif flow == "couette":
        rules = ghost.channel_walls(nx, ny, 0.1)
        after = lambda G: g.bounce_back_channel(G, 0.1)
    elif flow == "poiseuille":
        rules, pbc = ghost.channel_walls(nx, ny, 0.02), ("before", 1.01, 0.99)
        before = lambda G: g.pressure_periodic(G, 1.01, 0.99)
        after = lambda G: g.bounce_back_channel(G, 0.02)
    elif flow == "canal":
        rules = ghost.side_walls(nx, ny, 0.05) + ghost.obstacle_faces(*ob)
        pbc = ("after", 1.01, 0.99)

        def after(G):
            g.pressure_periodic_after(G, 1.01, 0.99)
            g.bounce_back_walls(G, 0.05)
            g.apply_obstacle(G, *ob)
    elif flow == "sides":
        rules = ghost.side_walls(nx, ny, left=True, right=True, bottom=False, top=False)
        after = lambda G: g.bounce_back_walls(G, 0.0, left=True, right=True, bottom=False, top=False)
    else:
        rules = [ghost.Rule(3, 5, 2, 9, 1, 3, nx - 6, 4)]

        def after(G):
            G[1, 3:5, 2:9] = G[3, nx - 3:nx - 1, 6:13]
    r = np.random.default_rng(nx + steps)
    rho = (1 + 0.02 * r.standard_normal((nx, ny))).astype(ndt)
    ux, uy = ((0.03 * r.standard_normal((nx, ny))).astype(ndt) for _ in range(2))
    lat = ghost.GhostLattice(nx, ny, 1.3, rules, pbc, dtype=tdt,
                             layout="soa" if steps == 6 else "rows")
    lat.init_equilibrium(rho, ux, uy)
    mom = lat.moment_buffers()
    lat.step(steps, moments=mom)
    G = g.equilibrium(rho, ux, uy)
    for _ in range(steps):
        if before:
            before(G)
        g.stream(G)
        after(G)
        omom = g.collide(G, 1.3)
    same(lat, mom, G, omom)


@pytest.mark.parametrize("flow,nx,ny", [("lid", 45, 67), ("canal", 102, 52), ("poiseuille", 700, 500)])
@pytest.mark.parametrize("steps", [1, 2, 4, 5, 10, 12, 20, 100])
def test_step_ends_in_the_buffer_of_single_steps(gpu, flow, nx, ny, steps):
    # n steps leave the state where n single-step launches would, so graphs of an
    # even number of steps (StepGraph's, or captured by a program) can be replayed
    from latticeboltzmann_amd import ghost
    from latticeboltzmann_amd.lattice import StepGraph
    rules = {"lid": lambda: ghost.cavity_walls(nx, ny, 0.1), "poiseuille": lambda: ghost.channel_walls(nx, ny, 0.02),
             "canal": lambda: ghost.side_walls(nx, ny) + ghost.obstacle_faces(50, 24, 53, 27)}[flow]()
    pbc = {"lid": None, "canal": ("after", 1.01, 0.99), "poiseuille": ("before", 1.01, 0.99)}[flow]
    lat, ref = (ghost.GhostLattice(nx, ny, 1.3, rules, pbc) for _ in range(2))
    print("buffers", flow, nx, ny, steps, flush=True)

    def eager(n):
        for _ in range(n):
            ref.step(1)

    a, b = lat.f, lat._g
    lat.step(steps)
    eager(steps)
    assert lat.f.data_ptr() == (b if steps % 2 else a).data_ptr()
    assert torch.equal(lat.f, ref.f)
    with StepGraph(lat, steps) as advance:
        for odd in (0, 1, 0, 3):  # replays, with eager work that moves the state in between
            advance()
            lat.step(odd)
            eager(steps + odd)
            assert torch.equal(lat.f, ref.f) and lat.time == ref.time


@pytest.mark.parametrize("tdt,ndt", DT)
@pytest.mark.parametrize("nx,ny,steps", [(45, 67, 8), (45, 67, 10), (361, 1067, 8), (352, 1058, 10)])
@pytest.mark.parametrize("flow", ["lid", "poiseuille", "canal"])
def test_launch_splits_match_oracle(gpu, flow, tdt, ndt, nx, ny, steps):
    # launches of 4 + 4, 3 + 3 + 2 + 2 (small tiles) and 4 + 4 + 1 + 1 steps
    test_several_steps_per_launch_match_oracle(gpu, flow, tdt, ndt, nx, ny, steps)


@pytest.mark.parametrize("tdt,ndt", DT)
@pytest.mark.parametrize("flow", ["walls", "before", "after"])
@pytest.mark.parametrize("where", ["smallest", "small", "largest", "mixed"])
def test_densities_at_the_ends_of_the_type(gpu, tdt, ndt, flow, where):
    # 2 rho / 9 and rho / 36 where they round as subnormals or overflow, as in ghost
    # nodes that cleared walls have drained for thousands of steps, beside others
    from latticeboltzmann_amd import ghost
    nx, ny, info = 45, 67, np.finfo(ndt)
    lo, hi = np.log2(float(info.smallest_subnormal)), np.log2(float(info.max))
    a, b = {"smallest": (lo, lo + 6), "small": (lo, lo + 70), "largest": (hi - 3, hi - 0.1), "mixed": (lo, 1)}[where]
    r = np.random.default_rng(len(where))
    rho = (2.0 ** r.uniform(a, b, (nx, ny))).astype(ndt)
    ux, uy = ((0.03 * r.standard_normal((nx, ny))).astype(ndt) for _ in range(2))
    rules, pbc, before, after = [], None, None, lambda G: None
    if flow == "before":
        pbc, before = ("before", 1.01, 0.99), lambda G: g.pressure_periodic(G, 1.01, 0.99)
    elif flow == "after":
        pbc, after = ("after", 1.01, 0.99), lambda G: g.pressure_periodic_after(G, 1.01, 0.99)
    else:
        rules, after = ghost.side_walls(nx, ny, 0.05), lambda G: g.bounce_back_walls(G, 0.05)
    with np.errstate(all="ignore"):
        start = g.equilibrium(rho, ux, uy)
        for steps in (1, 4, 7):
            print("ends", tdt, flow, where, steps, flush=True)
            lat = ghost.GhostLattice(nx, ny, 1.3, rules, pbc, dtype=tdt).load(start)
            mom = lat.moment_buffers()
            lat.step(steps, moments=mom)
            G = start.copy()
            for _ in range(steps):
                if before:
                    before(G)
                g.stream(G)
                after(G)
                omom = g.collide(G, 1.3)
            assert np.array_equal(lat.populations(), G, equal_nan=True)
            for x, y in zip(mom, omom):
                assert np.array_equal(x.cpu().numpy(), y, equal_nan=True)


def test_drained_ghost_nodes_match_oracle(gpu):
    # clearing walls: after 6000 steps the cleared nodes' densities are subnormal
    from latticeboltzmann_amd import ghost
    nx, ny, steps = 24, 20, 6000
    r = np.random.default_rng(0)
    start = g.at_rest(nx, ny) + 1e-3 * r.standard_normal((9, nx, ny))
    lat = ghost.GhostLattice(nx, ny, 0.5, ghost.pulse_walls(nx, ny, True)).load(start)
    lat.step(steps)
    G, m = start.copy(), nx - 1
    with np.errstate(all="ignore"):
        for _ in range(steps):
            g.stream(G)
            for ch, src in ((1, 3), (5, 7), (8, 6)):
                G[ch, 1] = G[src, 0]
            G[[3, 7, 6], 0] = 0
            for ch, src in ((3, 1), (6, 8), (7, 5)):
                G[ch, m - 1] = G[src, m]
            G[[1, 8, 5], m] = 0
            g.collide(G, 0.5)
    rho = np.abs(G.sum(0))
    assert rho[rho > 0].min() < np.finfo(np.float64).tiny
    assert np.array_equal(lat.populations(), G, equal_nan=True)


@pytest.mark.parametrize("tdt,ndt", DT)
@pytest.mark.parametrize("layout", ["rows", "soa"])
@pytest.mark.parametrize("mode", ["before", "after"])
@pytest.mark.parametrize("nx", [3, 4, 5, 9, 40])
def test_single_steps_near_inlet_and_outlet(gpu, tdt, ndt, layout, mode, nx):
    # grids of nothing but columns near the inlet and outlet, and rules whose
    # sources lie up to the whole grid away
    from latticeboltzmann_amd import ghost
    ny, far = 600, nx - 1
    rules = [ghost.Rule(0, 1, 2, 590, 1, 3, far, 4), ghost.Rule(far, nx, 3, 599, 6, 8, -far, -2)]
    args = (1.01, 0.99)
    r = np.random.default_rng(nx)
    rho = (1 + 0.02 * r.standard_normal((nx, ny))).astype(ndt)
    ux, uy = ((0.03 * r.standard_normal((nx, ny))).astype(ndt) for _ in range(2))
    lat = ghost.GhostLattice(nx, ny, 1.3, rules, (mode,) + args, dtype=tdt, layout=layout)
    lat.init_equilibrium(rho, ux, uy)
    mom = lat.moment_buffers()
    G = g.equilibrium(rho, ux, uy)
    for _ in range(3):
        print("near", tdt, layout, mode, nx, flush=True)
        lat.step(1, moments=mom)
        if mode == "before":
            g.pressure_periodic(G, *args)
        g.stream(G)
        if mode == "after":
            g.pressure_periodic_after(G, *args)
        a = G[3, far, 6:594].copy()
        b = G[8, 0, 1:597].copy()
        G[1, 0, 2:590], G[6, far, 3:599] = a, b
        omom = g.collide(G, 1.3)
        same(lat, mom, G, omom)


@pytest.mark.parametrize("tdt,ndt", DT)
@pytest.mark.parametrize("mode", ["before", "after"])
@pytest.mark.parametrize("nx,ny,steps", [(45, 67, 8), (45, 67, 7), (45, 67, 10), (120, 130, 8), (361, 1067, 8)])
def test_wall_density_rules_with_inlet_and_outlet(gpu, tdt, ndt, mode, nx, ny, steps):
    # the lid weighted by the wall's density where an inlet and outlet are, over all
    # columns, from the inlet and outlet columns and from one beside them, and from
    # two columns away; several steps a launch against the oracle
    from latticeboltzmann_amd import _native as nat
    from latticeboltzmann_amd import ghost
    k = nat.RULE_LID_RHO
    rules = [ghost.Rule(0, nx, ny - 2, ny - 1, 7, 5, 0, 1, k, -0.02),
             ghost.Rule(0, nx, ny - 2, ny - 1, 8, 6, 0, 1, k, 0.02),
             ghost.Rule(1, 2, 3, ny - 6, 4, 3, -1, 0, k, 0.01),         # source: the inlet
             ghost.Rule(nx - 2, nx - 1, 3, ny - 6, 4, 1, 1, 0, k, 0.01),  # the outlet
             ghost.Rule(4, 5, 3, ny - 6, 4, 2, -2, 0, k, 0.03),         # column 2, two away
             ghost.Rule(2, 3, 4, 9, 4, 0, -1, 1, k, 0.01)]              # column 1, beside the inlet
    args = (1.01, 0.99)
    r = np.random.default_rng(nx + steps)
    rho = (1 + 0.02 * r.standard_normal((nx, ny))).astype(ndt)
    ux, uy = ((0.03 * r.standard_normal((nx, ny))).astype(ndt) for _ in range(2))
    print("wall density", tdt, mode, nx, ny, steps, flush=True)
    lat = ghost.GhostLattice(nx, ny, 1.3, rules, (mode,) + args, dtype=tdt,
                             layout="soa" if steps == 7 else "rows")
    lat.init_equilibrium(rho, ux, uy)
    mom = lat.moment_buffers()
    lat.step(steps, moments=mom)
    G = g.equilibrium(rho, ux, uy)
    for _ in range(steps):
        if mode == "before":
            g.pressure_periodic(G, *args)
        g.stream(G)
        if mode == "after":
            g.pressure_periodic_after(G, *args)
        for q in rules:
            s = G[:, q.x0 + q.dx:q.x1 + q.dx, q.y0 + q.dy:q.y1 + q.dy]
            wall = 2.0 * (s[2] + s[5] + s[6]) + s[0] + s[1] + s[3]
            G[q.ch, q.x0:q.x1, q.y0:q.y1] = s[q.src_ch] + q.coef * wall
        omom = g.collide(G, 1.3)
    same(lat, mom, G, omom)


@pytest.mark.parametrize("tdt,ndt", DT)
@pytest.mark.parametrize("nx,ny,steps", [(329, 999, 11), (700, 500, 7), (120, 517, 6), (250, 250, 11)])
@pytest.mark.parametrize("flow", ["lid", "couette", "sides", "canal"])
def test_tile_shapes_match_oracle(gpu, flow, tdt, ndt, nx, ny, steps):
    # on 256 CUs: 22 x 32 tiles (inlet and outlet: 17 x 32) on the first two grids,
    # 17 x 32 on the third, 6 x 16 on the last; launches of 4 + 4 + 3, 4 + 2 + 1 and 4 + 2
    test_several_steps_per_launch_match_oracle(gpu, flow, tdt, ndt, nx, ny, steps)
