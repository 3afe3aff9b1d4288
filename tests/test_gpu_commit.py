"""Round commits at the sizes where one can go wrong -- slots around the
64-slot blocks a commit reads ahead, chains around the rows it moves at a
time, with the dynamic domain (a block reads radii the block before wrote) and
without -- bit for bit against the oracle's round-synchronous planner on the
point robot, whose arithmetic both share."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nnc", [1, 63, 64, 65, 130, 300])
@pytest.mark.parametrize("dd", [0, 1])
def test_commits_equal_the_oracle(nnc, dd, gpu, oracle_robots):
    from oracle import oracle
    from prrtc_amd import scenes as S
    R = oracle_robots["sphere"]
    # a wall with a gap far from the straight line: several rounds, chains of
    # many lengths (range 0.3: up to 20 nodes and more)
    sc = S.Scene.build(cuboids=[S.cuboid((0, -1.2, 0), (0, 0, 0), (0.2, 4.0, 6.0))],
                       spheres=[S.sphere((2, 2, 1), 0.7)])
    start, goal = np.array([-4, -1, 0.5], np.float32), np.array([4, -1.5, -0.5], np.float32)
    oracle.set_fused(True)
    try:
        for rng_, rounds in ((0.3, 4), (2.5, 6), (0.3, 400)):
            st = dict(num_new_configs=nnc, granularity=16, range=rng_, balance=2, tree_ratio=1.0, dynamic_domain=dd,
                      dd_alpha=0.05, dd_radius=2.0, dd_min_radius=0.5, max_samples=20000, max_iters=rounds,
                      seed=7)
            res, path = gpu.solve("sphere", start, goal[None], sc, st)
            _, want, opath = R.plan(sc, start, goal[None], st, mode=0)
            got = (res["solved"], res["iters"], res["start_tree_size"], res["goal_tree_size"], res["edge_checks"])
            assert got == (want.solved, want.iters, want.start_tree_size, want.goal_tree_size, want.edge_checks)
            assert path.tobytes() == opath.tobytes()
    finally:
        oracle.set_fused(False)


@pytest.mark.parametrize("robot", ["fetch", "baxter"])
def test_largest_scene_and_chains(robot, gpu):
    """The most LDS a planner workgroup can ask for: full obstacle tables (64
    KiB, and half as much for their balls) and chains of nearly 255 steps,
    alone and in a batch of two robots (one grid laid out for the largest)."""
    from prrtc_amd import scenes as S
    from prrtc_amd.robots import limits
    rng = np.random.default_rng(2)
    sc = S.Scene.build(z_cuboids=[S.cuboid(rng.uniform(3, 5, 3), (0, 0, 1.0), (0.05, 0.05, 0.05)) for _ in range(1024)])
    lo, span = limits(robot)
    q = (lo + span * rng.random((4096, len(lo)), dtype=np.float32)).astype(np.float32)
    q = q[gpu.check_poses(robot, sc, q)][:2]
    st = dict(num_new_configs=16, granularity=8, range=float(np.linalg.norm(span)) / 250, balance=2, tree_ratio=1.0,
              dynamic_domain=0, max_samples=20000, max_iters=3, seed=1)
    p = {"robot": robot, "start": q[0], "goals": q[1][None], "scene": sc}
    other = "fetch" if robot == "baxter" else "baxter"
    lo2, span2 = limits(other)
    q2 = (lo2 + span2 * rng.random((4096, len(lo2)), dtype=np.float32)).astype(np.float32)
    q2 = q2[gpu.check_poses(other, sc, q2)][:2]
    p2 = {"robot": other, "start": q2[0], "goals": q2[1][None], "scene": sc}
    alone, path = gpu.solve(robot, p["start"], p["goals"], sc, st)
    res, paths, _ = gpu.solve_batch([p, p2], [st, dict(st, range=float(np.linalg.norm(span2)) / 250)])
    for k in ("solved", "status", "iters", "start_tree_size", "goal_tree_size", "edge_checks", "path_nodes"):
        assert alone[k] == res[0][k]
    assert path.tobytes() == paths[0].tobytes()
    assert alone["start_tree_size"] + alone["goal_tree_size"] > 2
