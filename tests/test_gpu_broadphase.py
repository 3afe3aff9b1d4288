"""The broad phase lists the obstacles a wave's poses can touch, 64 at a time
and dealt to the waves that share a pass.  Verdicts at the sizes where a list
can go wrong -- one obstacle, the ends of a 64-obstacle block in each table,
full tables -- against the oracle, for edges and for poses; a pose that is no
number; negative radii; and (on the CPU) the generated lists and balls.  The
balls' own arithmetic is run by test_reach.py."""
import numpy as np
import pytest

from conftest import NEAR, edge_margins

F32 = np.float32
# spheres, capsules, z-capsules, cuboids, z-cuboids
COUNTS = [(1, 0, 0, 0, 0), (0, 0, 0, 1, 0), (63, 1, 0, 0, 0), (64, 0, 1, 0, 0), (0, 65, 0, 0, 0), (0, 0, 64, 0, 1),
          (20, 20, 20, 20, 20), (0, 0, 0, 63, 2), (0, 0, 0, 0, 129), (4096, 0, 0, 0, 0), (0, 2048, 0, 0, 0),
          (0, 0, 0, 0, 1024)]


def _scene(counts, seed):
    """Small obstacles through the workspace, off the base axis."""
    from prrtc_amd import scenes as S
    rng = np.random.default_rng(seed)
    size = 0.12 / max(1.0, sum(counts) / 24.0) ** (1 / 3)   # about the same share of the space in obstacles

    def centre():
        while True:
            c = rng.uniform([-0.9, -0.9, 0.0], [0.9, 0.9, 1.3])
            if np.hypot(c[0], c[1]) > 0.35:
                return c
    sph = [S.sphere(centre(), size) for _ in range(counts[0])]
    cap = [S.cylinder_center(centre(), rng.uniform(-3, 3, 3), size / 2, 2 * size) for _ in range(counts[1])]
    zcap = [S.cylinder_center(centre(), (0, 0, 0), size / 2, 2 * size) for _ in range(counts[2])]
    cub = [S.cuboid(centre(), rng.uniform(-3, 3, 3), rng.uniform(size / 2, size, 3)) for _ in range(counts[3])]
    zcub = [S.cuboid(centre(), (0, 0, rng.uniform(-3, 3)), rng.uniform(size / 2, size, 3)) for _ in range(counts[4])]
    return S.Scene.build(sph, cap, zcap, cub, zcub)


@pytest.mark.gpu
@pytest.mark.parametrize("robot", ["panda", "fetch", "baxter", "ur5"])
@pytest.mark.parametrize("counts", COUNTS, ids=str)
def test_edges_against_oracle(robot, counts, gpu, oracle_robots):
    from prrtc_amd.robots import limits
    R = oracle_robots[robot]
    sc = _scene(counts, 5 + sum(counts))
    lo, span = limits(robot)
    rng = np.random.default_rng(11)
    n = 200 if sum(counts) < 1000 else 60
    a = (lo + span * rng.random((n, len(lo)), dtype=F32)).astype(F32)
    b = np.clip(a + rng.normal(size=a.shape) * rng.choice([0.01, 0.2], (n, 1)), lo, lo + span).astype(F32)
    edges = np.stack([a, b], 1)
    got = gpu.validate_edges(robot, sc, edges, 32)
    want = R.validate_edges(sc, edges, 32)
    flips = np.nonzero(got != want)[0]
    assert np.all(edge_margins(R, sc, edges[flips], 32) < NEAR)


@pytest.mark.gpu
@pytest.mark.parametrize("robot", ["panda", "fetch", "baxter", "ur5"])
@pytest.mark.parametrize("counts", COUNTS, ids=str)
def test_poses_against_oracle(robot, counts, gpu, oracle_robots):
    """Pose checks answer lane by lane, so lanes retire one by one while the
    balls of the gate pass stand: paths (checked by balls over the wave) and
    samples (checked pose by pose), in whole waves and a ragged one."""
    from prrtc_amd.robots import limits
    R = oracle_robots[robot]
    sc = _scene(counts, 7 + sum(counts))
    lo, span = limits(robot)
    rng = np.random.default_rng(13)
    few = sum(counts) > 1000
    samples = (lo + span * rng.random((70 if few else 301, len(lo)), dtype=F32)).astype(F32)
    u = rng.normal(size=(2 if few else 5, 1, len(lo)))
    u /= np.linalg.norm(u, axis=2, keepdims=True)
    paths = samples[:len(u), None, :] + np.linspace(0, 0.8, 64)[None, :, None] * u
    for q in (samples, paths.reshape(-1, len(lo)).astype(F32)[:-7]):
        got = gpu.check_poses(robot, sc, q)
        want, margin = R.check(sc, q, margin=True)
        assert np.all(margin[got != want] < NEAR)


@pytest.mark.gpu
def test_negative_radius(gpu, oracle_robots):
    """Obstacles of negative radius reach as far as the tests say, which square
    the sum of the radii: bit for bit against the oracle on the point robot,
    whose arithmetic both share."""
    from oracle import oracle
    from prrtc_amd import scenes as S
    R = oracle_robots["sphere"]
    rng = np.random.default_rng(4)
    sc = S.Scene.build([S.sphere((-2, 0, 0), -3.4)], [S.cylinder_center((2, 1, 0), (0.3, 1, 2), -3.1, 0.5)],
                       [S.cylinder_center((0, -3, 1), (0, 0, 0), -3.3, 0.4)])
    a = rng.uniform(-5, 5, (4000, 3)).astype(F32)
    edges = np.stack([a, a + rng.normal(size=a.shape).astype(F32) * F32(0.2)], 1)
    oracle.set_fused(True)
    try:
        want = R.validate_edges(sc, edges, 16)
        poses = R.check(sc, a)
    finally:
        oracle.set_fused(False)
    assert 0.1 < want.mean() < 0.9
    assert np.array_equal(gpu.validate_edges("sphere", sc, edges, 16), want)
    assert np.array_equal(gpu.check_poses("sphere", sc, a), poses)


@pytest.mark.gpu
def test_pose_that_is_no_number(gpu, oracle_robots):
    """A cuboid's test takes a NaN position for a hit (utils.cuh:158-175: the
    NaN is dropped by max(0, .)), a sphere's for none; neither may be lost
    because the wave's ball has no radius."""
    import torch
    from prrtc_amd import scenes as S
    far = (3.0, 3.0, 3.0)
    a = np.tile(np.array([0, -0.8, 0, -2.0, 0, 1.6, 0.8], F32), (3, 1))
    b = a + F32(0.1)
    b[1, 0] = np.nan      # every pose
    edges = torch.from_numpy(np.stack([a, b], 1)).cuda()
    for sc, want in ((S.Scene.build(cuboids=[S.cuboid(far, (0, 0, 0), (0.1,) * 3)]), [1, 0, 1]),
                     (S.Scene.build(spheres=[S.sphere(far, 0.1)]), [1, 1, 1])):
        packed = torch.from_numpy(gpu.pack_scene(sc)).cuda()
        out = torch.full((3,), 7, dtype=torch.uint8, device="cuda")
        gpu.validate_edges_async("panda", packed.data_ptr(), packed.numel(), edges.data_ptr(), 3, 32, out.data_ptr())
        torch.cuda.synchronize()
        assert out.cpu().tolist() == want


@pytest.mark.parametrize("robot", ["panda", "fetch", "baxter"])
def test_self_group_words(robot):
    """Each self group's word names its two gates by the number of their ball
    and holds at least the sum of their radii (padded by 1 mm, rounded up)."""
    import os
    import re
    from prrtc_amd.robots import load_model
    m = load_model(robot)
    here = os.path.join(os.path.dirname(__file__), "..", "prrtc_amd", "csrc", "robots")
    text = open(os.path.join(here, robot + ".gen.h")).read()
    words = [int(w, 16) for w in re.findall(r"0x[0-9a-f]+", re.search(r"self_gates\[\d+\] = \{(.*)\}", text).group(1))]
    selfs = [m["self_checks"][k] for kind, k in m["order"] if kind == "self"]
    number = [c["gate"] for c in m["env_checks"]]
    # gates that never move follow the environment gates, by their fixed_gate lines
    for k, xyz in re.findall(r"ctx\.fixed_gate\((\d+), (.*)\);", text):
        at = [np.float32(v.strip(" f")) for v in xyz.split(",")]
        number.append(next(i for i, s in enumerate(m["spheres"])
                           if s["frame"] < 0 and np.allclose(s["local"], at, atol=1e-7)))
        assert int(k) == len(number) - 1
    assert len(words) == len(selfs) and len(number) <= 64
    for w, chk in zip(words, selfs):
        a, b = chk["gate"]
        assert (number[w & 0xff], number[w >> 8 & 0xff]) == (a, b)
        reach = float(np.array(w >> 16, np.uint16).view(np.float16))
        rs = m["spheres"][a]["r"] + m["spheres"][b]["r"]
        assert rs + 0.99e-3 <= reach <= (rs + 1e-3) * 1.002


@pytest.mark.parametrize("robot", ["panda", "fetch"])
def test_split_groups_hold_every_pair(robot, oracle_robots):
    """Self groups tested sphere by sphere against the other link's ball: every
    pair of the group is emitted once, under its outer sphere, and on random
    poses the ball's reach holds each inner sphere with most of the 1 mm pad
    to spare (so a sphere out of reach collides with none of them)."""
    import os
    import re
    from prrtc_amd.robots import limits, load_model
    m = load_model(robot)
    sph = m["spheres"]
    here = os.path.join(os.path.dirname(__file__), "..", "prrtc_amd", "csrc", "robots")
    text = open(os.path.join(here, robot + ".gen.h")).read()
    by_label = {c["label"]: c for c in m["self_checks"]}
    lo, span = limits(robot)
    rng = np.random.default_rng(21)
    c = np.asarray(oracle_robots[robot].fk((lo + span * rng.random((500, len(lo)), dtype=F32)).astype(F32)))
    split = 0
    for label, body in re.findall(r"/\* self: (.*?) \*/(.*?)(?=/\* self: |\Z)", text, re.S):
        near = re.findall(r"near_point\(s(\d+)x, .*?, cx, cy, cz, ([0-9.e+-]+)f\)\)\) \{(.*?)\n            \}", body, re.S)
        if not near:
            continue
        split += 1
        chk = by_label[label]
        pairs = []
        for x, reach2, tests in near:
            x = int(x)
            got = [(int(a), int(b)) for a, b in re.findall(r"ctx\.self\(s(\d+)x, .*?, s(\d+)x, ", tests)]
            assert all(x in p for p in got)
            pairs += got
            inner = [p[0] if p[1] == x else p[1] for p in got]
            # the ball is about the gate of the inner spheres' side
            gate = chk["gate"][1 if chk["pairs"][0][0] == x or x in [p[0] for p in chk["pairs"]] else 0]
            hold = max(float(np.linalg.norm(c[:, y] - c[:, gate], axis=1).max()) + sph[y]["r"] for y in inner)
            assert hold + sph[x]["r"] <= np.sqrt(float(reach2)) - 0.9e-3
        assert sorted(pairs) == sorted(map(tuple, chk["pairs"]))
    assert split >= 5
