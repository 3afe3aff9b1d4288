"""Pose and edge checks on host buffers: the thread's kept buffers serve calls
of any order of sizes, from several threads, and calls above their limit take
the route of their own; every call answers as the device-buffer entry does."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _edges(n, seed):
    from prrtc_amd.robots import limits
    lo, span = limits("panda")
    rng = np.random.default_rng(seed)
    a = (lo + span * rng.random((n, 7), dtype=np.float32)).astype(np.float32)
    return np.stack([a, a + rng.normal(size=a.shape).astype(np.float32) * np.float32(0.05)], 1)


def _device_answer(gpu, scene, edges, g):
    import torch
    packed = torch.from_numpy(gpu.pack_scene(scene)).cuda()
    e = torch.from_numpy(edges).cuda()
    out = torch.full((len(edges),), 9, dtype=torch.uint8, device="cuda")
    gpu.validate_edges_async("panda", packed.data_ptr(), packed.numel(), e.data_ptr(), len(edges), g, out.data_ptr())
    torch.cuda.synchronize()
    return out.cpu().numpy().astype(bool)


def test_sizes_and_threads(gpu):
    from prrtc_amd import scenes as S
    sc = S.scene_obb_cylinders(3)
    # 400k edges are 22 MB: above the kept buffers
    sets = [(n, _edges(n, n)) for n in (3, 70_000, 1, 400_000, 5000)]
    want = {n: _device_answer(gpu, sc, e, 2) for n, e in sets}
    bad = []

    def work():
        for n, e in sets:
            if not np.array_equal(gpu.validate_edges("panda", sc, e, 2), want[n]):
                bad.append(("edges", n))
            poses = np.ascontiguousarray(e[:, 1])
            # an edge at granularity 1 is its end pose
            if not np.array_equal(gpu.check_poses("panda", sc, poses), gpu.validate_edges("panda", sc, e, 1)):
                bad.append(("poses", n))
    threads = [threading.Thread(target=work) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.parametrize("n", [5, 400_000])
def test_refused_as_before(gpu, n):
    from prrtc_amd import scenes as S
    from prrtc_amd.lib import PrrtcError
    sc = S.scene_obb_cylinders(3)
    e = _edges(n, 1)
    e[n - 1, 1, 6] = np.inf
    for call in (lambda: gpu.validate_edges("panda", sc, e, 4),
                 lambda: gpu.check_poses("panda", sc, np.ascontiguousarray(e[:, 1]))):
        with pytest.raises(PrrtcError) as err:
            call()
        assert err.value.code == -1 and "non-finite" in str(err.value)
    big = S.Scene.build(spheres=[S.sphere((9, 9, 9), 0.1)] * 4097)
    e[n - 1, 1, 6] = 0.0
    with pytest.raises(PrrtcError) as err:
        gpu.validate_edges("panda", big, e, 4)
    assert err.value.code == -1 and "scene tables exceed" in str(err.value)
    ok = gpu.validate_edges("panda", sc, e[:3], 4)
    assert ok.shape == (3,)
