"""Downloads of finished jobs while the engine's worker renders others."""

import threading
import time

import numpy as np
import pytest

from ordinarylight_amd import _native as N
from ordinarylight_amd import workloads
from ordinarylight_amd.batch import BatchEngine, EngineSettings, Job
from ordinarylight_amd.renderers.hip import DeviceContext, DeviceScene, HipRendererConfig

pytestmark = pytest.mark.gpu

NAMES = ("depth", "normal", "primitive", "variance")


@pytest.fixture(scope="module")
def ctx(hip_device):
    c = DeviceContext(hip_device)
    yield c
    c.close()


@pytest.fixture(scope="module")
def scenes(ctx):
    built = {
        "room": workloads.tessellated_room(2, 4000),
        "textured": workloads.textured_room(1, open_sky=True),
        "inst": workloads.instanced_spheres(3, meshes=2, subdivisions=2, instances=40, box=10.0, emitters=30,
                                            emitter_size=0.3),
    }
    built["inst"][0].add_point_light((0.0, 12.0, 0.0), (1.0, 0.9, 0.8), 20.0)
    out = {k: (DeviceScene(ctx, s, 2, instanced=k == "inst"), cam) for k, (s, cam) in built.items()}
    yield out
    for ds, _ in out.values():
        ds.close()


def alone(ctx, job):
    with BatchEngine(ctx, EngineSettings(path_slots=1 << 20)) as engine:
        k = engine.submit(job)
        engine.run()
        products = engine.products(k)
        return products, engine.result(k)[0]


def same(got, want):
    return all(np.array_equal(got[n], want[n]) for n in NAMES)


@pytest.mark.parametrize("graph", [True, False])
def test_products_while_the_worker_meets_new_step_shapes(ctx, scenes, graph):
    """Products of done jobs, fetched while the worker captures and replays
    step shapes that it has not met (other scene kinds, reservoir passes,
    other accumulations), equal those of engines that render nothing else;
    so do the products and images of the jobs rendered meanwhile, and a job
    whose result is taken by another thread during the fetches."""
    both = N.PRODUCT_PRIMARY | N.PRODUCT_VARIANCE

    def job(key, w, h, samples, frame, bounces, **options):
        ds, cam = scenes[key]
        return Job(ds, cam, w, h, samples, frame, HipRendererConfig(max_bounces=bounces, **options), products=both)

    early = [job("room", 97, 65, 3, 0, 3), job("room", 640, 360, 2, 1, 2)]
    later = [job("inst", 96, 64, 2, 2, 5), job("textured", 80, 60, 3, 3, 4),
             job("inst", 64, 64, 3, 4, 4, wavefront_restir_di=True, wavefront_restir_candidates=8),
             job("room", 33, 17, 5, 5, 6), job("textured", 128, 72, 1, 6, 2), job("inst", 160, 90, 1, 7, 3)]
    want = {id(j): alone(ctx, j) for j in early + later}
    for _ in range(4):  # a new engine has captured nothing
        with BatchEngine(ctx, EngineSettings(path_slots=1 << 20, use_graph=graph)) as engine:
            engine.start()
            ids = [engine.submit(j) for j in early]
            taken = engine.submit(early[0])
            for k in ids + [taken]:
                assert engine.wait(k, 60) == N.JOB_DONE
            rendered, failures = [], []

            def feed():
                try:
                    for j in later:  # one after the other: each changes the resident kinds
                        k = engine.submit(j)
                        assert engine.wait(k, 60) == N.JOB_DONE
                        rendered.append((j, engine.products(k), engine.result(k)[0]))
                    image = engine.result(taken)[0]
                    rendered.append((early[0], want[id(early[0])][0], image))
                except BaseException as e:  # noqa: BLE001 - reported by the main thread
                    failures.append(e)

            feeder = threading.Thread(target=feed)
            feeder.start()
            fetched = 0
            while feeder.is_alive() or fetched < 2:
                for j, k in zip(early, ids):
                    assert same(engine.products(k), want[id(j)][0])
                try:
                    assert same(engine.products(taken), want[id(early[0])][0])
                except (KeyError, ValueError):
                    pass  # its result has been taken
                fetched += 1
            feeder.join()
            assert not failures, failures
            for j, products, image in rendered:
                assert same(products, want[id(j)][0])
                assert np.array_equal(image, want[id(j)][1])
            for j, k in zip(early, ids):
                assert np.array_equal(engine.result(k)[0], want[id(j)][1])


def test_scenes_and_rays_while_the_worker_meets_new_step_shapes(ctx, scenes):
    """A scene built and rays traced on the worker's context, while it captures
    step shapes, give what they give alone, and so do the worker's images."""
    built, _ = workloads.tessellated_room(5, 3000)
    rng = np.random.default_rng(1)
    o = rng.uniform(-1.0, 1.0, (5000, 3)).astype(np.float32)
    d = rng.normal(size=o.shape).astype(np.float32)
    d /= np.linalg.norm(d, axis=1, keepdims=True)

    def build_and_trace():
        ds = DeviceScene(ctx, built, 2)
        try:
            nodes, tri = ds.bvh_arrays()
            return [nodes, tri.view(np.uint32), *ds.trace(o, d, 0.001, 1e30), *ds.trace(o[:100], d[:100], 0.001, 1e30)]
        finally:
            ds.close()

    want = build_and_trace()
    jobs = [Job(*scenes[key], w, h, samples, 0, HipRendererConfig(max_bounces=bounces, **options), products=3)
            for key, w, h, samples, bounces, options in (
                ("room", 97, 65, 3, 3, {}), ("inst", 96, 64, 2, 5, {}), ("textured", 80, 60, 3, 4, {}),
                ("inst", 64, 64, 3, 4, {"wavefront_restir_di": True, "wavefront_restir_candidates": 8}),
                ("textured", 128, 72, 1, 2, {}))]
    images = [alone(ctx, j)[1] for j in jobs]
    for _ in range(4):
        with BatchEngine(ctx, EngineSettings(path_slots=1 << 20)) as engine:
            engine.start()
            done, failures = [], []

            def feed():
                try:
                    for j in jobs:
                        k = engine.submit(j)
                        assert engine.wait(k, 60) == N.JOB_DONE
                        done.append(engine.result(k)[0])
                except BaseException as e:  # noqa: BLE001 - reported by the main thread
                    failures.append(e)

            feeder = threading.Thread(target=feed)
            feeder.start()
            while feeder.is_alive():
                assert all(np.array_equal(a, b) for a, b in zip(build_and_trace(), want))
            feeder.join()
            assert not failures, failures
            assert all(np.array_equal(a, b) for a, b in zip(done, images))


@pytest.mark.parametrize("streams", range(4))
def test_a_result_does_not_wait_for_the_worker(hip_device, streams):
    """A finished image comes back beside a rendering worker about as fast as
    from an idle device: its copy neither needs compute units nor queues up
    behind the worker's steps, whichever of the process's four hardware queues
    the streams share (`streams`: contexts made before, one stream each)."""
    others = [DeviceContext(hip_device) for _ in range(streams)]
    ctx = DeviceContext(hip_device)
    heavy, heavy_cam = workloads.instanced_spheres(1, instances=2000, emitters=2000)
    light, light_cam = workloads.tessellated_room(1, 2000)
    heavy_scene, light_scene = DeviceScene(ctx, heavy, 2), DeviceScene(ctx, light, 2)
    with BatchEngine(ctx, EngineSettings(path_slots=1 << 24)) as engine:
        done = [engine.submit(Job(light_scene, light_cam, 512, 512, max_bounces=1)) for _ in range(64)]
        engine.run()

        frames = []

        def fetch(count, pause, worker):
            took = []
            for _ in range(count):
                while worker and sum(engine.poll(k) != N.JOB_DONE for k in frames[-4:]) < 3:
                    frames.append(engine.submit(Job(heavy_scene, heavy_cam, 1920, 1080, 4, 0, max_bounces=16)))
                time.sleep(pause)
                begin = time.perf_counter()
                engine.result(done.pop())
                took.append(time.perf_counter() - begin)
            return sorted(took)[int(0.9 * count)]

        fetch(8, 0.0, False)
        idle = fetch(16, 0.002, False)
        engine.start()
        fetch(4, 0.05, True)
        busy = fetch(32, 0.003, True)
        for k in frames:
            assert engine.wait(k, 60) == N.JOB_DONE
            engine.result(k, copy_image=False)
    for thing in (heavy_scene, light_scene, ctx, *others):
        thing.close()
    # 4 MB: 0.15 ms over the link; a launch of the worker's traversal lasts milliseconds.
    assert busy < 3.0 * idle + 0.5e-3, f"idle {1e3 * idle:.2f} ms, busy {1e3 * busy:.2f} ms"
