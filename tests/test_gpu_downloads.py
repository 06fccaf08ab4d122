"""Downloads through the pinned rings that a device's contexts share: from
several threads, and as the first of a new context."""

import threading
import time

import numpy as np
import pytest

from ordinarylight_amd import _native as N
from ordinarylight_amd import workloads
from ordinarylight_amd.batch import Job, plain_render
from ordinarylight_amd.renderers.hip import DeviceContext, DeviceScene

pytestmark = pytest.mark.gpu


class Frame:
    """A context whose last frame of edge x edge pixels stays on the device."""

    def __init__(self, device, edge):
        self.ctx = DeviceContext(device)
        scene, cam = workloads.tessellated_room(1, 2000)
        self.scene = DeviceScene(self.ctx, scene, 2)
        self.out = np.full((edge, edge, 4), -1.0, np.float32)
        plain_render(Job(self.scene, cam, edge, edge, max_bounces=1), copy_image=False)

    def download(self):
        begin = time.perf_counter()
        N.check(N.library().olhip_frame_download(self.ctx.handle, N.ptr(self.out)))
        return time.perf_counter() - begin

    def close(self):
        self.scene.close()
        self.ctx.close()


def test_downloads_from_many_threads(hip_device):
    """One image from six contexts in six threads at once: more than there are
    rings, so some are made and some downloads wait for one."""
    frames = [Frame(hip_device, 601) for _ in range(6)]
    frames[0].download()
    want = frames[0].out.copy()
    assert np.all(want[..., :3] >= 0.0) and want[..., :3].max() > 0.0
    wrong = []

    def loop(frame):
        for _ in range(20):
            frame.out.fill(-1.0)
            frame.download()
            if not np.array_equal(frame.out, want):
                wrong.append(frame)

    threads = [threading.Thread(target=loop, args=(f,)) for f in frames]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    for frame in frames:
        frame.close()


def test_the_first_download_of_a_context_costs_no_more_than_the_next(hip_device):
    """A context made beside another prepares nothing for its downloads: with
    pinned memory of its own its first 1 MB took 1 ms, the next ones 0.07."""
    other = Frame(hip_device, 512)
    other.download()
    first, later, new = [], [], []
    for _ in range(7):  # all open: what a closed one frees, the runtime hands to the next
        new.append(Frame(hip_device, 256))
        first.append(new[-1].download())
        later += [new[-1].download() for _ in range(5)]
    for frame in (other, *new):
        frame.close()
    first, later = sorted(first)[3], sorted(later)[17]
    assert first < 2.0 * later + 0.15e-3, f"first {1e3 * first:.3f} ms, later {1e3 * later:.3f} ms"


@pytest.mark.parametrize("edge", [1440, 601])
def test_downloads_right_after_device_memory_was_freed(hip_device, edge):
    """The driver wipes freed memory with the copy engine; a download that finds
    it late goes on by a kernel.  Same bytes, and not much slower (by the copy
    engine alone 33 MB took 4.7 ms then, 1.4 otherwise)."""
    frame = Frame(hip_device, edge)
    frame.download()
    want = frame.out.copy()
    idle = sorted(frame.download() for _ in range(9))[4]
    late = []
    for _ in range(3):
        ms = N.ctypes.c_double(0.0)  # allocates 4 GB and frees them
        N.check(N.library().olhip_bandwidth_probe(frame.ctx.handle, 1 << 31, 1, N.ctypes.byref(ms)))
        for _ in range(3):
            frame.out.fill(-1.0)
            late.append(frame.download())
            assert np.array_equal(frame.out, want)
    frame.close()
    late = sorted(late)[4]
    assert late < 2.5 * idle + 0.5e-3, f"idle {1e3 * idle:.2f} ms, after freeing {1e3 * late:.2f} ms"
