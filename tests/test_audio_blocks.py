"""What the audio decoder's calls allocate (host/phonon_audio.c on stub_device.c,
without a GPU): nothing once as many calls as ever have run at the same moment,
everything given back with the last model and state, and a call that finds no
memory refused with its request unharmed."""
import ctypes
import os
import subprocess
import threading

import numpy as np
import pytest

import helpers

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CALLS = 8


@pytest.fixture(scope="module")
def host(pkg, tmp_path_factory):
    path = str(tmp_path_factory.mktemp("audio") / "libaudio_host.so")
    src = [os.path.join(ROOT, "tests", "stub_device.c")] + [
        os.path.join(ROOT, "speech-mac_amd", "host", f) for f in ("phonon_audio.c", "ph_runtime.c")]
    subprocess.run(["gcc", "-std=gnu17", "-O1", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "include"), *src, "-o", path, "-lm", "-lpthread"],
                   check=True)
    lib = ctypes.CDLL(path)
    for name, (restype, argtypes) in pkg.EXPORTS.items():
        if name.startswith(("phonon_mimi_", "phonon_conv_", "phonon_pcm_")) and hasattr(lib, name):
            getattr(lib, name).restype, getattr(lib, name).argtypes = restype, argtypes
    lib.stub_held.restype = ctypes.c_size_t
    return lib


def fp(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_float))


class Request:
    def __init__(self, lib, model):
        self.lib, self.h = lib, ctypes.c_void_p()
        assert lib.phonon_pcm_state_create(model, ctypes.byref(self.h)) == 1

    def call(self, frames):
        x, y = np.zeros((frames, 32), np.float32), np.zeros(frames * 1920, np.float32)
        self.ok = self.lib.phonon_pcm_process(self.h, fp(x), frames, fp(y), y.size, None, 0)
        return self.ok


def together(lib, requests, frames):
    """One call of each request, all of them in flight at the same moment."""
    lib.stub_wait_for(len(requests))
    threads = [threading.Thread(target=r.call, args=(frames,)) for r in requests]
    for t in threads:
        t.start()
    for t in threads:
        t.join(30)
    lib.stub_wait_for(0)
    assert all(r.ok == 1 for r in requests)


@pytest.fixture
def model(host, pkg):
    views = pkg.Views()
    before = host.stub_held()
    _, handle = helpers.pcm_model(host, pkg, views, helpers.mimi_identity_model(route_only=True),
                                  helpers.pcm_scalar_convs())
    requests = [Request(host, handle) for _ in range(CALLS)]
    yield requests, handle
    for r in requests:
        host.phonon_pcm_state_destroy(r.h)
    host.phonon_pcm_model_destroy(handle)
    # All but what the process keeps from the first state on: the phase table and
    # the library's stream.
    assert host.stub_held() - before in (0, 8192 * 16 * 64 * 4 + 1)


def test_calls_in_step_allocate_once(host, model):
    requests, _ = model
    for frames in (1, 9):
        together(host, requests, frames)
        made, released = host.stub_made(), host.stub_released()
        for _ in range(3):
            together(host, requests, frames)
        assert (host.stub_made(), host.stub_released()) == (made, released)


def test_a_frame_at_a_time_holds_little(host, model):
    """Eight states a frame at a time hold 8 x 11.5 MB of intermediates and 8 x 0.13
    of pinned memory; a block for 64 frames alone is 92."""
    requests, _ = model
    before = host.stub_held()
    together(host, requests, 1)
    assert 0 < host.stub_held() - before < CALLS * 12_000_000


def test_states_that_go_give_theirs_back(host, model):
    requests, handle = model
    held = host.stub_held()
    requests.append(Request(host, handle))
    state = host.stub_held() - held
    together(host, requests, 1)
    full = host.stub_held()
    while len(requests) > 1:
        host.phonon_pcm_state_destroy(requests.pop().h)
    given = full - host.stub_held() - CALLS * state
    assert given >= (CALLS - 2) * 11_500_000
    # Requests that come and go one after another allocate no intermediates.
    assert requests[0].call(1) == 1
    held = host.stub_held()
    r = Request(host, handle)
    assert r.call(1) == 1 and host.stub_held() - held == state
    host.phonon_pcm_state_destroy(r.h)


def test_a_call_without_memory_leaves_its_request_usable(host, model):
    requests, _ = model
    r = requests[0]
    assert r.call(2) == 1 and host.phonon_pcm_samples(r.h) == 2 * 1920
    host.stub_fail(1)
    assert r.call(40) == 0  # no block of that size yet
    host.stub_fail(0)
    assert host.phonon_pcm_samples(r.h) == 2 * 1920
    assert r.call(40) == 1 and host.phonon_pcm_samples(r.h) == 42 * 1920


def test_a_mimi_call_without_memory_leaves_its_state_usable(host, pkg):
    views, h = pkg.Views(), ctypes.c_void_p()
    m = helpers.mimi_model(host, pkg, views, helpers.mimi_identity_model())
    assert host.phonon_mimi_state_create(ctypes.byref(m), ctypes.byref(h)) == 1
    x, y = np.zeros((3, 32), np.float32), np.zeros((48, 512), np.float32)
    host.stub_fail(1)
    assert host.phonon_mimi_process(h, fp(x), 3, fp(y), 48) == 0
    host.stub_fail(0)
    assert host.phonon_mimi_positions(h) == 0
    assert host.phonon_mimi_process(h, fp(x), 3, fp(y), 48) == 1
    assert host.phonon_mimi_positions(h) == 48
    host.phonon_mimi_state_destroy(h)
