"""What the audio decoder's calls allocate (host/phonon_audio.c on stub_device.c,
without a GPU): everything is given back with the last model and state, and a call
that finds no memory is refused with its request unharmed."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import helpers

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


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


@pytest.fixture
def model(host, pkg):
    views = pkg.Views()
    before = host.stub_held()
    _, handle = helpers.pcm_model(host, pkg, views, helpers.mimi_identity_model(route_only=True),
                                  helpers.pcm_scalar_convs())
    requests = [Request(host, handle)]
    yield requests, handle
    for r in requests:
        host.phonon_pcm_state_destroy(r.h)
    host.phonon_pcm_model_destroy(handle)
    # All but what the process keeps from the first state on: the phase table and
    # the library's stream.
    assert host.stub_held() - before in (0, 8192 * 16 * 64 * 4 + 1)


def test_a_call_without_memory_leaves_its_request_usable(host, model):
    requests, _ = model
    r = requests[0]
    host.stub_fail(1)
    assert r.call(40) == 0
    host.stub_fail(0)
    assert host.phonon_pcm_samples(r.h) == 0
    assert r.call(40) == 1 and host.phonon_pcm_samples(r.h) == 40 * 1920


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
