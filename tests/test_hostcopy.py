"""The pinned copy pipeline when several threads use it at once: one has the
buffers, the others take the runtime's copy.  On the CPU the pipeline's source
runs over host memory under the thread sanitizer (hostcopy_stub.cpp); on the
GPU, several threads fetch from one server.  Memory that the runtime knows
(pinned, managed) is the runtime's to copy."""
import os
import subprocess
import threading

import numpy as np
import pytest

import mfmhd

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = [os.path.join(HERE, "hostcopy_stub.cpp"),
       os.path.join(os.path.dirname(HERE), "ms-flukss-multifluid_amd", "csrc", "mfm_hostcopy.cpp")]
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def build(tmp, flags):
    """The host half of the pipeline with the stub's HIP calls."""
    cxx = os.path.join(ROCM, "bin", "amdclang++")
    objs = []
    for src in SRC:
        objs.append(str(tmp / (os.path.basename(src) + ".o")))
        subprocess.run([cxx, "-x", "hip", "--offload-host-only", "--offload-arch=gfx950", "-O1",
                        "-std=c++17", *flags, "-c", src, "-o", objs[-1]], check=True)
    exe = str(tmp / "hostcopy")
    subprocess.run([cxx, *flags, "-o", exe, *objs, "-lpthread"], check=True)
    return exe


def test_threads_share_one_link(tmp_path):
    exe = build(tmp_path, ["-Xarch_host", "-fsanitize=thread"])
    r = subprocess.run([exe, "race"], capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, TSAN_OPTIONS="halt_on_error=1"))
    assert r.returncode == 0, r.stderr[:2000]
    assert "copies right" in r.stdout


@pytest.mark.parametrize("program", ["pinned", "small"])
def test_runtime_copies(tmp_path, program):
    """Memory that the runtime knows, and copies below the pipeline's size: one
    runtime copy where the bytes between the segments may go along (a small
    state's components), else one per segment."""
    r = subprocess.run([build(tmp_path, []), program], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "copies right" in r.stdout, r.stdout + r.stderr[:2000]


def test_threads_that_do_not_start(tmp_path):
    """A thread's own allocation fails: its part is copied by the caller, and
    no exception leaves the C entry point."""
    r = subprocess.run([build(tmp_path, []), "alloc"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "copies right" in r.stdout, r.stdout + r.stderr[:2000]


@pytest.mark.gpu
def test_threads_fetch_from_one_server():
    from test_serve import req_params, run_until_done
    p, dx = req_params(40)  # 11 MB of state each
    srv = mfmhd.Server(p, 8 << 30)
    ids = [srv.submit(p, dx, q + 1, 0.5) for q in range(4)]
    run_until_done(srv, lambda: ids)
    want = [srv.fetch(q) for q in ids]
    wrong = []

    def fetch(q):
        for _ in range(4):
            if not np.array_equal(srv.fetch(ids[q]), want[q]):
                wrong.append(q)
    threads = [threading.Thread(target=fetch, args=(q,)) for q in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    srv.close()
    assert not wrong
