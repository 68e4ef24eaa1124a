"""The library's host code on the CPU, against a HIP runtime of host memory whose
events and launches do what a test says (tests/host_stub): orders of events that
a device gives rarely, and waits between threads."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), 'hydro-cl-lua_amd', 'csrc')
STUB = os.path.join(HERE, 'host_stub')


@pytest.fixture(scope='module')
def objects(tmp_path_factory):
    """the host halves of hydro_hip.cpp and hydro_server.cpp, and the stub runtime"""
    if shutil.which('hipcc') is None:
        pytest.skip('needs hipcc')
    out = tmp_path_factory.mktemp('host_stub')
    objs = []
    for src in (os.path.join(CSRC, 'hydro_hip.cpp'), os.path.join(CSRC, 'hydro_server.cpp'), os.path.join(STUB, 'hip_stub.cpp')):
        obj = str(out / (os.path.basename(src) + '.o'))
        _compile(src, obj)
        objs.append(obj)
    return out, objs


def _compile(src, obj):
    subprocess.run(['hipcc', '-x', 'hip', '--offload-host-only', '-O1', '-fPIC', '-std=c++17', '-w', '-c', src, '-o', obj],
                   check=True)


def _run(objects, name):
    out, objs = objects
    obj, exe = str(out / (name + '.o')), str(out / name)
    _compile(os.path.join(STUB, name + '.cpp'), obj)
    # the system's linker driver: the stub stands in for the HIP runtime library
    subprocess.run(['g++', '-o', exe, obj, *objs, '-lpthread'], check=True)
    return subprocess.run([exe], capture_output=True, text=True, timeout=120)


def test_server_completes_chunks_in_launch_order(objects):
    r = _run(objects, 'server_order')
    assert r.returncode == 0 and 'in order' in r.stdout, r.stdout + r.stderr


def test_transfers_share_the_slots(objects):
    r = _run(objects, 'shared_slots')
    assert r.returncode == 0 and 'shared' in r.stdout, r.stdout + r.stderr


def test_launch_shape_round_trip(objects):
    r = _run(objects, 'launch_shape')
    assert r.returncode == 0 and 'as reported' in r.stdout, r.stdout + r.stderr


def test_launches_of_1d_steps(objects):
    r = _run(objects, 'launch_1d')
    assert r.returncode == 0 and 'as ruled' in r.stdout, r.stdout + r.stderr
