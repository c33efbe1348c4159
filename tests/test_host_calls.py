"""What an operator asks of the HIP runtime, seen from a program that stands in for the runtime
(tests/cxx/host_calls.cpp): no GPU is needed and nothing is launched."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def host_calls(tmp_path_factory):
    """Runs the program; returns its lines after each argument that is a word, as (word, lines)."""
    exe = str(tmp_path_factory.mktemp("host_calls") / "host_calls")
    lib = os.path.join(ROOT, "meltpooldg_amd")
    r = subprocess.run(["g++", "-std=c++17", "-O1", os.path.join(ROOT, "tests", "cxx", "host_calls.cpp"), "-o", exe, "-L" + lib,
                        "-lmpdg_heat", "-Wl,-rpath," + lib, "-rdynamic"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def run(*words):
        r = subprocess.run([exe] + [str(w) for w in words], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stdout + r.stderr
        steps = []
        for line in r.stdout.splitlines():
            if line.split()[0] in ("alloc", "launch", "rc"):
                steps[-1][1].append(line)
            else:
                steps.append((line, []))
        return steps

    return run


def lines(step, word):
    return [line for line in step[1] if line.startswith(word)]


# the first apply of an operator can stand in a graph capture, where nothing may be allocated: also on the
# meshes whose applies share no rows between columns of cells
@pytest.mark.parametrize("degree", [1, 2, 3])
@pytest.mark.parametrize("nc", [(64, 64, 64), (40, 3, 2), (5, 40, 3), (33, 17, 9)])
def test_first_apply_allocates_nothing(host_calls, degree, nc):
    for precision, apply in ((0, "vmult"), (0, "vmult_noalloc"), (1, "vmult_f32")):
        create, first = host_calls("create", degree, *nc, precision, apply)
        assert lines(create, "rc") == ["rc 0"]
        assert not lines(first, "alloc")
        assert lines(first, "launch") and lines(first, "rc") == ["rc 0"]


# an operator made before its caller selects the GPU that it runs on
@pytest.mark.parametrize("degree,precision,apply", [(1, 0, "vmult"), (2, 1, "vmult_f32"), (3, 0, "vmult"), (3, 1, "vmult_f32")])
def test_scratch_follows_the_device_of_the_apply(host_calls, degree, precision, apply):
    create, _, there, again = host_calls("create", degree, 20, 9, 10, precision, "device", 1, apply, apply)
    assert [line.split()[1] for line in lines(create, "alloc")] == ["0"]
    assert [line.split()[1] for line in lines(there, "alloc")] == ["1"]
    assert lines(there, "launch") and lines(there, "rc") == ["rc 0"]
    assert not lines(again, "alloc") and lines(again, "launch") and lines(again, "rc") == ["rc 0"]


def test_noalloc_refuses_scratch_of_another_device(host_calls):
    _, _, there, _, back = host_calls("create", 2, 20, 9, 10, 0, "device", 1, "vmult_noalloc", "device", 0, "vmult_noalloc")
    assert there[1] == ["rc -2"]
    assert not lines(back, "alloc") and lines(back, "launch") and lines(back, "rc") == ["rc 0"]
    # no planes are shared here: no scratch is needed
    _, _, there = host_calls("create", 2, 3, 1, 2, 0, "device", 1, "vmult_noalloc")
    assert lines(there, "launch") and lines(there, "rc") == ["rc 0"]


@pytest.mark.parametrize("degree", [1, 2, 3])
def test_noalloc_of_a_tangent_without_scratch_is_out_of_memory(host_calls, degree):
    _, create, _, tangent, apply = host_calls("refuse", 64, "create", degree, 20, 9, 10, 0, "refuse", 2 ** 40, "tangent", "vmult_noalloc")
    assert create[1] == ["rc 0"] and lines(tangent, "rc") == ["rc 0"]
    assert apply[1] == ["rc -2"]


# the metric (7 values per point) and the tangent's coefficients (8) take no room for cells that are not there,
# but for one block of 16 cells
@pytest.mark.parametrize("degree", [1, 2, 3, 4])
@pytest.mark.parametrize("nc", [(1, 9, 7), (17, 5, 6), (16, 2, 3), (31, 3, 1)])
def test_point_data_is_not_padded(host_calls, degree, nc):
    points = (degree + 1) ** 3
    cells = nc[0] * nc[1] * nc[2]
    blocks = cells if degree == 4 else (cells + 15) // 16 * 16
    for precision, item in ((0, 8), (1, 4)):
        _, mapping = host_calls("create", degree, *nc, precision, "mapping")
        assert lines(mapping, "alloc") == ["alloc 0 %d" % (item * 7 * points * blocks)]
    _, tangent = host_calls("create", degree, *nc, 0, "tangent")
    assert lines(tangent, "alloc")[0] == "alloc 0 %d" % (8 * 8 * points * blocks)
