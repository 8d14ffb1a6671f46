"""A batch's verdict on the host - the words that a plan writes, who holds them until it has - without a GPU: the operators' source
built with one function more, which makes a verdict of words that the test fills in as the plan's kernel would."""
import importlib.util
import subprocess
import sys

import pytest
import torch

from conftest import ROOT


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    spec = importlib.util.spec_from_file_location("gact_build", ROOT + "/gact-icml_amd/build.py")
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    out = str(tmp_path_factory.mktemp("host") / "verdict_host.so")
    cmd = ["-O0" if c == "-O2" else out if c == build.TORCH_OUT else ROOT + "/tests/verdict_host.cpp" if c == build.TORCH_SRC else c
           for c in build.torch_command()]
    subprocess.run(cmd + ["-Wl,-rpath," + build.OUT_DIR], check=True)
    spec = importlib.util.spec_from_file_location("verdict_host", out)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


def words(need=-1, good=-1):
    return torch.tensor([need, good], dtype=torch.int64)


def test_a_verdict_that_is_there(host):
    w = words(1024, 1)
    assert host.verdict_wait(host.verdict(w)) == (1024, 1)
    assert w._use_count() == 1


def test_words_of_a_dropped_verdict_are_held_until_they_are_written(host):
    """And no longer: they went to nobody again where the memory's allocator refused to watch the stream for them."""
    held = [words() for _ in range(20)]
    for w in held:
        host.verdict(w)
    host.verdict(words(1, 1))
    assert all(w._use_count() == 2 for w in held)
    for w in held[:10]:
        w[0] = 512
    host.verdict(words(1, 1))
    assert all(w._use_count() == 2 for w in held)       # the second word is still to come
    for w in held[:10]:
        w[1] = 0
    host.verdict(words(1, 1))
    assert [w._use_count() for w in held] == [1] * 10 + [2] * 10
    for w in held[10:]:
        w.fill_(0)
    host.verdict(words(1, 1))
    assert all(w._use_count() == 1 for w in held)


def test_an_error_while_the_gil_is_released_is_raised(host):
    """No such GPU, or none that has such a plan: the wait ends with an exception, not with the interpreter."""
    code = ("import importlib.util, torch\n"
            "spec = importlib.util.spec_from_file_location('verdict_host', %r)\n"
            "host = importlib.util.module_from_spec(spec)\n"
            "spec.loader.exec_module(host)\n"
            "v = host.verdict(torch.full((2,), -1, dtype=torch.int64))\n"
            "for _ in range(2):\n"
            "    try:\n"
            "        host.verdict_wait(v)\n"
            "    except RuntimeError as e:\n"
            "        print('raised', e)\n" % host.__file__)
    done = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert done.returncode == 0 and done.stdout.count("raised") == 2, (done.returncode, done.stdout, done.stderr[-2000:])
