"""The native host path (mograd_amd/native/graph.cpp) without a GPU: the package over a library that
records its calls (tests/host_cpp/stub_library.cpp)."""
import ctypes as C
import gc
import subprocess
import threading
from pathlib import Path

import numpy as np
import pytest

from mograd_amd import _lib
from mograd_amd import runtime as R
from mograd_amd.runtime import F32, AnyBuffer, Device, Layout, Node, evaluate, evaluate_many

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def stub_path(tmp_path_factory):
    out = tmp_path_factory.mktemp("stub") / "libstub.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", f"-I{ROOT / 'include'}",
                    str(ROOT / "tests" / "host_cpp" / "stub_library.cpp"), "-o", str(out)], check=True)
    return out


class Host:
    """The package's Device over the stub, and the stub's record."""

    def __init__(self, lib):
        self.dll, self.device = lib._dll, Device()
        self.dll.stub_log.restype = C.c_int64
        self.dll.stub_log.argtypes = [C.c_char_p, C.c_int64]
        self.reset()

    def reset(self, pause_us=0):
        self.dll.stub_reset(pause_us)

    def log(self):
        n = self.dll.stub_log(None, 0)
        text = C.create_string_buffer(n + 1)
        self.dll.stub_log(text, n + 1)
        return text.value.decode().splitlines()

    def leaf(self, *shape, dtype=F32, value=1.0):
        array = np.full(shape, value, np.float32 if dtype == F32 else np.int32)
        return Node.leaf(Layout(*shape), dtype, AnyBuffer.from_numpy(self.device, array, dtype))


@pytest.fixture
def host(stub_path, monkeypatch):
    before = _lib._LIB
    lib = _lib._Lib(stub_path)
    monkeypatch.setattr(_lib, "_LIB", lib)
    yield Host(lib)
    gc.collect()
    if before is not None:  # the extension calls the library that was bound last
        before.__init__(before.path)


def linear_grad(host, n=3, k=4, m=2):
    """LINEAR_GRAD of an (m, k) input and an (n, k) weight, and its selectors."""
    lin = Node("LINEAR_GRAD", Layout(m, k), F32, [host.leaf(m, n), host.leaf(m, k), host.leaf(n, k)], {"has_bias": True})
    return lin, [Node("GETTUPLE", Layout(*shape), F32, [lin], {"index": i}) for i, shape in enumerate([(m, k), (n, k), (n,)])]


def test_threads_that_share_a_graph_keep_each_others_operands(host):
    # Two threads evaluate the same eight-node chain: whoever comes second replaces the buffers that
    # the first one's call is reading, which must stay allocated until that call is over.
    host.reset(pause_us=50)
    for _ in range(40):
        leaf = host.leaf(16)
        chain = leaf
        for i in range(8):
            chain = Node("ADD", Layout(16), F32, [chain, leaf]) if i % 2 else Node("RELU", Layout(16), F32, [chain])
        out, start = [], threading.Barrier(2)

        def work():
            start.wait()
            out.append(evaluate(chain, host.device).to_numpy())

        threads = [threading.Thread(target=work) for _ in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        for values in out:
            np.testing.assert_array_equal(values, np.full(16, 5.0, np.float32))
    assert host.dll.stub_violations() == 0


def test_what_a_walk_reads_of_a_node_is_the_walks_own(host, monkeypatch):
    # A walk that starts while another one is under way (here from an op's own exec function, as it
    # would on another thread) must not change which results the first one makes.
    lin, (dx, dw, _) = linear_grad(host)

    def probe(node, inputs, device):
        with pytest.raises(R.MogradError, match="without a buffer"):
            evaluate_many([Node.leaf(Layout(1), F32), dw], device)
        return [inputs[0]]

    monkeypatch.setitem(R.SCHEDULER_RULES, "PROBE", probe)
    del lin
    evaluate_many([Node("PROBE", Layout(2), F32, [host.leaf(2)]), dx, dw], host.device)
    assert host.log() == ["linear_bwd dx dw db"]


def test_a_left_out_result_is_made_when_it_is_asked_for(host):
    # evaluate_many([dW]) leaves out the dX that nobody holds; evaluating the LINEAR_GRAD itself
    # afterwards gives dX, and dW and db stay the buffers they were.
    lin, (_, dw, db) = linear_grad(host)
    del _, lin
    bw, bb = evaluate_many([dw, db], host.device)
    assert host.log() == ["linear_bwd dw db"] and dw.src(0).bufs == [None, bw, bb]
    got = evaluate(dw.src(0), host.device)
    assert got.to_numpy((2, 4))[0, 0] == 1.0
    assert host.log() == ["linear_bwd dw db", "linear_bwd dx"] and dw.src(0).bufs == [got, bw, bb]
    assert evaluate(dw.src(0), host.device) is got and evaluate(dw, host.device) is bw
    assert len(host.log()) == 2


@pytest.mark.parametrize("how", ["selector", "operand", "root"])
def test_a_left_out_result_reaches_every_reader(host, how):
    lin, (_, dw, _) = linear_grad(host)
    del _, lin
    evaluate(dw, host.device)
    lin = dw.src(0)
    if how == "selector":
        node = Node("GETTUPLE", Layout(2, 4), F32, [lin], {"index": 0})
    elif how == "operand":
        node = Node("RELU", Layout(2, 4), F32, [lin])
    else:
        node = lin
    assert evaluate_many([dw, node], host.device)[1].to_numpy()[0] == 1.0
    assert host.log()[:2] == ["linear_bwd dw db", "linear_bwd dx"]


def test_a_result_that_is_still_held_is_not_left_out(host):
    # Its selector is kept for later: dX is that of the weights as they are at the first evaluation.
    _, (dx, dw, _) = linear_grad(host)
    del _
    evaluate(dw, host.device)
    assert host.log() == ["linear_bwd dx dw db"]
    assert evaluate(dx, host.device).to_numpy()[0] == 1.0 and len(host.log()) == 1
