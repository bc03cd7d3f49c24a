"""The native host path (mograd_amd/native/graph.cpp) without a GPU: the package over a library that
records its calls (tests/host_cpp/stub_library.cpp)."""
import collections
import copy
import ctypes as C
import gc
import pickle
import subprocess
import sys
import threading
import weakref
from pathlib import Path

import numpy as np
import pytest

from mograd_amd import _lib
from mograd_amd import runtime as R
from mograd_amd.rewrites import GPU_REWRITES, Pat, Rule, Simplifier
from mograd_amd.runtime import F32, AnyBuffer, Device, Layout, Node, evaluate, evaluate_many

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def stub_path(tmp_path_factory):
    out = tmp_path_factory.mktemp("stub") / "libstub.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-Wl,-Bsymbolic", f"-I{ROOT / 'include'}",
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


def packed_attention(host, grad=False, **attrs):
    B, S, H, D = 1, 4, 2, 8
    qkv = host.leaf(B, S, 3, H, D)
    if not grad:
        return Node("FLASH_ATTN_PACKED", Layout(B, S, H, D), F32, [qkv], attrs)
    return Node("FLASH_ATTN_PACKED_GRAD", Layout(B, S, 3, H, D), F32,
                [host.leaf(B, S, H, D), host.leaf(B, S, H, D), qkv, host.leaf(B, H, S)], attrs)


def test_missing_attributes_are_errors(host):
    x, g = host.leaf(2, 4), host.leaf(4)
    norm = Node("LAYER_NORM_STATS", Layout(2, 4), F32, [x, g, g], {"eps": 1e-5})
    cases = {
        "scale": [packed_attention(host, is_causal=True), packed_attention(host, True, is_causal=True)],
        "is_causal": [packed_attention(host, scale=0.5), packed_attention(host, True, scale=0.5)],
        "eps": [Node("LAYER_NORM_STATS", Layout(2, 4), F32, [x, g, g])],
        "index": [Node("GETTUPLE", Layout(2, 4), F32, [norm])],
    }
    for name, nodes in cases.items():
        for node in nodes:
            with pytest.raises(KeyError, match=name):
                evaluate(node, host.device)
            assert node.bufs is None
    assert all(line.startswith("layer_norm_stats") for line in host.log())  # GETTUPLE's source alone ran


def test_attributes_are_converted_as_the_python_forms_do(host):
    evaluate(packed_attention(host, scale=np.float32(0.5), is_causal=np.bool_(True), has_bias=0), host.device)
    evaluate(packed_attention(host, scale="0.25", is_causal=1, has_bias=[]), host.device)
    assert host.log() == ["attn_packed 0.500000 1.000000 0.000000", "attn_packed 0.250000 1.000000 0.000000"]


def test_operands_without_dimensions_are_errors(host):
    s, ids = Node.leaf(Layout(), F32, host.leaf(1).bufs[0]), host.leaf(1, dtype=R.I32)
    m, one = host.leaf(2, 2), host.leaf(1)
    for op, srcs, attrs in (("CROSS_ENTROPY_IDS", [s, ids], {}), ("CROSS_ENTROPY_IDS_GRAD", [s, ids, one], {}),
                            ("LAYER_NORM_STATS", [s, one, one], {"eps": 1e-5}),
                            ("LAYER_NORM_STATS_GRAD", [s, s, one, one, one], {}), ("MATMUL_BT", [m, m], {}),
                            ("SCATTER_ADD", [ids, host.leaf(1, 3)], {})):
        with pytest.raises(IndexError):
            evaluate(Node(op, Layout(), F32, srcs, attrs), host.device)
    loss = Node("CROSS_ENTROPY_IDS", Layout(), F32, [s, ids])
    with pytest.raises(IndexError):
        evaluate_many([loss, Node("CROSS_ENTROPY_IDS_GRAD", Layout(), F32, [s, ids, one])], host.device)
    assert host.log() == []


def test_dtypes_and_ops_that_are_none_of_ours(host):
    for dtype in (99, -1, 1 << 80):
        with pytest.raises(R.MogradError, match="dtype"):
            evaluate(Node("RELU", Layout(2), dtype, [host.leaf(2)]), host.device)
    for op in (7, None, "NO_SUCH_OP"):
        with pytest.raises(R.MogradError, match="no scheduler rule"):
            evaluate(Node(op, Layout(2), F32, [host.leaf(2)]), host.device)
        node = Node(op, Layout(2), F32, [host.leaf(2)])
        assert Simplifier(GPU_REWRITES()).run(node) is node


def test_a_loss_and_its_gradient_are_one_pass(host):
    logits, ids, one = host.leaf(3, 5), host.leaf(3, dtype=R.I32, value=2), host.leaf(1)
    loss = Node("CROSS_ENTROPY_IDS", Layout(1), F32, [logits, ids])
    grad = Node("CROSS_ENTROPY_IDS_GRAD", Layout(3, 5), F32, [logits, ids, one])
    a, b = evaluate_many([loss, grad], host.device)
    assert (a.item(), b.to_numpy()[0]) == (4.0, 5.0) and host.log() == ["ce_fused_ids 3.000000 5.000000"]
    # not where the upstream comes from the walk, or another loss does
    host.reset()
    up = Node("RELU", Layout(1), F32, [host.leaf(1)])
    loss = Node("CROSS_ENTROPY_IDS", Layout(1), F32, [logits, ids])
    evaluate_many([loss, Node("CROSS_ENTROPY_IDS_GRAD", Layout(3, 5), F32, [logits, ids, up])], host.device)
    assert host.log() == ["ce_ids 3.000000 5.000000 dtype 3", "relu", "ce_grad_ids 3.000000 5.000000"]


def test_sources_without_results_are_errors(host, monkeypatch):
    with pytest.raises(R.MogradError, match="without a buffer"):
        evaluate(Node("RELU", Layout(2), F32, [Node.leaf(Layout(2), F32)]), host.device)
    monkeypatch.setitem(R.SCHEDULER_RULES, "EMPTY", lambda node, inputs, device: [])
    with pytest.raises(IndexError):
        evaluate(Node("RELU", Layout(2), F32, [Node("EMPTY", Layout(2), F32, [host.leaf(2)])]), host.device)


def test_sources_may_be_any_sequence(host):
    leaf = host.leaf(4)
    for make in (tuple, list, collections.deque):
        mid = Node("ADD", Layout(4), F32, make([leaf, leaf]))
        out = Node("RELU", Layout(4), F32, make([mid]))
        assert R._toposort(out) == [leaf, mid, out]
        assert Simplifier(GPU_REWRITES()).run(out) is out
        (g,) = R.gradient(out, host.leaf(4), [leaf])
        assert g.op_type == "ADD"
        np.testing.assert_array_equal(evaluate(out, host.device).to_numpy(), np.full(4, 2.0))
    for bad in (None, 3, [leaf, "x"]):
        with pytest.raises(TypeError):
            evaluate(Node("RELU", Layout(4), F32, bad), host.device)


def test_a_rewritten_graph_over_tuples(host):
    x, w, r = host.leaf(2, 4), host.leaf(3, 4), host.leaf(2, 3)
    out = Node("ADD", Layout(2, 3), F32, (Node("MATMUL_BT", Layout(2, 3), F32, (x, w)), r))
    top = Node("RELU", Layout(2, 3), F32, (out,))
    new = Simplifier(GPU_REWRITES()).run(top)
    assert new.src(0).op_type == "MATMUL_BT_ADD" and new.src(0).srcs == [x, w, r]


def test_gettuple_counts_from_the_end(host):
    lin, _ = linear_grad(host)
    get = lambda i: Node("GETTUPLE", Layout(3), F32, [lin, lin], {"index": i})  # noqa: E731
    got = [evaluate(get(i), host.device) for i in (-1, -2, -3, 2)]
    assert got == [lin.bufs[2], lin.bufs[1], lin.bufs[0], lin.bufs[2]] and len(host.log()) == 1
    for i in (3, -4):
        with pytest.raises(IndexError):
            evaluate(get(i), host.device)


def test_results_may_be_any_sequence(host, monkeypatch):
    buf = host.leaf(4).bufs[0]
    monkeypatch.setitem(R.SCHEDULER_RULES, "PAIR", lambda node, inputs, device: (buf, inputs[0]))
    pair = Node("PAIR", Layout(4), F32, [host.leaf(4)])
    assert evaluate(Node("GETTUPLE", Layout(4), F32, [pair], {"index": -1}), host.device) is pair.src(0).bufs[0]
    leaf = Node("BUFFER", Layout(4), F32, bufs=(buf,))
    evaluate(Node("RELU", Layout(4), F32, [leaf]), host.device)


def test_nodes_are_ordinary_objects(host):
    class Tagged(Node):
        def __init__(self, *args, tag="", **kw):
            super().__init__(*args, **kw)
            self.tag = tag

        def layout(self):
            return Layout(2, 2)

    leaf = host.leaf(4)
    node = Node("RELU", Layout(4), F32, [leaf], {"a": 1})
    node.note = "kept"
    assert weakref.ref(node)() is node and node.note == "kept" and vars(node) == {"note": "kept"}
    with pytest.raises(AttributeError):
        del node.srcs
    tagged = Tagged("RELU", Layout(4), F32, [leaf], tag="t")
    assert isinstance(tagged, Node) and tagged.tag == "t" and tagged in {tagged} and tagged != node
    assert evaluate(tagged, host.device).numel == 4  # by the Python form: node.numel() is the node's own
    for copied in (copy.copy(node), copy.copy(tagged)):
        assert copied.srcs[0] is leaf and copied.op_type == "RELU"
    assert copy.copy(node).note == "kept" and copy.copy(tagged).tag == "t" and type(copy.copy(tagged)) is Tagged
    # a graph without results goes through deepcopy and pickle, shared nodes shared
    shared = Node("RELU", Layout(4), F32, [Node.leaf(Layout(4), F32)])
    add = Node("ADD", Layout(4), F32, [shared, shared], {"axis": 0})
    add.note = 5
    for proto in range(pickle.HIGHEST_PROTOCOL + 1):
        for again in (copy.deepcopy(add), pickle.loads(pickle.dumps(add, proto))):
            assert again is not add and again.srcs[0] is again.srcs[1] and again.srcs[0] is not shared
            assert (again.layout(), again.attrs(), again.note, again.bufs) == (Layout(4), {"axis": 0}, 5, None)
    ref = weakref.ref(add)
    del add
    assert ref() is None


def test_layouts_are_copied_and_pickled():
    for layout in (Layout(), Layout(3), Layout(2, 3, strides=[1, 2], base_offset=7), Layout((4, 5))):
        for proto in range(pickle.HIGHEST_PROTOCOL + 1):
            for again in (copy.copy(layout), copy.deepcopy(layout), pickle.loads(pickle.dumps(layout, proto))):
                assert again == layout and hash(again) == hash(layout) and again.is_contiguous() == layout.is_contiguous()
        assert weakref.ref(layout)() is layout


def test_buffers_are_ordinary_objects(host):
    buf = host.leaf(4).bufs[0]
    buf.name = "b"
    again = copy.copy(buf)
    assert again.name == "b" and again.storage is buf.storage and weakref.ref(buf)() is buf
    buf.numel = buf.offset_elems = 2
    assert buf.to_numpy().shape == (2,) and buf.data_ptr().value == again.data_ptr().value + 8
    buf.storage = host.leaf(8).bufs[0].storage
    with pytest.raises(TypeError):
        buf.storage = 3
    # a device that keeps buffers of its own: both go when the last outside reference does
    dev = Device()
    dev.cache = AnyBuffer.create(F32, dev, 4)
    gone = weakref.ref(dev)
    del dev
    gc.collect()
    assert gone() is None


def test_the_dtype_of_indices_is_the_nodes(host):
    # as in the Python forms: a leaf declared float32 over int32 ids is what the library is told
    logits, ids = host.leaf(3, 5), host.leaf(3, dtype=R.I32)
    evaluate(Node("CROSS_ENTROPY_IDS", Layout(1), F32, [logits, Node.leaf(Layout(3), F32, ids.bufs[0])]), host.device)
    evaluate(Node("CROSS_ENTROPY_IDS", Layout(1), F32, [logits, ids]), host.device)
    assert host.log() == ["ce_ids 3.000000 5.000000 dtype 0", "ce_ids 3.000000 5.000000 dtype 3"]


@pytest.mark.parametrize("first", ["runtime", "_lib", "Node", "load"])
def test_the_package_alone_gives_its_modules_and_names(first):
    code = (f"import mograd_amd as m; m.{first}; m.runtime.Node is m.Node or 1 / 0; m._lib.load is m.load or 1 / 0\n"
            "try:\n    m.no_such_name\nexcept AttributeError:\n    pass\nelse:\n    1 / 0")
    subprocess.run([sys.executable, "-c", code], check=True, cwd=ROOT)


@pytest.mark.parametrize("op", ["RELU", "ADD", "CROSS_ENTROPY_IDS", "CROSS_ENTROPY_IDS_GRAD", "LINEAR_GRAD"])
def test_a_replaced_rule_is_the_one_that_runs(host, monkeypatch, op):
    seen, own = [], R.SCHEDULER_RULES[op]

    def traced(node, inputs, device):
        seen.append(node.op_type)
        return own(node, inputs, device)

    def graph():
        logits, ids, leaf = host.leaf(3, 5), host.leaf(3, dtype=R.I32), host.leaf(4)
        lin, (_, dw, _) = linear_grad(host)
        return [Node("RELU", Layout(4), F32, [Node("ADD", Layout(4), F32, [leaf, leaf])]), dw,
                Node("CROSS_ENTROPY_IDS", Layout(1), F32, [logits, ids]),
                Node("CROSS_ENTROPY_IDS_GRAD", Layout(3, 5), F32, [logits, ids, host.leaf(1)])]

    rules = dict(R.SCHEDULER_RULES)
    monkeypatch.setattr(R, "SCHEDULER_RULES", rules)
    rules[op] = traced
    evaluate_many(graph(), host.device)
    assert seen == [op]
    del rules[op]
    with pytest.raises(R.MogradError, match=f"no scheduler rule for op {op}"):
        evaluate_many(graph(), host.device)


def test_a_replaced_run_is_the_one_that_runs(host, monkeypatch):
    seen, own = [], R.run
    monkeypatch.setattr(R, "run", lambda node, inputs, device: (seen.append(node.op_type), own(node, inputs, device))[1])
    evaluate(Node("RELU", Layout(4), F32, [host.leaf(4)]), host.device)
    assert seen == ["RELU"]


def test_rewrite_rules_belong_to_the_caller(host):
    def flat(rules):
        pats = [r.pat for r in rules]
        for p in pats:
            pats.extend(p.srcs)
        return list(rules) + pats

    first, second = GPU_REWRITES(), GPU_REWRITES()
    assert first == second and [r.name for r in first] == [r.func.__name__ for r in first]
    assert not {id(o) for o in flat(first)} & {id(o) for o in flat(second)}
    for rule in first:
        rule.func = lambda node, sim: None
        rule.pat.op_type = "NO_SUCH_OP"
    first[1].pat.srcs.clear()
    assert GPU_REWRITES() == second
    mm = Node("MATMUL_BIAS_BT", Layout(2, 3), F32, [host.leaf(2, 4), host.leaf(3, 4), host.leaf(3)])
    assert Simplifier(GPU_REWRITES()).run(Node("RELU", Layout(2, 3), F32, [mm])).op_type == "MATMUL_BIAS_RELU_BT"


def test_cycles_are_errors(host):
    a = Node("RELU", Layout(4), F32, [host.leaf(4)])
    b = Node("RELU", Layout(4), F32, [a])
    a.srcs[0] = b
    with pytest.raises(R.MogradError, match="cycle"):
        evaluate(b, host.device)
    flip = [Rule(Pat(x), lambda node, sim, y=y: Node(y, node.layout(), node.dtype(), node.srcs)) for x, y in ("AB", "BA")]
    with pytest.raises(R.MogradError, match="cycled"):
        Simplifier(flip).run(Node("A", Layout(4), F32, [host.leaf(4)]))
    a.srcs.clear()


def test_a_walk_keeps_its_places_when_an_attribute_lookup_walks_too(host):
    # A key with the hash of "index" that compares by Python code evaluates another graph over the same
    # nodes while the outer walk looks its attributes up.
    lin, (_, dw, _) = linear_grad(host)
    del _, lin
    evaluate(dw, host.device)  # without dX
    lin = dw.src(0)

    class Key:
        def __hash__(self):
            return hash("index")

        def __eq__(self, other):
            evaluate_many([Node("RELU", Layout(4), F32, [host.leaf(4)]), dw], host.device)
            return False

    get = Node("GETTUPLE", Layout(3, 4), F32, [lin], {Key(): 0, "index": 1})
    got = evaluate_many([get, lin], host.device)
    assert got[0] is dw.bufs[0] and got[1].to_numpy()[0] == 1.0


def structure(roots):
    """What a graph is, whatever its nodes: each node's op, layout, dtype, attributes and sources by place."""
    order, place = [], {}
    for node in R._toposort(Node("SINK", Layout(1), F32, [r for r in roots if r is not None])):
        place[node] = len(order)
        order.append((node.op_type, node.layout().dims, node.layout().strides, node.layout().base_offset, node.dtype(),
                      node.attrs(), type(node.srcs), [place[s] for s in node.srcs]))
    return order, [None if r is None else place[r] for r in roots]


def classifier(host, srcs=list, extra=None):
    params = [host.leaf(4, 6), host.leaf(4), host.leaf(4), host.leaf(4), host.leaf(3, 4), host.leaf(3)]
    w1, b1, gam, bet, w2, b2 = params
    x = Node("RESHAPE", Layout(5, 6), F32, srcs([host.leaf(30)]))
    h = Node("RELU", Layout(5, 4), F32, srcs([Node("MATMUL_BIAS_BT", Layout(5, 4), F32, srcs([x, w1, b1]))]))
    ln = Node("LAYER_NORM_STATS", Layout(5, 4), F32, srcs([h, gam, bet]), {"eps": 1e-5})
    y = Node("GETTUPLE", Layout(5, 4), F32, srcs([ln]), {"index": 0, **(extra or {})})
    h2 = Node("ADD", Layout(5, 4), F32, srcs([Node("MATMUL_BT", Layout(5, 4), F32, srcs([y, host.leaf(4, 4)])), h]))
    logits = Node("MATMUL_BIAS_BT", Layout(5, 3), F32, srcs([h2, w2, b2]))
    loss = Node("CROSS_ENTROPY_IDS", Layout(1), F32, srcs([logits, host.leaf(5, dtype=R.I32)]))
    return loss, params + [x, host.leaf(2)]


def transformer(host, **_):
    from mograd_amd.tiny_transformer import TinyTransformer

    for name in ("mg_fill", "mg_deferred_create"):
        setattr(host.device.lib, name, lambda *args: 0)  # (the stub has neither)
    model = TinyTransformer(host.device, 11, 16, 32, 2, 2, compute_dtype=F32)
    ids, labels = (AnyBuffer.from_numpy(host.device, np.zeros(6, np.int32)) for _ in range(2))
    loss, leaves = model.graph(ids, labels, 2, 3)
    return loss, list(leaves.values())


@pytest.mark.parametrize("build", [
    classifier, transformer,
    lambda host: classifier(host, srcs=tuple),
    lambda host: classifier(host, extra={"note": [1, 2]}),  # an attribute that only the Python rules look at
    lambda host: classifier(host, extra={"index": np.int64(0)}),
], ids=["classifier", "transformer", "tuples", "unusual", "numpy"])
def test_native_rules_are_the_python_ones(host, monkeypatch, build):
    def once(table, rules):
        monkeypatch.setattr(R, "GRAD_RULES", table)
        loss, targets = build(host)
        grads = R.gradient(loss, host.leaf(1), targets)
        plain = structure([loss] + grads)
        sim = Simplifier(rules)
        new = sim.run_many([loss] + [g for g in grads if g is not None])
        return plain, structure(new), sorted(sim.uses.values())

    table = dict(R.GRAD_RULES)
    own = once(table, GPU_REWRITES())
    calls = collections.Counter()

    def counted(f):  # another function, which the native walk does not know
        return lambda *args: (calls.update([f.__name__]), f(*args))[1]

    python = once({op: counted(f) for op, f in table.items()}, [Rule(r.pat, counted(r.func), r.name) for r in GPU_REWRITES()])
    assert own == python and calls["linear_grad"] and calls["fuse_matmul_add"]


def test_a_replaced_gradient_rule_is_the_one_that_runs(host, monkeypatch):
    x, w = host.leaf(4, 8), host.leaf(3, 8)
    y = Node("MATMUL_BT", Layout(4, 3), F32, [x, w])
    mark = host.leaf(4, 8)
    monkeypatch.setitem(R.GRAD_RULES, "MATMUL_BT", lambda node, upstream: (mark,))  # shorter than the sources
    assert R.gradient(y, host.leaf(4, 3), [x, w]) == [mark, None]

    class Mine(Simplifier):
        def single_use(self, node):
            return False

    relu = Node("RELU", Layout(4, 3), F32, [Node("MATMUL_BIAS_BT", Layout(4, 3), F32, [x, w, host.leaf(3)])])
    assert Mine(GPU_REWRITES()).run(relu) is relu
    sim = Simplifier(GPU_REWRITES())
    sim.single_use = lambda node: False
    assert sim.run(relu) is relu


@pytest.mark.parametrize("method", ["single_use", "replace", "consumers_of", "resolve"])
def test_a_method_replaced_on_the_class_is_the_one_that_runs(host, monkeypatch, method):
    def rewritten():
        loss, targets = transformer(host)
        grads = R.gradient(loss, host.leaf(1), targets)
        return structure(Simplifier(GPU_REWRITES()).run_many([loss] + [g for g in grads if g is not None]))

    own, calls, was = rewritten(), [], getattr(Simplifier, method)
    with monkeypatch.context() as m:
        m.setattr(Simplifier, method, lambda *args: (calls.append(args), was(*args))[1])
        assert rewritten() == own and calls
        if method == "single_use":
            m.setattr(Simplifier, method, lambda self, node: False)
            relu = Node("RELU", Layout(4, 3), F32, [Node("MATMUL_BIAS_BT", Layout(4, 3), F32, [host.leaf(4, 8), host.leaf(3, 8), host.leaf(3)])])
            assert Simplifier(GPU_REWRITES()).run(relu) is relu
    assert rewritten() == own
