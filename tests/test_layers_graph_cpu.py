"""The layer-graph front end without a GPU: dimensions, the reference's asserts, and the byte-arena
layout.  The arena sizes are the ones the reference's generated module allocates for its own test
graphs with 24 blocks per grid (`cp.empty(N, dtype=cp.uint8)` at ml/layers.py:4736-4737, 5194-5195,
5548-5549, 6085-6086, 6640-6641: workspace, then weights; the adjoint arena is empty)."""
import pytest
import torch

from ml import layers as L


@pytest.fixture(autouse=True)
def blocks_24():
    L.set_blocks_per_grid(24)
    yield
    L.set_blocks_per_grid(24)


def sizes(graph):
    return [p["size"] for p in L.pass_calculate_partitions(graph, {})]


def tanh_mlp(k):
    return L.pipe(L.input("input", (24, 1, k)), L.matmul((k, 4)), L.tanh, L.matmul((4, 4)), L.tanh, L.matmul((4, 2)),
                  L.tanh)


def graph_of_test3():
    return L.pipe(L.input("input", (24, 64, 64)), L.matmul((64, 64)), L.ln_l2, L.relu, L.matmul((64, 64)), L.ln_l2,
                  L.relu, L.matmul((64, 64)), L.softmax_and_discrete_sample)


def ensemble_graph(e, deep, size=None):
    out = L.pair(L.apply("ensemble", L.input("output_probs", (e, 24, 64, 64))),
                 L.apply("ensemble", L.input("output_indices", (e, 24, 64), "int")))
    x = L.pipe(L.input("input", (24, 64, 64)), L.matmul_ensemble((e, 64, 64)))
    if deep:
        x = L.pipe(x, L.ln_l2, L.relu, L.matmul_ensemble((e, 64, 64)), L.ln_l2, L.relu, L.matmul_ensemble((e, 64, 64)))
    return L.softmax_and_discrete_sample_(out, x) if size is None else \
        L.masked_softmax_and_discrete_sample_(size, out, x)


def test_arena_sizes_match_the_reference():
    assert sizes(tanh_mlp(4)) == [160, 2304, 0]                    # layers test1
    assert sizes(tanh_mlp(2)) == [128, 2112, 0]                    # layers test2
    assert sizes(graph_of_test3()) == [49152, 3545088, 0]             # layers test3
    assert sizes(ensemble_graph(16, True)) == [786432, 9535488, 0]  # layers test4
    assert sizes(ensemble_graph(4, False, 11)) == [65536, 2383872, 0]  # layers test5


def test_offsets_are_depth_first_and_16_byte_aligned():
    g = L.pipe(L.input("input", (24, 1, 3)), L.matmul((3, 5)), L.tanh)     # 12- and 20-byte rows: padding appears
    parts = L.pass_calculate_partitions(g, {})
    ws = sorted((o.offset, o.spec.dim) for o in parts[L.workspace_id()]["partition"].values())
    assert [d for _, d in ws] == [(24, 1, 3), (24, 1, 5), (24, 1, 5)]
    assert [o for o, _ in ws] == [0, 288, 288 + 480]
    assert all(o % 16 == 0 for o, _ in ws)
    g2 = L.pipe(L.input("input", (24, 1, 1)), L.matmul((1, 1)), L.matmul((1, 1)))
    parts = L.pass_calculate_partitions(g2, {})
    assert sorted(o.offset for o in parts[L.weight_id()]["partition"].values()) == [0, 16]   # 4-byte weights, 16 apart
    assert parts[L.weight_id()]["size"] == 20                                            # the end is not padded


def test_dimension_asserts_are_the_reference_ones():
    with pytest.raises(AssertionError, match="batch dimension in the matmul node"):
        L.get_dim({}, L.pipe(L.input("input", (7, 4, 4)), L.matmul((4, 4))))
    with pytest.raises(AssertionError, match="inner dimensions of the matrix multiplication"):
        L.get_dim({}, L.BlockMatmul(L.input("input", (24, 4, 4)), L.weight((8, 5))))
    with pytest.raises(AssertionError, match="dimensions of the first output"):
        L.get_dim_pair({}, L.softmax_and_discrete_sample_(
            L.pair(L.input_((24, 4, 8)), L.input_((24, 4), "int")), L.input("input", (24, 4, 4))))
    d = L.get_dim_pair({}, graph_of_test3())
    assert d[0].dim == (24, 64, 64) and d[1].dim == (24, 64) and d[1].dtype == torch.int32
    assert L.get_dim({}, L.argmax(L.input("x", (24, 8, 12)))).dim == (24, 8)
    assert L.get_dim({}, L.binarize(7, L.input("x", (24, 8, 12)))).dim == (24, 8)


def test_extract_and_model_ptrs_on_host_memory():
    g = ensemble_graph(4, False, 11)
    m = L.create_model(g, device="cpu")
    for x in m.data:
        x["array"].zero_()
    w = L.key_extract(m, "weights")
    assert w.shape == (4, 64, 64) and w.dtype == torch.float32
    w[2, 1, 3] = 5.0
    probs, idx = L.graph_extract(m, {"ensemble": 3})
    assert probs.shape == (24, 64, 64) and idx.shape == (24, 64) and idx.dtype == torch.int32
    idx[0, 0] = 77
    assert L.key_extract(m, "output_indices")[3, 0, 0] == 77
    with pytest.raises(KeyError, match="missing .scalar. key"):
        L.graph_extract(m, {})
    with pytest.raises(KeyError, match="Cannot find the input tensor"):
        L.key_extract(m, "nothing")
    # the same arenas seen through a second model built around the pointers
    m2 = L.model_ptrs_to_model(g, L.model_to_model_ptrs(m))
    assert L.key_extract(m2, "weights")[2, 1, 3] == 5.0
    with pytest.raises(AssertionError, match="length of the partition"):
        L.model_ptrs_to_model(g, tuple(torch.empty(8, dtype=torch.uint8) for _ in range(3)))
    assert [sid for sid, _, _ in L.extract_layers(m)] == [1, 0, 1, 1]
    L.set_random_seed(1, device="cpu")
    L.pass_init(m)
    w = L.key_extract(m, "weights")
    assert abs(float(w.std()) - 0.1) < 0.01 and L.key_extract(m, "input").abs().sum() == 0


def test_printing_uses_the_golden_text_format():
    m = L.create_model(tanh_mlp(4), device="cpu")
    for x in m.data:
        x["array"].zero_()
    lines = []
    L.print_weights(m, lines.append)
    # the first three lines of the reference's layers/test1/layers.txt after "---"
    row = "[0.000000; 0.000000; 0.000000; 0.000000]"
    assert lines == ["[" + "; ".join([row] * 4) + "]"] * 2 + ["[" + "; ".join([row] * 2) + "]"]


def test_fused_plan_takes_only_the_shapes_the_fused_kernel_runs():
    """A 16-bit relu stack with a sampling head is planned as one fused launch only for the widths the fused
    kernel accepts (input a multiple of 16, hidden widths multiples of 32, nothing above 256, head <= 64)."""
    def stack(dims, dtype="f16"):
        x = L.input("input", (24, 16, dims[0]), dtype)
        for i, (k, n) in enumerate(zip(dims[:-1], dims[1:])):
            x = L.matmul((k, n), x)
            if i + 2 < len(dims):
                x = L.relu(x)
        return L.create_model(L.masked_softmax_and_discrete_sample(3, x), device="cpu")

    assert L._fused_plan(stack([32, 256, 256, 64])) is not None
    assert L._fused_plan(stack([32, 64, 3 * 32, 16])) is not None
    assert L._fused_plan(stack([32, 48, 16])) is None          # hidden width not a multiple of 32
    assert L._fused_plan(stack([32, 256, 128])) is None        # head wider than 64
    assert L._fused_plan(stack([24, 256, 64])) is None         # input width not a multiple of 16
    assert L._fused_plan(stack([32, 512, 64])) is None         # wider than 256
    assert L._fused_plan(stack([32, 256, 64], "float")) is None   # f32 graphs run node by node


def test_ensemble_with_adjoint_places_the_dual_in_the_adjoint_arena():
    """`matmul_ensemble_with_adjoint` (ml/layers.spi:472-479): weights (E, out, in) in the weights arena, their dual
    ((out, in), E) in the third arena, both reachable under "cem_weight_layer_dual", the product as matmul_ensemble's."""
    e, k, n = 4, 32, 64
    x = L.pipe(L.input("input", (24, 64, k)), L.matmul_ensemble_with_adjoint((e, k, n)))
    g = L.softmax_and_discrete_sample(x)
    plain = L.softmax_and_discrete_sample(L.pipe(L.input("input", (24, 64, k)), L.matmul_ensemble((e, k, n))))
    assert sizes(g) == sizes(plain)[:2] + [n * k * e * 4]
    m = L.create_model(g, device="cpu")
    w, wt = L.key_extract(m, "cem_weight_layer_dual")
    assert tuple(w.shape) == (e, n, k) and tuple(wt.shape) == (n, k, e)
    assert w.data_ptr() == L.key_extract(m, "weights").data_ptr()
    assert wt.data_ptr() == L.model_to_model_ptrs(m)[L.weight_adjoint_id()].data_ptr()
    assert L.get_dim({}, x).dim == (24, 64, n)


def test_stack_plan_takes_whole_chains_only():
    """The graphs that run as one launch of the f32 stack kernel: a chain whose inner nodes nobody can look at."""
    plan = lambda g, key=None: L._stack_plan(L.Model(g, {}, []), key)
    x, ws, acts, head, mask, outs, middle = plan(graph_of_test3())
    assert len(ws) == 3 and head == "softmax" and mask == 0 and outs is None and acts[0] == acts[1] != 0 and acts[2] == 0 and len(middle) == 7
    assert plan(ensemble_graph(4, True), "ensemble")[5] is not None and plan(ensemble_graph(4, True)) is None
    inp = lambda: L.input("input", (24, 64, 64))
    named = L.pipe(L.key_graph("hidden", L.pipe(inp(), L.matmul((64, 64)))), L.relu, L.matmul((64, 64)), L.softmax_and_discrete_sample)
    kept = L.pipe(L.copy_(L.input("kept", (24, 64, 64)), L.pipe(inp(), L.matmul((64, 64)))), L.matmul((64, 64)), L.softmax_and_discrete_sample)
    swapped = L.pipe(inp(), L.matmul((64, 64)), L.relu, L.ln_l2, L.matmul((64, 64)), L.softmax_and_discrete_sample)   # norm behind the map
    first = L.pipe(inp(), L.relu, L.matmul((64, 64)), L.softmax_and_discrete_sample)                                    # a map of the input
    assert [plan(g) for g in (named, kept, swapped, first)] == [None] * 4


class Answering:
    """Stands in for the library: sizes are answered by the real one or with a code, launches are recorded."""

    def __init__(self, takes=None, launch=0):
        self.takes, self.launch, self.calls = takes, launch, []

    def sp_stack_forward_takes(self, *args):
        return L._lib.lib.sp_stack_forward_takes(*args) if self.takes is None else self.takes

    def sp_stack_forward_f32(self, *args):
        self.calls.append(args)
        return self.launch


def without_a_gpu(monkeypatch, lib):
    monkeypatch.setattr(L, "lib", lib)
    monkeypatch.setattr(L, "ptr", lambda t, dtype=None, name="": None if t is None else t.data_ptr())
    monkeypatch.setattr(L, "stream_ptr", lambda: None)
    monkeypatch.setattr(L._lib, "stream_ptr", lambda: None)
    return lib


def test_a_stack_the_entry_point_refuses_runs_node_by_node(monkeypatch):
    """Which sizes run as one launch is sp_stack_forward_takes' answer alone: what it refuses for its size falls back to the
    walk and leaves the generator where it was, errors of a launch are raised."""
    lib = without_a_gpu(monkeypatch, Answering())
    build = lambda *widths: L.create_model(L.softmax_and_discrete_sample(L.pipe(L.input("input", (24, 64, widths[0])), *[
        L.matmul(pair) for pair in zip(widths[:-1], widths[1:])])), device="cpu")
    model, ls = build(64, 64, 16), L.create_layer_state()
    for lib.takes in (-2, -6):
        assert L._run_fused_stack(model, None, 1, ls) is False and ls.draws == 0 and not lib.calls
    lib.takes = 0
    lib.launch = -5
    with pytest.raises(L._lib.SpiralError):
        L._run_fused_stack(model, None, 1, ls)
    lib.takes, lib.launch = None, 0
    assert L._run_fused_stack(model, None, 1, ls) is True and ls.draws > 0
    # the real answers: widths, depth, the LDS
    for widths in ((4, 16, 4), (128, 64), (100, 128, 96, 64), (64,) * 9):
        assert L._run_fused_stack(build(*widths), None, 1, ls) is True, widths
    for widths in ((132, 64, 16), (64, 72, 16), (64, 256, 16), (64, 64, 68), (64,) * 10, (128, 128, 128, 128, 64)):
        assert L._run_fused_stack(build(*widths), None, 1, ls) is False, widths


def test_a_node_somebody_looks_at_is_written(monkeypatch):
    """A fused stack leaves the tensors in its middle out.  Looked up before the run, such a node keeps the model on the walk;
    looked up behind a fused run for the first time, it is computed then, and the recorded launch is not replayed any more."""
    calls, walked = without_a_gpu(monkeypatch, Answering()).calls, []
    monkeypatch.setattr(L, "graph_run", lambda model, ls, indices: walked.append(model.graph))
    hidden = L.pipe(L.input("input", (24, 64, 64)), L.matmul((64, 64)), L.relu)
    build = lambda: L.create_model(L.pipe(hidden, L.matmul((64, 16)), L.softmax), device="cpu")
    run = lambda m: L.graph_run_host(m)
    look = lambda m: L.graph_extract(L.Model(hidden, m.dims, m.data))

    first = build()
    look(first)
    run(first)
    assert walked == [first.graph] and not calls

    then = build()
    run(then)
    assert len(calls) == 1 and len(walked) == 1                 # one launch, nothing computed besides
    L.graph_extract(then)                                       # the result: always written
    L.key_extract(then, "input")
    assert len(walked) == 1
    look(then)
    assert walked[1] is hidden                                  # computed for the first look
    look(then)
    run(then)
    run(then)
    assert len(calls) == 1 and walked[2] is then.graph and hidden not in walked[2:]
    other = build()
    run(other)
    assert len(calls) == 2                                      # another model of the same graph is not concerned
