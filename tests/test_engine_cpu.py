"""Host side of the engine (batching, cache manager, step function) on a CPU, with the kernels'
plain PyTorch references standing in for the kernels, against the plain whole-sequence model."""
import pytest
import torch

from helpers import PAGE_SIZE, Harness, make_folder, random_tokens
from plain_qwen2 import qwen2_logits, read_model_folder
from torch_ops import TorchOps


@pytest.mark.parametrize("name", ["A", "B", "C"])
def test_whole_then_decode_matches_plain(tmp_path, name):
    folder = make_folder(tmp_path, name)
    config, weights = read_model_folder(folder)
    tokens = random_tokens(config["vocab_size"], 45, seed=7)
    expected = qwen2_logits(config, weights, tokens)
    h = Harness(folder, TorchOps(), torch.float32, "cpu", PAGE_SIZE[name], num_pages=32)
    split = 30
    got = [h.feed([("a", tokens[:split], list(range(split)))])]
    for i in range(split, len(tokens)):
        got.append(h.feed([("a", [tokens[i]], [0])]))
    got = torch.cat(got)
    torch.testing.assert_close(got, expected, rtol=1e-4, atol=1e-5)
    h.feed([], end=["a"]) if False else h.cache.free_sequence(h.live.pop("a")[0])
    h.cache.assert_consistent([])


def test_mixed_batch_with_page_reuse(tmp_path):
    name = "B"
    folder = make_folder(tmp_path, name)
    config, weights = read_model_folder(folder)
    prompts = {rid: random_tokens(config["vocab_size"], n, seed=i) for i, (rid, n) in enumerate([("a", 23), ("b", 17), ("c", 9), ("d", 31)])}
    expected = {rid: qwen2_logits(config, weights, toks) for rid, toks in prompts.items()}
    h = Harness(folder, TorchOps(), torch.float32, "cpu", PAGE_SIZE[name], num_pages=9)  # 8 usable pages of 8
    got = {rid: [] for rid in prompts}
    # a and b start; a finishes, its pages go to c; then d takes what b and c give back
    def run(batch, end=()):
        out = h.feed([(rid, prompts[rid][lo:hi], list(range(hi - lo))) for rid, lo, hi in batch], end=end)
        row = 0
        for rid, lo, hi in batch:
            got[rid].append(out[row:row + hi - lo])
            row += hi - lo
    run([("a", 0, 7), ("b", 0, 2)])
    run([("a", 7, 8), ("b", 2, 11)])
    run([("a", 8, 23), ("b", 11, 12)], end=["a"])
    run([("b", 12, 13), ("c", 0, 9)], end=["c"])
    run([("b", 13, 17), ("d", 0, 5)], end=["b"])
    run([("d", 5, 31)], end=["d"])
    for rid in prompts:
        torch.testing.assert_close(torch.cat(got[rid]), expected[rid], rtol=1e-4, atol=1e-5)
    h.cache.assert_consistent([])
    assert h.cache.num_used_pages() == 0


def test_a_step_padded_up_to_a_timed_number_of_rows_keeps_its_logits(tmp_path):
    """A step of portions a little short of a row count the matrix library was timed for gets rows of a sequence on the
    null page: with every slot but one decoding beside the portions (the padding is then one sequence more than
    ``max_num_seqs``), the logits are those of the same step unpadded, and the null page is all the padding wrote to."""
    name = "B"
    folder = make_folder(tmp_path, name)
    config, weights = read_model_folder(folder)
    prompts = {rid: random_tokens(config["vocab_size"], n, seed=50 + i) for i, (rid, n) in enumerate([("a", 12), ("b", 9), ("c", 15), ("d", 40)])}

    def run(tuned):
        h = Harness(folder, TorchOps(), torch.float32, "cpu", PAGE_SIZE[name], num_pages=32, max_num_seqs=4, max_num_tokens=64)
        h.runner.tuned_row_counts = tuned
        for rid in "abc":  # three of the four slots decode
            h.feed([(rid, prompts[rid][:-1], [])])
        batch = [(rid, prompts[rid][-1:], [0]) for rid in "abc"] + [("d", prompts["d"], [0, 39])]
        out = h.feed(batch)
        return h, out

    plain, want = run([])
    padded, got = run([48])  # 43 rows -> 48: five rows more, within the 12% that a step may grow by
    assert padded.runner.num_padded_steps == 1 and plain.runner.num_padded_steps == 0
    torch.testing.assert_close(got, want, rtol=0, atol=0)
    torch.testing.assert_close(got[-1], qwen2_logits(config, weights, prompts["d"])[-1], rtol=1e-4, atol=1e-5)
    for mine, theirs in zip(padded.cache.groups, plain.cache.groups):
        for name in mine.tensors:
            assert torch.equal(mine.tensors[name][:, 1:], theirs.tensors[name][:, 1:])  # everything but the null page


def test_a_fixed_workspace_refuses_to_replace_a_buffer():
    import pytest
    import torch

    from velox_amd.engine.batch import Workspace, WorkspaceError

    workspace = Workspace(torch.device("cpu"))
    first = workspace.get("a", 10)
    assert workspace.get("a", 4).data_ptr() == first.data_ptr()
    grown = workspace.get("a", 100)  # not fixed: grows on demand
    assert grown.numel() == 100
    workspace.reserve("b", 50)
    workspace.fix()
    assert workspace.get("a", 100).data_ptr() == grown.data_ptr()
    assert workspace.get("b", 50).numel() == 50
    with pytest.raises(WorkspaceError, match="'a'"):
        workspace.get("a", 101)
    with pytest.raises(WorkspaceError, match="nothing"):
        workspace.get("c", 1)


def test_without_a_gpu_the_engine_refuses_loudly(tmp_path, monkeypatch):
    """No CPU path stands behind the kernels: asking for the product's operations without a GPU, or on the CPU, is one
    clear error, also through the Python entry point; so is a box without the compiler and without built libraries."""
    from velox_amd import Engine, EngineConfig
    from velox_amd.kernels import KernelError, build, load_ops

    with pytest.raises(KernelError, match="no CPU path"):
        load_ops("cpu")
    if not torch.cuda.is_available():
        with pytest.raises(KernelError, match="no GPU is visible"):
            load_ops("cuda")
        folder = make_folder(tmp_path, "A")
        with pytest.raises(KernelError, match="no GPU is visible"):
            Engine.from_pretrained(EngineConfig(model=folder, dtype="bfloat16"))
    monkeypatch.setenv("HIPCC", str(tmp_path / "no_such_compiler"))
    monkeypatch.setenv("PATH", str(tmp_path))
    real_isfile = build.os.path.isfile
    monkeypatch.setattr(build.os.path, "isfile", lambda path: False if str(path).endswith("hipcc") else real_isfile(path))
    with pytest.raises(build.BuildError, match="hipcc not found"):
        build.find_hipcc()


def rules_of_the_kernels(num_cus: int = 256):
    """The rules by which calls take one kernel or another, without a GPU."""
    from velox_amd.kernels.hip_ops import HipOps

    ops = HipOps.__new__(HipOps)
    ops.num_cus, ops.use_skinny_gemm, ops.fuse_residual_norm = num_cus, True, True
    return ops


def an_output_product(heads, kv_heads, dim, width):
    """A mixer whose output weight is prepared, the handle of that weight, and a sink for its product."""
    from velox_amd.kernels.hip_ops import PreparedWeight
    from velox_amd.parts.attention import AttentionMixer
    from velox_amd.parts.base import ResidualSink
    from velox_amd.parts.norms import RMSNorm

    mixer = AttentionMixer("", width, heads, kv_heads, dim)
    mixer.o_weight = torch.zeros((width, heads * dim), dtype=torch.bfloat16)
    weight = mixer._prepared["o_weight"] = PreparedWeight(mixer.o_weight)
    weight.copies[1] = torch.zeros(0)
    norm = RMSNorm("", width, 1e-5)
    norm.weight = torch.ones(width)
    return mixer, weight, ResidualSink(torch.zeros(1, width), norm)


@pytest.mark.parametrize("heads,kv_heads,dim,width,page,taken", [
    (12, 2, 128, 1536, 16, True), (12, 2, 128, 1536, 4, True), (16, 1, 64, 1024, 4, True),
    (12, 2, 128, 1536, 2, False), (12, 2, 128, 1536, 1, False),  # fewer than four keys a page
    (32, 1, 64, 2048, 16, False), (20, 1, 128, 2560, 16, False), (40, 2, 64, 2560, 16, False),  # more heads per KV head than a tile has rows
])
def test_an_attention_is_left_in_parts_only_by_the_kernel_that_leaves_them(heads, kv_heads, dim, width, page, taken):
    """Captured bounds and steps alike: what the streaming kernel does not take is merged by the attention itself."""
    ops = rules_of_the_kernels()
    mixer, weight, sink = an_output_product(heads, kv_heads, dim, width)
    assert (ops.attention_parts(1, heads, kv_heads, dim, weight, sink, 391, page) > 0) == taken
    assert (ops.attention_parts_keys in mixer.capture_key_bounds_of_pages(ops, 1, 32768, page)) == taken


@pytest.mark.parametrize("sequences,kv_heads,shared", [(64, 4, True), (128, 8, True), (129, 8, False), (1024, 4, False), (1024, 1, False),
                                                       (1, 16, False), (2, 8, False), (4, 4, False), (16, 1, False), (1, 32, True), (8, 4, True), (32, 1, True)])
def test_keys_are_shared_out_among_enough_sequences_that_are_soon_looked_through(sequences, kv_heads, shared):
    assert rules_of_the_kernels().shares_keys(sequences, kv_heads) == shared


@pytest.mark.parametrize("tokens,heads,kv_heads,width,parts", [
    (1, 12, 2, 1536, (0, 2, 4, 4, 8, 0)), (1, 16, 4, 3584, (0, 2, 4, 4, 8, 0)),  # a piece of activations a lane
    (2, 12, 2, 1536, (0, 2, 4, 4, 8, 0)), (1, 24, 4, 2048, (0, 2, 4, 4, 8, 0)),  # two
    (1, 28, 4, 3584, (0,) * 6), (1, 20, 4, 2560, (0,) * 6),  # two in more workgroups than there are compute units
    (4, 12, 2, 1536, (0,) * 6), (5, 12, 2, 1536, (0,) * 6),
])
def test_in_how_many_parts_an_attention_is_left(tokens, heads, kv_heads, width, parts):
    _, weight, sink = an_output_product(heads, kv_heads, 128, width)
    ops = rules_of_the_kernels()
    assert tuple(ops.attention_parts(tokens, heads, kv_heads, 128, weight, sink, keys) for keys in (64, 128, 384, 385, 1025, 2049)) == parts


@pytest.mark.parametrize("page,keys,rows", [(16, 1 << 20, 3364), (4, 1 << 20, 12964), (2, 1 << 20, 12964), (64, 1 << 20, 1600), (16, 1 << 17, 1600)])
def test_scratch_for_shares_of_keys_is_that_of_the_caches_pages(page, keys, rows):
    """100 single tokens of 28 heads over 4: workgroups per KV head that share out the step's keys, as many as hold the page ids of so many keys, or
    what the splits of portions take."""
    assert rules_of_the_kernels().attention_scratch_elems(28, 4, 128, 100, 100, keys, block_size=page) == (rows * 28 * 128, rows * 28)


@pytest.mark.parametrize("rows,outputs,streamed", [(17, 16384, True), (17, 16383, False), (32, 18000, True), (32, 152064, True), (33, 16384, True), (33, 18000, False),
                                                   (64, 22000, False), (64, 24576, True), (64, 32000, True), (33, 34000, False), (48, 65536, True), (33, 152064, False)])
def test_heads_of_some_rows_that_fill_whole_rounds_of_workgroups_are_streamed(rows, outputs, streamed):
    assert rules_of_the_kernels().streams_head(rows, outputs) == streamed


def test_no_garbage_is_collected_while_a_step_is_captured(monkeypatch):
    """A collector that runs in the middle of a capture may give back what an engine that is gone had captured, which ends the process.  (Stand-ins
    for the GPU's calls: what is asked is only when the collector is held.)"""
    import contextlib
    import gc
    import threading

    from velox_amd.engine import runner as module

    class Anything:
        def __getattr__(self, name):
            return lambda *args, **more: None

    for name in ("Stream", "CUDAGraph"):
        monkeypatch.setattr(torch.cuda, name, lambda **more: Anything())
    for name in ("stream", "graph"):
        monkeypatch.setattr(torch.cuda, name, lambda *args, **more: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "current_stream", Anything)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    seen, runner = [], module.ModelRunner.__new__(module.ModelRunner)
    runner.ops, runner.device, runner._graph_pool = object(), torch.device("cpu"), None
    runner._forward = lambda ctx: seen.append(gc.isenabled())
    assert gc.isenabled()
    runner._capture(None, 2)
    assert seen == [True, True, False] and gc.isenabled()
    inside, leave = threading.Event(), threading.Event()

    def other():
        with module.collection_held():
            inside.set()
            leave.wait(10)

    thread = threading.Thread(target=other)
    with pytest.raises(ValueError), module.collection_held():
        thread.start()
        assert inside.wait(10) and not gc.isenabled()
        raise ValueError
    assert not gc.isenabled()  # (the other thread is still capturing)
    leave.set()
    thread.join()
    assert gc.isenabled()
    gc.disable()
    try:
        with module.collection_held():
            pass
        assert not gc.isenabled()  # (a program that holds it itself goes on doing so)
    finally:
        gc.enable()
