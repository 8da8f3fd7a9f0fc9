"""A shared expert on the second stream beside the routed experts, in steps of fewer rows than always take it."""
import pytest
import torch

import plain_model
import util
from test_engine_gpu import CONFIG_WIDE, bound

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,rows", [("float32", 17), ("float32", 200), ("bfloat16", 65), ("bfloat16", 200)])
def test_short_steps_on_two_streams(tmp_path, dtype, rows):
    """Steps whose weights are many take the second stream from far fewer rows on: the same products (in 32-bit the same
    bits; the first stream's logits are the plain model's within the usual bound)."""
    import ninfer_amd
    from ninfer_amd import EngineOptions, load_model
    ninfer_amd.write_random_model(str(tmp_path), CONFIG_WIDE, 77, dtype=dtype, std=0.06)
    rcfg, w = util.read_folder(str(tmp_path))
    toks = util.safe_prompt(w, rcfg, rows, 5)
    runner = load_model(str(tmp_path), EngineOptions(dtype=dtype, max_context=704, prefill_chunk=640, num_sequences=2,
                                                   page_size=16))
    ops, got = runner.ops, {}
    try:
        for two in (False, True):
            ops.pays_beside = lambda rows, weight_bytes, dtype: two
            got[two] = util.run_schedule(runner, util.schedule_whole(f"s{two}", toks))[f"s{two}"]
    finally:
        del ops.pays_beside
    assert ops._side is not None and not ops._side_open
    if dtype == "float32":
        assert torch.equal(got[True], got[False])
    torch.testing.assert_close(got[True], plain_model.forward(w, rcfg, toks), **bound(dtype))


def test_one_stream_when_it_is_asked_for(tmp_path, monkeypatch):
    """`beside_min_rows` out of reach is one stream, also where a step's weights are many."""
    import ninfer_amd
    from ninfer_amd import EngineOptions, load_model
    ninfer_amd.write_random_model(str(tmp_path), CONFIG_WIDE, 77, dtype="bfloat16", std=0.06)
    runner = load_model(str(tmp_path), EngineOptions(dtype="bfloat16", max_context=704, prefill_chunk=640, num_sequences=2, page_size=16))
    ops, blocks = runner.ops, []
    inner = ops.beside
    monkeypatch.setattr(ops, "pays_beside", lambda rows, weight_bytes, dtype: True)
    monkeypatch.setattr(ops, "beside", lambda: (blocks.append(1), inner())[1])
    for min_rows, some in ((512, True), (1 << 30, False)):
        monkeypatch.setattr(ops, "beside_min_rows", min_rows)
        blocks.clear()
        util.run_schedule(runner, util.schedule_whole(f"r{min_rows}", list(range(5, 205))))
        assert bool(blocks) == some


@pytest.mark.parametrize("dtype,batch,kept", [("float32", 40, False), ("bfloat16", 4, False), ("bfloat16", 40, True)])
def test_streams_without_the_librarys_products_keep_no_workspace(tmp_path, monkeypatch, dtype, batch, kept):
    """A graph of few rows or in 32-bit, and the second stream of a 32-bit engine, hold no product of the library's."""
    import ninfer_amd
    from ninfer_amd import Chunk, EngineOptions, load_model
    ninfer_amd.write_random_model(str(tmp_path), CONFIG_WIDE, 78, dtype=dtype, std=0.06)
    runner = load_model(str(tmp_path), EngineOptions(dtype=dtype, max_context=704, prefill_chunk=640, num_sequences=48, page_size=16,
                                                   use_graph=True))
    ops, streams = runner.ops, []
    inner = ops.library_workspace
    monkeypatch.setattr(ops, "library_workspace", lambda stream: (streams.append(stream), inner(stream)))
    monkeypatch.setattr(ops, "_side_library", False)
    monkeypatch.setattr(ops, "side_own_max_rows", 0)   # (the second stream's short products would stay out of the library)
    monkeypatch.setattr(ops, "pays_beside", lambda rows, weight_bytes, dtype: True)
    slots = [runner.open() for _ in range(batch)]
    runner.step([Chunk(s, list(range(5)), []) for s in slots])   # rows on two streams
    beside = len(streams)
    for i in range(4):   # eager, captured, replayed
        runner.step([Chunk(s, [7 + i], [0]) for s in slots])
    assert runner._graphs and ops._side is not None
    assert (beside > 0) == (dtype == "bfloat16" and 5 * batch > 32) and (len(streams) > beside) == kept
