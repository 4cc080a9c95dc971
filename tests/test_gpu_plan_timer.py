"""Timing one entry point's launches inside planned steps: the memory commit
too where a small fp32 batch has it in the memory update's launches."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gemm", ["fp32", "bf16"])
def test_every_stage_of_the_front_part_is_timed(gpu, gemm):
    from starry_unigraph import SchedulerSession, synth
    from starry_unigraph.data import from_stream
    s = synth.bipartite_stream(num_src=200, num_dst=50, num_events=3000, edge_dim=4, seed=1)
    cfg = {"model": {"family": "tgn", "hidden_dim": 32}, "data": {"name": "t", "format": "synthetic"},
           "train": {"batch_size": 100, "lr": 1e-3}, "runtime": {"device": "cuda"},
           "ctdg": {"mailbox_slots": 1, "dim_time": 16, "num_head": 2, "dropout": 0.0, "att_dropout": 0.0,
                    "memory_gemm_dtype": gemm},
           "sampling": {"neighbor_limit": [10], "history": 1, "strategy": "recent"}}
    sess = SchedulerSession.from_config(cfg).with_events(from_stream(s))
    sess.build_runtime()
    rt = sess.ctdg_session.online_runtime
    rt.collect_results = False
    batches = list(rt.iter_batches("train", 100))
    rt.train_step(batches[0])
    assert rt.step.commits_in_update(rt._gru) == (gemm == "fp32")
    update = "sgl_memory_update" if gemm == "fp32" else "sgl_memory_update_bf16"
    for batch, name in zip(batches[1:], (update, "sgl_memory_commit", "sgl_edge_rows", "sgl_conv_forward")):
        pair = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        for e in pair:   # torch creates the HIP event at its first record
            e.record()
        torch.cuda.synchronize()
        rt.plan_timer = (name, lambda: pair)
        rt.train_step(batch)
        rt.plan_timer = None
        torch.cuda.synchronize()
        assert 0.0 < pair[0].elapsed_time(pair[1]) < 100.0, name
