"""Blocks of TorchMemory on the library's stream, whether it is torch's current
stream (the block is allocated at once) or not (torch enters it): a build on
the default stream, on a side stream given by argument, on one that is
current, and with the two of them changed about, all equal, and the blocks
reused on the stream they were made on."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("current", ["default", "side"])
@pytest.mark.parametrize("given", ["none", "default", "side", "other"])
def test_blocks_follow_the_stream(current, given):
    import cubql_amd as cq
    print(f"[gpu] memory: current {current}, given {given}", flush=True)
    rng = np.random.default_rng(3)
    P = torch.from_numpy(rng.random((20000, 3), dtype=np.float32)).cuda()
    B = cq.points_to_boxes(P)
    want = cq.gpuBuilder(B, cq.BuildConfig(makeLeafThreshold=4))
    torch.cuda.synchronize()
    streams = {"none": None, "default": torch.cuda.default_stream(), "side": torch.cuda.Stream(),
               "other": torch.cuda.Stream()}
    mem = cq.TorchMemory(B.device)
    with torch.cuda.stream(streams[current]):
        got = [cq.gpuBuilder(B, cq.BuildConfig(makeLeafThreshold=4), stream=streams[given], mem=mem)
               for _ in range(3)]
    torch.cuda.synchronize()
    assert torch.cuda.current_stream() == torch.cuda.default_stream()
    for b in got:
        assert np.array_equal(cq.nodes_to_numpy(b), cq.nodes_to_numpy(want))
        assert torch.equal(b.prim_ids_tensor(), want.prim_ids_tensor())
    # the nodes, the primIDs, and no scratch
    assert len(mem.live) == 6
