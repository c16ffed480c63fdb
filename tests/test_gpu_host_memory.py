"""Pinned host memory of the builders: what a build needs is lent and given back,
so that builds from ever new threads allocate no more than one thread's."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def _builds(out):
    import cubql_amd as cq
    g = torch.Generator("cuda").manual_seed(1)
    B = cq.points_to_boxes(torch.rand((2000, 3), device="cuda", generator=g))
    with torch.cuda.stream(torch.cuda.Stream()):
        torch.cuda.current_stream().wait_stream(torch.cuda.default_stream())
        trees = [b(B, cq.BuildConfig(makeLeafThreshold=8, maxAllowedLeafSize=8))
                 for b in (cq.gpuBuilder, cq.cuda.radixBuilder, cq.cuda.rebinRadixBuilder, cq.cuda.sahBuilder)]
        wide = cq.wideGpuBuilder(B, 4, cq.BuildConfig(makeLeafThreshold=8))
        torch.cuda.current_stream().synchronize()
        out.append([t.nodes_tensor()[2:, :6].sum().item() for t in trees] + [wide.numNodes])


def test_threads_give_their_memory_back():
    print("[gpu] pinned memory of builds from threads", flush=True)
    out = []
    _builds(out)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU,
                                            torch.profiler.ProfilerActivity.CUDA]) as prof:
        for _ in range(6):
            t = threading.Thread(target=_builds, args=(out,))
            t.start()
            t.join()
        torch.cuda.synchronize()
    calls = [e.name for e in prof.events() if e.name.startswith("hip")]
    assert sum(c == "hipLaunchKernel" or "LaunchKernel" in c for c in calls) > 6 * 20
    assert not [c for c in calls if "HostMalloc" in c or "HostAlloc" in c]
    assert len(out) == 7 and all(o[-1] == out[0][-1] for o in out)


def test_builds_at_the_same_time():
    print("[gpu] builds from eight threads at once", flush=True)
    one, out = [], []
    _builds(one)
    threads = [threading.Thread(target=_builds, args=(out,)) for _ in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    # (the rebin builder does not fix the numbering of its nodes, nor a sum its order)
    assert len(out) == 8
    for o in out:
        assert o[-1] == one[0][-1]
        assert all(abs(a - b) <= 1e-4 * abs(b) for a, b in zip(o, one[0]))
