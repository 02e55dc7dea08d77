"""The step that runs its two cell lists on two streams: in a stream capture the
second one joins the first again, and replays, with other work and
synchronizations between them, give the bits of the eager step each time."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_captured_steps_match_eager_steps():
    import torch
    from salsa_amd import capi, workload as W
    desc = capi.bin_desc()
    f = W.config_fields(desc, 4, grid_override=(40, 16, 25))
    g = f.grid
    T = lambda a: torch.from_numpy(np.array(a)).cuda()
    fd = {k: T(getattr(f, k)) for k in ("press", "temp", "rsl", "rsi", "dn", "rv")}
    n, m = [T(x) for x in f.n[:3]], [T(x) for x in f.m[:3]]
    out = [torch.zeros_like(x) for x in n + m + [fd["rv"]]]
    ctx = capi.Context(desc, capi.params(level=4), g.nzp, g.nxp, g.nyp)
    stream = torch.cuda.ExternalStream(ctx.stream)
    step = lambda: ctx.step_device(fd, n, m, out[:3], out[3:6], out[6])
    step()
    ctx.sync()
    want = [x.clone() for x in out]
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        step()
    for _ in range(4):
        for x in out:
            x.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, want):
            assert torch.equal(a, b)
    ctx.close()
