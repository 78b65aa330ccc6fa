"""Scratch buffers of a handle and captured calls: what a graph uses stays, later eager calls' buffers are freed as they
grow, and a smaller call than an eager one before it can be captured."""
import numpy as np
import pytest

from common import default_scalars, look_at_rays, random_params, spec_cfg0

pytestmark = pytest.mark.gpu

SIZES = [1 << 20, 3 << 19, 1 << 21, 5 << 19, 3 << 20]


def model():
    from gpu_helpers import GpuModel
    spec = spec_cfg0(n_levels=16, f_per_level=2, log2_T=[10] * 16, res=[4.0 + 2 * i for i in range(16)])
    return GpuModel(spec, random_params(spec, seed=1))


def encode(m, x, out, n):
    import ffn_lib as fl
    fl.check(m.lib.ffn_hash_encode_fwd(m.h.h, fl.ptr(x), n, fl.ptr(out), None, fl.stream_ptr()), "encode")


def free_bytes():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def capture(call):
    import torch
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        call()
    return graph


# growing eager calls after a capture hold what they would hold without one, and the captured call's buffers
@pytest.mark.parametrize("captured", ["nothing", "encode", "sample"])
def test_later_buffers_are_freed(monkeypatch, captured):
    import ffn_lib as fl
    import torch
    monkeypatch.setenv("FFN_ORDER", "0")
    m = model()
    n0 = 1 << 18
    x, out = torch.rand((SIZES[-1], 3), device="cuda"), torch.empty((SIZES[-1], 32), device="cuda")
    rays = torch.from_numpy(look_at_rays(64, m.spec, seed=1)).cuda()
    ts, dts = torch.empty(64 * 64, device="cuda"), torch.empty(64 * 64, device="cuda")
    flags = torch.empty(128, dtype=torch.int32, device="cuda")

    def sample():  # no scratch
        fl.check(m.lib.ffn_sample(m.h.h, fl.ptr(rays), 64, 64, 3, 1, fl.ptr(ts), fl.ptr(dts), fl.ptr(flags),
                                  fl.stream_ptr()), "sample")

    print(f"[graph scratch] captured={captured}", flush=True)
    encode(m, x, out, n0)
    before = free_bytes() + n0 * 32 * 4
    graph = None
    if captured == "encode":
        graph = capture(lambda: encode(m, x, out, n0))
    elif captured == "sample":
        graph = capture(sample)
    for n in SIZES:
        encode(m, x, out, n)
    held = before - free_bytes()
    kept = n0 * 32 * 4 if captured == "encode" else 0
    assert held <= (SIZES[-1] * 32 * 4 + kept) + (64 << 20), held  # torch's graph pool and dense copies: far below 64 MB
    if graph is not None:
        ref = torch.empty((n0, 32), device="cuda")
        encode(m, x, ref, n0)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        if captured == "encode":
            assert torch.equal(out[:n0], ref)
