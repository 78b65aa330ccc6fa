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


# A step of fewer samples takes the small batches' buckets, which need more scratch a sample than the large ones of the
# eager step before it; under capture nothing can be allocated.
@pytest.mark.parametrize("marched", [False, True])
def test_smaller_step_is_captured(marched):
    import ctypes as C
    import ffn_lib as fl
    import torch
    from gpu_helpers import GpuModel
    spec = spec_cfg0(n_levels=8, f_per_level=2, log2_T=[19] * 8, res=[16.0 * 1.6 ** i for i in range(8)])
    p = random_params(spec, seed=2)
    n_large, n_small = (3000, 1000) if marched else (4800, 2900)
    rays = torch.from_numpy(look_at_rays(n_large, spec, seed=3)).cuda()
    tg, out = torch.rand((n_large, 4), device="cuda"), torch.zeros((n_large, 4), device="cuda")
    bits = torch.full((32 ** 3 // 32,), -1, dtype=torch.int32, device="cuda")
    mp = fl.march_params(32, np.float32(1.0 / 100), 200, T_stop=1e-3, sample_capacity=200000)
    d = default_scalars()
    sc = fl.FfnStepScalars()
    for k in ("lr", "lr_t", "color_rel_lr", "sh_multiplier", "occ_strength", "beta1", "beta2", "eps"):
        setattr(sc, k, float(d[k]))
    sc.rng_seed, sc.do_train = 5, 1

    def step(m, n):
        if marched:
            rc = m.lib.ffn_train_step_marched(m.h.h, fl.ptr(rays), fl.ptr(tg), fl.ptr(out), n, fl.ptr(bits),
                                              C.byref(mp), C.byref(sc), None, None, fl.stream_ptr())
        else:
            rc = m.lib.ffn_train_step(m.h.h, fl.ptr(rays), fl.ptr(tg), fl.ptr(out), n, 64, C.byref(sc), None,
                                      fl.stream_ptr())
        fl.check(rc, "step")

    print(f"[graph scratch] smaller step marched={marched}", flush=True)
    m, ref = GpuModel(spec, p), GpuModel(spec, p)
    step(m, n_large)
    step(ref, n_large)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        step(m, n_small)
    for _ in range(3):
        graph.replay()
        step(ref, n_small)
        torch.cuda.synchronize()
        a, b = m.state(), ref.state()
        for k in a:
            np.testing.assert_array_equal(a[k].view(np.uint32), b[k].view(np.uint32), err_msg=k)


# asked for the spatial order, a captured encode takes the plain one if no eager call has sized the order's scratch
def test_order_is_not_allocated_under_capture(monkeypatch):
    import torch
    m = model()
    n = 70000
    x, out, ref = torch.rand((n, 3), device="cuda"), torch.zeros((n, 32), device="cuda"), torch.zeros((n, 32), device="cuda")
    print("[graph scratch] order under capture", flush=True)
    monkeypatch.setenv("FFN_ORDER", "0")
    encode(m, x, ref, n)
    torch.cuda.synchronize()
    monkeypatch.setenv("FFN_ORDER", "1")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        encode(m, x, out, n)
    for _ in range(2):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
