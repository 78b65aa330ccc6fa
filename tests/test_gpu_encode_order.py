"""ffn_hash_encode_fwd in a spatial order of its points (FFN_ORDER=1) gives the encodings of the plain order bit for
bit: point counts around the sort's blocks and wavefronts, points that coincide, lie outside the box or are not
finite, every F and table type; and by its own rule beyond 2^20 points."""
import numpy as np
import pytest

from common import random_params, spec_cfg0

pytestmark = pytest.mark.gpu


def points(n, seed):
    rng = np.random.default_rng(seed)
    x = rng.random((n, 3), dtype=np.float32)
    x[rng.random(n) < 0.2] = np.float32(0.25)
    out = rng.random(n) < 0.05
    x[out] = x[out] * 7.0 - 3.0
    if n > 8:
        x[1] = np.nan
        x[3] = [np.inf, 0.5, -np.inf]
        x[5] = [1.0, 0.0, 1.0]
    return x


@pytest.mark.parametrize("n,F,table", [(1, 2, 0), (63, 1, 0), (4095, 2, 1), (4096, 4, 0), (4097, 2, 0), (70001, 1, 1),
                                       (262145, 4, 1)])
def test_order_changes_nothing(monkeypatch, n, F, table):
    from gpu_helpers import GpuModel
    L = 4
    spec = spec_cfg0(n_levels=L, f_per_level=F, log2_T=[9, 14, 16, 18], res=[5.0, 33.0, 130.0, 700.0],
                     table_dtype=table)
    m = GpuModel(spec, random_params(spec, seed=3))
    x = points(n, n)
    print(f"[encode order] n={n} F={F} table={table}", flush=True)
    res = []
    for env in ("0", "1", "1"):
        monkeypatch.setenv("FFN_ORDER", env)
        res.append(encode(m, x, L * F))
    np.testing.assert_array_equal(res[0].view(np.uint32), res[1].view(np.uint32))
    np.testing.assert_array_equal(res[1].view(np.uint32), res[2].view(np.uint32))


def encode(m, x, lf):
    import ffn_lib as fl
    import torch
    x_t = torch.from_numpy(x).cuda()
    out = torch.full((x.shape[0], lf), 7.0, device="cuda")
    fl.check(m.lib.ffn_hash_encode_fwd(m.h.h, fl.ptr(x_t), x.shape[0], fl.ptr(out), None, fl.stream_ptr()), "encode")
    return out.cpu().numpy()


def test_order_by_rule(monkeypatch):
    from gpu_helpers import GpuModel
    spec = spec_cfg0(n_levels=2, log2_T=[20, 20], res=[150.0, 900.0])
    m = GpuModel(spec, random_params(spec, seed=4))
    x = points((1 << 20) + 77, 5)
    print("[encode order] by rule", flush=True)
    monkeypatch.delenv("FFN_ORDER", raising=False)
    by_rule = encode(m, x, 4)
    monkeypatch.setenv("FFN_ORDER", "0")
    np.testing.assert_array_equal(by_rule.view(np.uint32), encode(m, x, 4).view(np.uint32))


def test_graph_outlives_larger_calls(monkeypatch):
    """An encode captured into a graph keeps its buffers when later eager calls outgrow them: its replays give the
    encodings of the points that the input holds then."""
    import ffn_lib as fl
    import torch
    from gpu_helpers import GpuModel
    spec = spec_cfg0(n_levels=2, log2_T=[16, 18], res=[40.0, 300.0])
    m = GpuModel(spec, random_params(spec, seed=6))
    monkeypatch.setenv("FFN_ORDER", "1")
    n = 70001
    x_t = torch.from_numpy(points(n, 7)).cuda()
    out = torch.zeros((n, 4), device="cuda")
    s = torch.cuda.Stream()

    def call():
        fl.check(m.lib.ffn_hash_encode_fwd(m.h.h, fl.ptr(x_t), n, fl.ptr(out), None, fl.stream_ptr()), "encode")

    print("[encode order] graph", flush=True)
    with torch.cuda.stream(s):
        call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        call()
    for rep in range(3):
        encode(m, points(4 * n * (rep + 1), 8 + rep), 4)
        x = points(n, 20 + rep)
        x_t.copy_(torch.from_numpy(x))
        graph.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy().view(np.uint32), encode(m, x, 4).view(np.uint32))


# The rule weighs what the levels gain: few large levels among none, or large levels so fine that no cell holds two
# points, keep the plain order; all 16 do not.  Seen by the order's scratch (36 bytes a point).
@pytest.mark.parametrize("log2_T,first,n,ordered", [([20, 20], 14, 1 << 20, False), ([22], 15, 1 << 20, False),
                                                    ([22] * 4, 12, 1 << 20, False), ([14] * 15 + [22], 0, 1 << 20, False),
                                                    ([22] * 16, 0, (1 << 20) - 1, False), ([22] * 16, 0, 1 << 20, True),
                                                    ([19] * 8, 8, 1 << 22, False), ([19] * 16, 0, 1 << 22, True)])
def test_rule_weighs_the_levels(monkeypatch, log2_T, first, n, ordered):
    import torch
    from gpu_helpers import GpuModel
    res = [float(np.rint(16.0 * 128.0 ** (l / 15))) for l in range(16)][first:first + len(log2_T)]
    spec = spec_cfg0(n_levels=len(log2_T), f_per_level=2, log2_T=log2_T, res=res)
    p = random_params(spec_cfg0(n_levels=len(log2_T), log2_T=[4] * len(log2_T), res=res), seed=4)
    for k in ("table", "m_table", "v_table"):
        p[k] = np.zeros(2 * sum(1 << t for t in log2_T), np.float32)
    p["table"] = np.resize(np.random.default_rng(n).random(999983, dtype=np.float32), p["table"].size)
    x = torch.rand((n, 3), device="cuda")
    held, outs = [], []
    for env in ("0", None):
        monkeypatch.setenv("FFN_ORDER", env) if env else monkeypatch.delenv("FFN_ORDER")
        m = GpuModel(spec, p)
        import ffn_lib as fl
        torch.cuda.synchronize()
        out = torch.zeros((n, 2 * len(log2_T)), device="cuda")
        before = torch.cuda.mem_get_info()[0]
        print(f"[encode order] rule levels={len(log2_T)} n={n} order={env}", flush=True)
        fl.check(m.lib.ffn_hash_encode_fwd(m.h.h, fl.ptr(x), n, fl.ptr(out), None, fl.stream_ptr()), "encode")
        torch.cuda.synchronize()
        held.append(before - torch.cuda.mem_get_info()[0])
        outs.append(out)
    assert torch.equal(outs[0].view(torch.int32), outs[1].view(torch.int32))
    assert (held[1] - held[0] > 30 * n) == ordered
