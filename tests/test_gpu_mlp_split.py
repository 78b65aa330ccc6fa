"""One layer through the split bfloat16 products of the fp32 networks' forward against float64 sums, beside the fp32
matrix instruction in the same order of inputs: dense rows, rows where one or three products are the sum, and operands
whose lower planes are as large as they get (the terms of a product that may not be left out)."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_math import _load
from test_gpu_mlp_view import planes

N = 4096
FULL = np.uint32(0x3F80FFFF).view(np.float32)  # h = 1, m and l one unit below their bounds 2^-7 and 2^-15


def operands(kind, K):
    rng = np.random.default_rng(K)
    x = rng.standard_normal((N, K)).astype(np.float32)
    W = (rng.standard_normal((64, K)) * np.sqrt(2.0 / K)).astype(np.float32)
    B = np.zeros(64, np.float32)
    if kind == "bias":
        B = rng.normal(0, 0.1, 64).astype(np.float32)
    elif kind == "relu":
        x = np.maximum(x, 0)
    elif kind == "positive":
        x, W = np.abs(x), np.abs(W)
    elif kind == "large":
        x[np.arange(N), rng.integers(0, K, N)] *= 4096  # one input far above the others
    elif kind != "dense":
        keep = np.zeros((64, K), bool)
        for o in range(64):
            keep[o, rng.permutation(K)[:1 if "one" in kind else 3]] = True
        if kind.startswith("full"):
            x, W = np.full_like(x, FULL), np.sign(W) * FULL
        W = np.where(keep, W, 0).astype(np.float32)
    return x, W, B


def layer(split, x, W, B):
    import torch
    lib = _load()
    lib.ffn_probe_layer.argtypes = [C.c_int, C.c_int] + [C.c_void_p] * 4 + [C.c_int]
    t = [torch.from_numpy(a).cuda() for a in (x, W, B)]
    out = torch.empty((N, 64), device="cuda")
    torch.cuda.synchronize()
    assert lib.ffn_probe_layer(x.shape[1] // 32, split, *[v.data_ptr() for v in t], out.data_ptr(), N) == 0
    return out.cpu().numpy().astype(np.float64)


MAX_TOL = 1.5 * 2.0 ** -24


# which products the layer test would miss: none of the eight
@pytest.mark.parametrize("term", [(0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0), (1, 2), (2, 1)])
def test_a_lost_term_shows(term):
    x, W, _ = operands("full one", 64)
    lost = np.abs(planes(x)[term[0]] @ planes(W)[term[1]].T)
    size = np.abs(x).astype(np.float64) @ np.abs(W).astype(np.float64).T
    assert (lost / size).max() > 2 * MAX_TOL


# The split sums may be no further from float64 than the fp32 instruction's (2-norm: of 262,144 sums, so steady to a
# per cent), nor, for their largest error, than that or one and a half roundings of the sum's terms.  With six of the
# eight terms a single product is off by up to 4.7e-7 and by 7e-8 in the 2-norm; with the fp32 instruction by 6.0e-8 and
# 2.5e-8.
@pytest.mark.gpu
@pytest.mark.parametrize("K", [32, 64])
@pytest.mark.parametrize("kind", ["dense", "bias", "relu", "positive", "large", "one", "three", "full one",
                                  "full three"])
def test_no_further_than_fp32(kind, K):
    x, W, B = operands(kind, K)
    ref = x.astype(np.float64) @ W.astype(np.float64).T + B
    size = np.abs(x).astype(np.float64) @ np.abs(W).astype(np.float64).T + np.abs(B)
    err = {}
    for split in (1, 0):
        print(f"[split layer] {kind} K={K} split={split}", flush=True)
        e = layer(split, x, W, B) - ref
        err[split] = np.linalg.norm(e) / np.linalg.norm(ref), np.max(np.abs(e) / size)
    print(f"[split layer] {kind} K={K}: split {err[1][0]:.2e} {err[1][1]:.2e}, fp32 {err[0][0]:.2e} {err[0][1]:.2e}")
    assert err[1][0] <= 1.02 * err[0][0]
    assert err[1][1] <= max(err[0][1], MAX_TOL)
