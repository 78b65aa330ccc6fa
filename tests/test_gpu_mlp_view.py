"""The fp32 networks' forward on split bfloat16 products (forward-only steps and the marched render) against the
same networks in float64 on the GPU's own encodings, for every built shape, with ragged sample counts."""
import numpy as np
import pytest

from common import default_scalars, look_at_rays, random_params, spec_cfg0
from oracle import oracle as ora

pytestmark = pytest.mark.gpu


def forward64(spec, p, a0, dirs, sh_mult):
    f = {k: np.asarray(v, np.float64) for k, v in p.items() if k[:2] in ("Wd", "Wc", "bd", "bc")}
    x = a0.astype(np.float64)
    dens = ["in"] + (["01"] if spec["nd"] >= 2 else []) + ["out"]
    for i, n in enumerate(dens):
        x = x @ f["Wd_" + n].T + f["bd_" + ("out" if n == "out" else str(i))]
        if n != "out":
            x = np.maximum(x, 0.0)
    d0 = np.clip(x[:, 0], -10, 10)
    sh = np.stack([ora_sh(d) for d in dirs]) * sh_mult
    x = np.concatenate([x, sh], 1)
    for i, n in enumerate(["in", "01", "out"]):
        x = x @ f["Wc_" + n].T + f["bc_" + ("out" if n == "out" else str(i))]
        if n != "out":
            x = np.maximum(x, 0.0)
    return np.log1p(np.exp(d0)), 1.0 / (1.0 + np.exp(-np.clip(0.5 * x, -18, 18)))


def ora_sh(d):
    import ctypes as C
    out = np.zeros(16, np.float32)
    d = np.ascontiguousarray(d, np.float32)
    ora.lib().ora_sh_encode(ora.fptr(d), ora.fptr(out))
    return out.astype(np.float64)


# Rounding of a layer: the split terms left out (2^-23) and one fp32 rounding per 32 products, of at most 64 products
# and a bias of a few units each, through five layers whose gains are near one; the activations add 1e-6 (their
# own test).  1e-5 of the largest output covers their sum; a wrong lane, plane or K order misses it by far.
@pytest.mark.parametrize("L,F,nd,n_rays,S", [(8, 2, 1, 33, 64), (16, 2, 1, 700, 16), (16, 4, 2, 129, 64),
                                             (16, 1, 1, 5, 4), (8, 4, 2, 65, 32), (16, 1, 2, 130, 64),
                                             (16, 4, 1, 40, 64), (32, 2, 2, 9, 64)])
def test_view_forward(L, F, nd, n_rays, S):
    from gpu_helpers import GpuModel
    spec = spec_cfg0(n_levels=L, f_per_level=F, log2_T=[12] * L, res=[4.0 + 3 * i for i in range(L)], nd=nd)
    p = random_params(spec, seed=L + F)
    rng = np.random.default_rng(L * F + nd)
    p["table"] = rng.normal(0, 0.5, p["table"].shape).astype(np.float32)
    rays = look_at_rays(n_rays, spec, seed=n_rays, miss_frac=0.2)
    sc = default_scalars(do_train=0, occ_strength=0.0)
    print(f"[view] LF={L * F} F={F} nd={nd} rays={n_rays} S={S}", flush=True)
    _, t = GpuModel(spec, p).train_step(rays, np.zeros((n_rays, 4), np.float32), S, sc, taps=True)
    dirs = np.repeat(rays[:, 4:7], S, axis=0)
    sig, rgb = forward64(spec, p, t["a0"].reshape(-1, L * F), dirs, sc["sh_multiplier"])
    on = t["DTs"].reshape(-1) > 0
    assert np.all(t["sigma"].reshape(-1)[~on] == 0)
    assert np.abs(t["sigma"].reshape(-1) - sig)[on].max() <= 1e-5 * max(1.0, sig.max())
    assert np.abs(t["rgb"].reshape(-1, 3) - rgb).max() <= 1e-5


def positive_params(spec, seed):
    p = random_params(spec, seed=seed)
    return {k: np.abs(v) if k == "table" or k[0] == "W" else v for k, v in p.items()}


def spoil(p, what):
    if what == "bias":
        p["bd_0"][5] = np.inf  # a hidden neuron of every sample
    elif what == "weight":
        p["Wd_in"][7, 3] = np.inf
    else:
        p["table"][::50] = 1e37  # the first layer's sums overflow where these entries are met
        p["Wd_in"] *= 1000.0
    return p


# All weights are positive, so infinities keep their sign through the layers and every output saturates (the
# density's and the colours' clamps), exactly as without the split: no sum becomes "not a number".
@pytest.mark.parametrize("what", ["bias", "weight", "table"])
def test_infinities(what):
    import ffn_lib as fl
    from gpu_helpers import GpuModel
    from test_gpu_march import shell_bits
    spec = spec_cfg0(n_levels=8, f_per_level=2, log2_T=[10] * 8, res=[4.0 + 3 * i for i in range(8)], occ_G=16)
    p = spoil(positive_params(spec, 3), what)
    n, S = 65, 32
    rays = look_at_rays(n, spec, seed=2, miss_frac=0.1)
    sc = default_scalars(do_train=0, occ_strength=0.0)
    print(f"[view infinities] {what}", flush=True)
    _, t = GpuModel(spec, p).train_step(rays, np.zeros((n, 4), np.float32), S, sc, taps=True)
    on = t["DTs"].reshape(-1) > 0
    with np.errstate(invalid="ignore"):
        sig, rgb = forward64(spec, p, t["a0"].reshape(-1, 16), np.repeat(rays[:, 4:7], S, axis=0), sc["sh_multiplier"])
    assert on.sum() > 200 and np.all(np.isfinite(sig[on])) and (sig[on] > 9.99).mean() > 0.2
    np.testing.assert_allclose(t["sigma"].reshape(-1)[on], sig[on], rtol=1e-5)
    np.testing.assert_allclose(t["rgb"].reshape(-1, 3)[on], rgb[on], rtol=1e-5, atol=1e-6)
    bits, dt = shell_bits(16, seed=1), np.float32(np.sqrt(3.0) / 64)
    ref, used_ref = ora.OracleModel(spec, p).render(rays, bits, ora.march_cfg(16, dt, 256, T_stop=1e-4))
    out, used = GpuModel(spec, p).render(rays, bits, fl.march_params(16, dt, 256, T_stop=1e-4, chunk=16))
    assert np.all(np.isfinite(ref)) and used_ref.sum() > 100
    assert np.mean(used == used_ref) > 0.99  # as test_render_matches_oracle
    same = used == used_ref
    np.testing.assert_allclose(out[same], ref[same], rtol=1e-3, atol=2e-5)
