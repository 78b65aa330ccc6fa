"""The marched step composites densities and colours that are the training kernel's own forward bit for bit (its
backward recomputes the activations, so the loss gradients belong to the ReLU branches that it takes)."""
import numpy as np
import pytest

from common import default_scalars, look_at_rays, random_params, spec_cfg0

pytestmark = pytest.mark.gpu


# A table of one value per level and feature encodes every point to that value within a rounding or two (to zero exactly
# on all levels but two), so samples of the marched and of the resampled step meet in the same encodings; a ray's
# direction is the same in both.
@pytest.mark.parametrize("L,F,nd", [(8, 2, 1), (16, 1, 2), (16, 2, 1), (8, 4, 2), (16, 4, 1), (32, 2, 2), (16, 4, 2)])
def test_forward_is_the_training_kernels(L, F, nd):
    import ffn_lib as fl
    from gpu_helpers import GpuModel
    spec = spec_cfg0(n_levels=L, f_per_level=F, log2_T=[8] * L, res=[3.0 + 2 * i for i in range(L)], nd=nd, occ_G=16)
    p = random_params(spec, seed=10 * L + F + nd)
    value = np.random.default_rng(L).uniform(-0.5, 0.5, (L, 1, F)).astype(np.float32)
    value[1:L - 1] = 0.0
    p["table"] = np.broadcast_to(value, (L, 256, F)).reshape(-1).copy()
    p["occ_in"][:] = 0xFFFFFFFF
    n, S, R = 40, 64, 32
    rays = look_at_rays(n, spec, seed=L, miss_frac=0.0)
    tg = np.zeros((n, 4), np.float32)
    print(f"[marched forward] LF={L * F} F={F} nd={nd}", flush=True)
    _, a = GpuModel(spec, p).train_step(rays, tg, S, default_scalars(occ_strength=0.0), taps=True)
    mp = fl.march_params(R, np.float32(1.0 / 200), 300, T_stop=0.0)
    _, _, b = GpuModel(spec, p).train_step_marched(rays, tg, np.full(R ** 3 // 32, 0xFFFFFFFF, np.uint32), mp,
                                                   default_scalars(occ_strength=0.0))
    on = a["DTs"].reshape(-1) > 0
    known = {(r, e.tobytes()): (s, c) for r, e, s, c in
             zip(np.repeat(np.arange(n), S)[on], a["a0"].reshape(n * S, -1)[on], a["sigma"].reshape(-1)[on],
                 a["rgb"].reshape(-1, 3)[on])}
    met = 0
    for r, e, s, c in zip(np.repeat(np.arange(n), b["n_march"]), b["a0"], b["sigma"], b["rgb"]):
        k = known.get((r, e.tobytes()))
        if k is not None:
            met += 1
            assert s == k[0] and np.array_equal(c, k[1])
    print(f"[marched forward] {met} of {len(b['sigma'])} samples met", flush=True)
    assert met >= 20
