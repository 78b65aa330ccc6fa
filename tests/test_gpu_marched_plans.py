"""A marched step sized for a sample capacity leaves the state of the waiting step bit for bit on both sides of the ray
count from which the scatter takes large buckets, also where the two steps' capacity and count ask for other dense
copies of the coarse levels."""
import numpy as np
import pytest

from common import default_scalars, look_at_rays, random_params, spec_cfg0, sphere_targets

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rays", [1535, 1536])
@pytest.mark.parametrize("max_steps,capacity", [(9, 14000), (60, 92160)])
def test_capacity_step_is_the_waiting_step(n_rays, max_steps, capacity):
    import ffn_lib as fl
    from gpu_helpers import GpuModel
    spec = spec_cfg0(log2_T=[14] * 4 + [17] * 4)
    p = random_params(spec, seed=17)
    R = 32
    rays = look_at_rays(n_rays, spec, seed=n_rays, miss_frac=0.1)
    tg = sphere_targets(rays, spec)
    bits = np.full(R ** 3 // 32, 0xFFFFFFFF, np.uint32)
    out = []
    for cap in (0, capacity if capacity <= n_rays * max_steps else n_rays * max_steps):
        m = GpuModel(spec, p)
        mp = fl.march_params(R, np.float32(1.0 / 100), max_steps, T_stop=1e-3, sample_capacity=cap)
        print(f"[marched plans] rays={n_rays} max_steps={max_steps} capacity={cap}", flush=True)
        for seed in (1, 2):
            rgb, used = m.step_marched_plain(rays, tg, bits, mp, default_scalars(rng_seed=seed))
        out.append((rgb, used, m.state()))
    (rgb0, used0, s0), (rgb1, used1, s1) = out
    assert used0.sum() > 5 * n_rays
    np.testing.assert_array_equal(rgb0.view(np.uint32), rgb1.view(np.uint32))
    np.testing.assert_array_equal(used0, used1)
    for k in s0:
        np.testing.assert_array_equal(s0[k].view(np.uint32), s1[k].view(np.uint32), err_msg=k)
