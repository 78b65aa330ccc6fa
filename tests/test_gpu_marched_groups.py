"""The marched step's compositing takes a ray's samples 64 at a time: rays whose sample counts and terminations lie
at the edges of a group, against the restatement."""
import numpy as np
import pytest

from common import default_scalars, look_at_rays, random_params, spec_cfg0, sphere_targets
from parity import compare_marched_step

pytestmark = pytest.mark.gpu


# every ray that meets the box takes max_steps samples of the full field; a dense field (density up to 10) ends its
# rays inside the first group, at T_stop 0.5 after a few samples, or not at all
@pytest.mark.parametrize("max_steps,T_stop,bias,background,occ", [(1, 0.0, 4.0, 1, 1.0), (63, 0.3, 8.0, 2, 1.0),
                                                                  (64, 0.0, 4.0, 2, 1.0), (65, 0.5, 8.0, 0, 1.0),
                                                                  (128, 1e-2, 8.0, 1, 0.0), (193, 0.0, 2.0, 2, 1.0)])
def test_marched_groups(max_steps, T_stop, bias, background, occ):
    import ffn_lib as fl
    import gpu_helpers as gh
    from oracle import oracle as ora
    R = 32
    spec = spec_cfg0(occ_G=R // 2, background=background)
    p = random_params(spec, seed=61)
    p["bd_out"][0] = bias
    p["occ_in"][:] = 0
    p["occ_st"][:] = 0
    n = 96
    rays = look_at_rays(n, spec, seed=62, miss_frac=0.1)
    print(f"[marched groups] max_steps={max_steps} T_stop={T_stop} background={background}", flush=True)
    mp = fl.march_params(R, np.float32(0.7 / 200), max_steps, T_stop=T_stop)
    compare_marched_step(spec, p, rays, sphere_targets(rays, spec), np.full(R ** 3 // 32, 0xFFFFFFFF, np.uint32), mp,
                         default_scalars(rng_seed=7, occ_strength=occ), gh, ora, flip_frac=0.03)
