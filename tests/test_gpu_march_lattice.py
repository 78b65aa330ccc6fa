"""The march's two walks (lattice points over a wavefront's lanes, cells one at a time per lane) give the same
samples bit for bit: FFN_MARCH_LATTICE=0 keeps the cell walk."""
import numpy as np
import pytest

from common import look_at_rays, random_params, spec_cfg0
from oracle import oracle as ora
from test_gpu_march import SPEC, shell_bits, special_rays

pytestmark = pytest.mark.gpu


def odd_rays(R):
    """Directions that are not unit vectors (a lattice of few or of very many points per ray), nearly parallel to
    an axis, or with zero, denormal, infinite and NaN components; origins inside, outside and far away."""
    rays = look_at_rays(24, SPEC, seed=R + 3)
    rays[:6, 4:7] *= np.float32(1e-3)
    rays[6:12, 4:7] *= np.float32(40.0)
    rays[12:14, 4] = np.float32(1e-6)
    rays[14, 5] = np.float32(1e-40)
    rays[15, 4:7] = 0.0
    rays[16, 4] = np.inf
    rays[17, 0] = np.nan
    rays[18, 5] = np.nan
    rays[19:24, :3] += (rays[19:24, :3] - 0.5) * np.float32(50.0)
    return rays


# (R, lattice points along the box diagonal, max_steps): fewer points than lanes, more cells than points and the
# reverse, ends that are multiples of a group of 64 points and not; ray counts that do not fill a wavefront
@pytest.mark.parametrize("R,K,max_steps,n", [(16, 33, 4096, 1), (32, 256, 5, 70), (44, 700, 4096, 333),
                                             (128, 1024, 64, 1500), (256, 1024, 1024, 900), (64, 4096, 4096, 300)])
def test_walks_agree(monkeypatch, R, K, max_steps, n):
    import ffn_lib as fl
    from gpu_helpers import GpuModel
    p = random_params(SPEC, seed=5)
    p["bd_out"][0] = 6.0
    g = GpuModel(SPEC, p)
    bits = shell_bits(R, seed=R, frac=0.01, half_width=0.03)
    dt = np.float32(np.sqrt(3.0) / K)
    rays = np.concatenate([look_at_rays(n, SPEC, seed=n, miss_frac=0.1), special_rays(R), odd_rays(R)])[:max(n, 1) + 400]
    res, img = [], []
    for env in ("1", "0"):  # these shapes take the lattice walk unless it is off
        monkeypatch.setenv("FFN_MARCH_LATTICE", env)
        print(f"[walks] R={R} K={K} max_steps={max_steps} walk={env}", flush=True)
        res.append(g.march(rays, bits, fl.march_params(R, dt, max_steps)))
        # rounds resume each ray where the last one paused it
        img.append([g.render(rays[:n], bits, fl.march_params(R, dt, max_steps, T_stop=1e-2, chunk=c)) for c in (7, 64)])
    for a, b in zip(res[0], res[1]):
        np.testing.assert_array_equal(a, b)
    for (a, ua), (b, ub) in zip(*img):
        np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(ua, ub)
    cfg, m = ora.make_cfg(SPEC), ora.march_cfg(R, dt, max_steps)
    counts, offsets, samples = res[0][:3]
    for r in range(0, len(rays), 5):
        t = ora.march_ray(cfg, m, bits, rays[r])
        assert counts[r] == len(t)
        np.testing.assert_array_equal(samples[int(offsets[r]):int(offsets[r]) + len(t), 3], t)


# A negative t_near reaches a box behind the ray's origin, where the largest |t| is the entry's: the points that lie
# within rounding of a cell's face are found from that, and the lattice is as many roundings coarser as it lies away.
@pytest.mark.parametrize("away", [3.0, 60.0, 1000.0])
def test_box_behind_the_origin(monkeypatch, away):
    import ffn_lib as fl
    from gpu_helpers import GpuModel
    spec = dict(SPEC, t_near=-1e4)
    g = GpuModel(spec, random_params(spec, seed=5))
    R, n = 256, 1500
    bits = shell_bits(R, seed=R, frac=0.3, half_width=0.1)
    rays = look_at_rays(n, spec, seed=6, radius=away, miss_frac=0.0)
    rays[::2, 4:7] *= -1.0  # every other one looks away from the box
    mp = fl.march_params(R, np.float32(np.sqrt(3.0) / 1024), 1024)
    res = []
    for env in ("1", "0"):
        monkeypatch.setenv("FFN_MARCH_LATTICE", env)
        print(f"[walks behind] away={away} walk={env}", flush=True)
        res.append(g.march(rays, bits, mp))
    assert res[1][0][::2].sum() > 10000
    for a, b in zip(res[0], res[1]):
        np.testing.assert_array_equal(a, b)
