"""The render's compositing loads a ray's samples a group at a time: rounds of chunks around the group give the image
and samples used of rounds of one sample, bit for bit, with rays that stop inside a group and rays that do not, and
those of the restatement within rounding."""
import numpy as np
import pytest

from common import look_at_rays, random_params, spec_cfg0
from test_gpu_no_wait import shell_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T_stop", [0.0, 1e-2, 0.5])
def test_groups_of_samples(T_stop):
    import ffn_lib as fl
    from gpu_helpers import GpuModel
    from oracle import oracle as ora
    spec = spec_cfg0()
    p = random_params(spec, seed=81)
    p["bd_out"][0] = 6.0
    R, max_steps, dt = 32, 60, np.float32(np.sqrt(3.0) / 128)
    bits = shell_bits(R, seed=82, frac=0.1)
    rays = look_at_rays(300, spec, seed=83, miss_frac=0.1)
    g = GpuModel(spec, p)
    one, used = g.render(rays, bits, fl.march_params(R, dt, max_steps, T_stop=T_stop, chunk=1))
    assert used.sum() > 1000
    for chunk in (2, 7, 8, 9, 17, 60):
        print(f"[render groups] T_stop={T_stop} chunk={chunk}", flush=True)
        out, u = g.render(rays, bits, fl.march_params(R, dt, max_steps, T_stop=T_stop, chunk=chunk))
        np.testing.assert_array_equal(out.view(np.uint32), one.view(np.uint32))
        np.testing.assert_array_equal(u, used)
    ref, used_ref = ora.OracleModel(spec, p).render(rays, bits, ora.march_cfg(R, dt, max_steps, T_stop=T_stop))
    same = used == used_ref  # a stop can move by one sample where T crosses T_stop within rounding
    assert np.mean(same) > 0.99
    np.testing.assert_allclose(one[same], ref[same], rtol=1e-3, atol=2e-5)
