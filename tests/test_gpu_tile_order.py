"""The MLP's order of 64-sample tiles (busy ones first) where each block takes at most one tile, where a block
places several thousand, and in between: a step that skips its empty tiles leaves the state and colours of the
full path, bit for bit; and the scan behind the march's offsets at its one- and two-launch sizes."""
import numpy as np
import pytest

from common import default_scalars, look_at_rays, random_params, spec_cfg0, sphere_targets

pytestmark = pytest.mark.gpu


# rays of 64 samples: a tile each; 16 rays of 4 samples share one.  512 blocks run at once.
@pytest.mark.parametrize("n_rays,S,mlp", [(1, 64, 0), (512, 64, 0), (513, 64, 1), (527, 64, 0), (4097, 64, 1),
                                          (8209, 64, 0), (16 * 600 + 3, 4, 0), (16 * 600 + 3, 4, 1)])
def test_tile_order_changes_nothing(n_rays, S, mlp):
    from gpu_helpers import GpuModel
    spec = spec_cfg0(hash_opt=1, background=2, mlp_precision=mlp)
    p = random_params(spec, seed=91)
    rays = look_at_rays(n_rays, spec, seed=n_rays, miss_frac=0.4)
    tg = sphere_targets(rays, spec)
    print(f"[tile order] rays={n_rays} S={S} mlp={mlp}", flush=True)
    full, fast = GpuModel(spec, p), GpuModel(spec, p)
    out_full, _ = full.train_step(rays, tg, S, default_scalars(), taps=True)
    out_fast, _ = fast.train_step(rays, tg, S, default_scalars(), taps=False)
    np.testing.assert_array_equal(out_full.view(np.uint32), out_fast.view(np.uint32))
    sf, ss = full.state(), fast.state()
    for k in sf:
        np.testing.assert_array_equal(sf[k].view(np.uint32), ss[k].view(np.uint32), err_msg=k)


@pytest.mark.parametrize("n_rays", [1, 4095, 4096, 12287, 12288, 50001])
def test_march_offsets(n_rays):
    import ffn_lib as fl
    from gpu_helpers import GpuModel
    spec = spec_cfg0(occ_G=16)
    g = GpuModel(spec, random_params(spec, seed=1))
    rays = look_at_rays(n_rays, spec, seed=n_rays, miss_frac=0.3)
    print(f"[march offsets] rays={n_rays}", flush=True)
    mp = fl.march_params(32, np.float32(0.02), 16)
    counts, offsets, _, ids, total = g.march(rays, np.full(1024, 0x0F0F0F0F, np.uint32), mp)
    ends = np.cumsum(counts.astype(np.int64))
    np.testing.assert_array_equal(offsets, np.concatenate([[0], ends[:-1]]))
    assert total == ends[-1]
    np.testing.assert_array_equal(ids[:total], np.repeat(np.arange(n_rays), counts))
