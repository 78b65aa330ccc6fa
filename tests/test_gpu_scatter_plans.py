"""The scatter's launch plans: bucket sizes per level (small and large batches), the strided and the transposed run
table, and the update's four-wide and scalar accesses, against the oracle's float64 sums and each other."""
import numpy as np
import pytest

from common import random_params, spec_cfg0, table_floats
from oracle import oracle as ora

pytestmark = pytest.mark.gpu


def scatter(m, x, g, n_tab, shift):
    """ffn_hash_encode_bwd into a zeroed gradient that starts `shift` elements past an aligned address."""
    import ffn_lib as fl
    import torch
    dt = torch.float16 if m.f16 else torch.float32
    buf = torch.zeros(n_tab + shift, dtype=dt, device="cuda")
    x_t, g_t = torch.from_numpy(x).cuda(), torch.from_numpy(g).cuda()
    fl.check(m.lib.ffn_hash_encode_bwd(m.h.h, fl.ptr(x_t), fl.ptr(g_t), x.shape[0],
                                       buf.data_ptr() + shift * buf.element_size(), fl.stream_ptr()), "scatter")
    torch.cuda.synchronize()
    assert not buf[:shift].any()
    return buf[shift:].cpu().numpy().astype(np.float32)


# levels from two entries up to more than 256 (512 at F = 4) of the smallest buckets; n around one emit round
# (1024 samples, 512 at F = 4), around the 512 rounds from which the run table is transposed, around the 3 2^16 samples
# from which large buckets are used, and one point
@pytest.mark.parametrize("F,log2_T,n", [(1, [1, 5, 13, 21], 1), (1, [1, 5, 13, 21], 1025), (2, [2, 9, 14, 20], 1023),
                                        (2, [2, 9, 14, 20], 33000), (2, [12, 19], 512 * 1024),
                                        (2, [12, 19], 512 * 1024 + 1), (2, [12, 19], 3 * 65536 - 1),
                                        (2, [12, 19], 3 * 65536), (4, [3, 13, 17, 19], 3 * 65536 - 1),
                                        (4, [3, 13, 17, 19], 3 * 65536), (4, [3, 13, 17, 20], 513),
                                        (4, [3, 13, 17, 20], 512 * 512 + 7)])
@pytest.mark.parametrize("table", [0, 1])
def test_scatter_plans(F, log2_T, n, table):
    from gpu_helpers import GpuModel
    L = len(log2_T)
    spec = spec_cfg0(n_levels=L, f_per_level=F, log2_T=log2_T, res=[2.0, 21.0, 64.0, 1025.0][:L], table_dtype=table,
                     nd=1, nc=2)
    rng = np.random.default_rng(F * 1000 + n)
    x = rng.random((n, 3), dtype=np.float32)
    g = rng.standard_normal((n, L * F), dtype=np.float32)
    n_tab = table_floats(spec)
    print(f"[scatter plans] F={F} log2_T={log2_T} n={n} table={table}", flush=True)
    m = GpuModel(spec, random_params(spec, seed=3))
    aligned, odd = scatter(m, x, g, n_tab, 0), scatter(m, x, g, n_tab, 1)
    np.testing.assert_array_equal(aligned, odd)
    ref = ora.hash_backward(ora.make_cfg(spec), x, g, n_tab)
    # products and run sums of up to 16 samples in fp32, then exact sums: 1e-5 of the largest entry (as the parity
    # suite); a binary16 gradient is that sum rounded once (2^-11 relative, 2^-25 near zero)
    tol = 1e-5 * np.abs(ref).max()
    if table:
        fits = np.abs(ref) < 65000
        assert np.all(np.abs(aligned - ref)[fits] <= tol + np.abs(ref)[fits] * 2.0 ** -11 + 2.0 ** -25)
    else:
        assert np.abs(aligned - ref).max() <= tol
