"""p3x_column_budget on columns of few levels: the sums are the oracle's bits at every
shape of its tiles (levels rounded up to a power of two, as many columns as that
leaves), and many columns of one level cost no more than the same points in deep ones."""
import numpy as np
import pytest

import oracle
from scream_amd import p3x

pytestmark = pytest.mark.gpu

FIELDS = ("pseudo_density", "T_mid", "qv", "qc", "qi", "qr")
LAYOUTS = {False: p3x.P3X_LEVEL_MAJOR, True: p3x.P3X_COLUMN_MAJOR}


@pytest.mark.parametrize("ncol,nlev", [(1023, 1), (1025, 1), (513, 2), (255, 3), (257, 4), (129, 5), (128, 8), (65, 9),
                                       (64, 16), (33, 17), (31, 32), (17, 33), (16, 127), (15, 128)])
@pytest.mark.parametrize("column_major", [False, True])
@pytest.mark.parametrize("full", [False, True])
def test_few_levels(host_tables, ncol, nlev, column_major, full):
    import torch
    rng = np.random.default_rng(ncol * 1000 + nlev)
    f = {k: rng.uniform(0.1, 1.0, (nlev, ncol)) for k in FIELDS}
    if full:
        f.update({k: rng.standard_normal((nlev, ncol)) for k in ("u", "v")})
        f.update({k: rng.uniform(0.5, 2.0, ncol) for k in ("ps", "phis")})
    d = {k: torch.from_numpy(np.ascontiguousarray(v.T if v.ndim == 2 and column_major else v)).to("cuda:0")
         for k, v in f.items()}
    m, e = (torch.full((ncol,), np.nan, dtype=torch.float64, device="cuda:0") for _ in range(2))
    ctx = p3x.Context(host_tables)
    p3x.column_budget(ctx, d, ncol, nlev, m, e, torch.cuda.current_stream().cuda_stream, layout=LAYOUTS[column_major])
    torch.cuda.synchronize()
    ctx.close()
    wm, we = oracle.column_budget(f)
    np.testing.assert_array_equal(m.cpu().numpy(), wm)
    np.testing.assert_array_equal(e.cpu().numpy(), we)


@pytest.mark.parametrize("column_major", [False, True])
def test_one_level_costs_no_more_than_many(host_tables, column_major):
    import torch
    ctx = p3x.Context(host_tables)
    stream = torch.cuda.current_stream().cuda_stream

    def best(ncol, nlev):
        f = {k: torch.rand(ncol * nlev, dtype=torch.float64, device="cuda:0") for k in FIELDS}
        m, e = (torch.zeros(ncol, dtype=torch.float64, device="cuda:0") for _ in range(2))
        times = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                p3x.column_budget(ctx, f, ncol, nlev, m, e, stream, layout=LAYOUTS[column_major])
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    # 64 MB against 48 MB of traffic; with 16 columns per block at any depth 3.1 and 17 times
    assert best(1_000_000, 1) <= 2.5 * best(15_625, 64)
    ctx.close()
