"""Sedimentation shapes chosen by the number of columns: on both sides of the line
between few and many columns (2048), single sets and batches of several classes
give the bits of an explicit shape."""
import numpy as np
import pytest

from p3_compare import FLOAT_FIELDS, device_fields
from scream_amd import p3x
from scream_amd.inputs import make_columns

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(host_tables):
    c = p3x.Context(host_tables)
    yield c
    c.close()


def _single(ctx, inp, dt, precision, lanes):
    import torch
    nlev, ncol = inp["qc"].shape
    d, _ = device_fields(inp)
    ctx.main(d, ncol, nlev, dt, precision=precision, exchange_zeroed=True, sed_lanes_per_column=lanes,
             stream=torch.cuda.current_stream().cuda_stream)
    return {k: d[k].cpu().numpy() for k in FLOAT_FIELDS}


@pytest.mark.parametrize("precision", [p3x.P3X_FP64, p3x.P3X_MIXED])
@pytest.mark.parametrize("ncol,nlev", [(2048, 40), (2049, 40), (2047, 72), (2050, 72), (2049, 100)])
def test_shape_by_columns(ctx, ncol, nlev, precision):
    inp = make_columns(ncol, nlev, seed=ncol + nlev, dry_every=7, evap_every=9)
    got, want = _single(ctx, inp, 600.0, precision, 0), _single(ctx, inp, 600.0, precision, 32)
    for k in FLOAT_FIELDS:
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)


@pytest.mark.parametrize("precision", [p3x.P3X_FP64, p3x.P3X_MIXED])
@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("ncols", [(1, 65, 200, 33, 517), (1100, 900, 260, 33, 517)])
def test_batch_classes(ctx, ncols, precision, graph):
    import torch
    sets = [(n, k, dt) for n, (k, dt) in zip(ncols, ((72, 100.0), (128, 1800.0), (40, 300.0), (150, 1800.0), (72, 1800.0)))]
    inps = [make_columns(n, k, seed=n + k, dry_every=7, evap_every=9) for n, k, _ in sets]
    fields = [device_fields(i)[0] for i in inps]
    start = [{k: f[k].clone() for k in p3x.STATE} for f in fields]
    b = p3x.Batch(ctx, [p3x.column_set(f, n, k, dt, exchange_zeroed=True) for f, (n, k, dt) in zip(fields, sets)],
                  p3x.batch_defaults(precision=precision, use_graph=graph))
    want = [_single(ctx, i, dt, precision, 64) for i, (_, _, dt) in zip(inps, sets)]
    for rep in range(3):  # replays, with the caller's own copies in between
        for f, s in zip(fields, start):
            for k in p3x.STATE:
                f[k].copy_(s[k])
        b.run(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        for j, (f, w) in enumerate(zip(fields, want)):
            for k in FLOAT_FIELDS:
                np.testing.assert_array_equal(f[k].cpu().numpy(), w[k], err_msg=f"replay {rep} set {j} {k}")
    b.close()
