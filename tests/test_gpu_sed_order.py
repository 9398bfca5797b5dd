"""Sedimentation with several columns per wavefront takes the wet columns first
(p3_order_kernel): on both sides of the sizes at which it does, at the edges of its
64-column words, 512-column blocks and 128-level chunks, in both layouts, the results
are the bits of one column per wavefront, which takes the columns as they come."""
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


def _fields(inp, layout):
    d, _ = device_fields(inp)
    if layout == p3x.P3X_COLUMN_MAJOR:
        d = {k: v.t().contiguous() if v.dim() == 2 else v for k, v in d.items()}
    return d


def _check(got, want, what):
    for k in FLOAT_FIELDS:
        g, w = got[k].cpu().numpy(), want[k].cpu().numpy()
        np.testing.assert_array_equal(g, w, err_msg=f"{what} {k}")


@pytest.mark.parametrize("layout", [p3x.P3X_LEVEL_MAJOR, p3x.P3X_COLUMN_MAJOR])
@pytest.mark.parametrize("precision", [p3x.P3X_FP64, p3x.P3X_MIXED])
@pytest.mark.parametrize("lanes", [16, 32])
def test_batch_order(ctx, lanes, precision, layout):
    import torch
    # (columns, levels, every how many-th column is dry)
    sets = [(63, 40, 3), (64, 16, 2), (65, 17, 3), (200, 15, 2), (511, 72, 2), (513, 128, 5), (100, 72, 1)]
    if lanes == 32:
        sets += [(70, 129, 2), (1030, 150, 3)]
    inps = [make_columns(n, k, seed=n + k, dry_every=dry, evap_every=9) for n, k, dry in sets]
    runs = []
    for l in (64, lanes):
        fields = [_fields(i, layout) for i in inps]
        b = p3x.Batch(ctx, [p3x.column_set(f, n, k, 600.0, exchange_zeroed=True, layout=layout)
                            for f, (n, k, _) in zip(fields, sets)],
                      p3x.batch_defaults(precision=precision, sed_lanes_per_column=l))
        b.run(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        b.close()
        runs.append(fields)
    for s, want, got in zip(sets, *runs):
        _check(got, want, s)


@pytest.mark.parametrize("layout", [p3x.P3X_LEVEL_MAJOR, p3x.P3X_COLUMN_MAJOR])
@pytest.mark.parametrize("precision", [p3x.P3X_FP64, p3x.P3X_MIXED])
@pytest.mark.parametrize("ncol,lanes", [(4096, 16), (4097, 16), (2049, 32)])
def test_single_order(ctx, ncol, lanes, precision, layout):
    import torch
    nlev = 20
    inp = make_columns(ncol, nlev, seed=ncol, dry_every=3, evap_every=9)
    runs = []
    for l in (64, lanes):
        d = _fields(inp, layout)
        ctx.main(d, ncol, nlev, 600.0, precision=precision, exchange_zeroed=True, sed_lanes_per_column=l,
                 layout=layout, stream=torch.cuda.current_stream().cuda_stream)
        runs.append(d)
    _check(runs[1], runs[0], (ncol, lanes))
