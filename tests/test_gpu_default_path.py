"""The step as large calls take it: no column status words, the exchange fields zeroed on
entry, several columns per wavefront and the columns in p3_order_kernel's order.

* Single steps on both sides of the sizes at which the order is taken (more than 1024
  wavefronts, so from 4100 columns on at 16 lanes per column and 2050 at 32) give the bits
  of one column per wavefront, which takes the columns as they come.
* Large steps with the default lanes equal the oracle.
* The default lanes on both sides of every line of the rule that chooses them (columns,
  levels, precision and the length of the step) give the bits of 64 lanes."""
import numpy as np
import pytest

import oracle
from p3_compare import FLOAT_FIELDS, device_fields, field_errors
from scream_amd import p3x
from scream_amd.inputs import make_columns

pytestmark = pytest.mark.gpu

LEVEL, COLUMN = p3x.P3X_LEVEL_MAJOR, p3x.P3X_COLUMN_MAJOR
FP64, MIXED = p3x.P3X_FP64, p3x.P3X_MIXED


@pytest.fixture(scope="module")
def ctx(host_tables):
    c = p3x.Context(host_tables)
    yield c
    c.close()


def _step(ctx, inp, dt, precision, lanes, layout=LEVEL):
    import torch
    nlev, ncol = inp["qc"].shape
    d, _ = device_fields(inp)
    if layout == COLUMN:
        d = {k: v.t().contiguous() if v.dim() == 2 else v for k, v in d.items()}
    ctx.main(d, ncol, nlev, dt, precision=precision, exchange_zeroed=True, sed_lanes_per_column=lanes, layout=layout,
             stream=torch.cuda.current_stream().cuda_stream)
    return {k: d[k].cpu().numpy().T if layout == COLUMN and d[k].dim() == 2 else d[k].cpu().numpy() for k in FLOAT_FIELDS}


def _same(got, want):
    for k in FLOAT_FIELDS:
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)


@pytest.mark.parametrize("layout", [LEVEL, COLUMN])
@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("lanes,ncol,nlev", [(16, 4099, 20), (16, 4100, 20), (16, 4161, 72), (32, 2049, 20), (32, 2050, 20),
                                             (32, 2050, 100), (32, 2113, 150), (16, 9000, 15), (16, 9000, 16)])
def test_order_lines(ctx, lanes, ncol, nlev, precision, layout):
    inp = make_columns(ncol, nlev, seed=ncol, dry_every=3, evap_every=9)
    _same(_step(ctx, inp, 600.0, precision, lanes, layout), _step(ctx, inp, 600.0, precision, 64, layout))


@pytest.mark.parametrize("ncol,nlev,dt,layout", [(21600, 72, 1800.0, LEVEL), (5400, 72, 1800.0, COLUMN),
                                                 (6000, 128, 600.0, LEVEL), (3000, 72, 900.0, LEVEL)])
def test_large_step_against_oracle(ctx, oracle_tables, ncol, nlev, dt, layout):
    inp = make_columns(ncol, nlev, seed=ncol + 1, dry_every=3, evap_every=9)
    want, _, nerr = oracle.run_oracle(inp, oracle_tables, dt, math="portable")
    assert nerr == 0
    errs = field_errors(_step(ctx, inp, dt, FP64, 0, layout), want)
    assert max(errs.values()) <= 1e-10, errs


@pytest.mark.parametrize("precision,ncol,nlev,dt", [
    # few columns, 64 lanes, on one side
    (FP64, 2560, 72, 300.0), (FP64, 2561, 72, 300.0), (FP64, 2560, 72, 600.0), (FP64, 2561, 72, 600.0),
    (MIXED, 2560, 48, 300.0), (MIXED, 2561, 48, 300.0), (MIXED, 2561, 49, 300.0),
    # 32 and 16 lanes between them and many columns
    (FP64, 3072, 72, 600.0), (FP64, 3073, 72, 600.0), (FP64, 3072, 72, 599.0), (MIXED, 8192, 50, 300.0), (MIXED, 8193, 50, 300.0),
    # 80 and 160 levels
    (FP64, 2700, 80, 300.0), (FP64, 2700, 81, 300.0), (FP64, 2700, 160, 300.0), (FP64, 2700, 161, 300.0),
    (MIXED, 4096, 80, 300.0), (MIXED, 4096, 81, 300.0), (MIXED, 4097, 81, 300.0),
    # the groups apart, FP64 from 97 to 128 levels, and together where the step is long
    (FP64, 2700, 96, 300.0), (FP64, 2700, 97, 300.0), (FP64, 2700, 128, 300.0), (FP64, 2700, 129, 300.0),
    (FP64, 4096, 100, 432.0), (FP64, 4097, 100, 432.0), (FP64, 4097, 100, 431.0)])
def test_default_lanes(ctx, precision, ncol, nlev, dt):
    inp = make_columns(ncol, nlev, seed=ncol + nlev, dry_every=3, evap_every=9)
    _same(_step(ctx, inp, dt, precision, 0), _step(ctx, inp, dt, precision, 64))
