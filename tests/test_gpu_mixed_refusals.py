"""The mixed form reports an inverse Exner function of 0, or too small to divide by, as a
bad temperature, in a single step and in a batch; the neighbouring steps are fine."""
import numpy as np
import pytest

from p3_compare import device_fields
from scream_amd import p3x
from scream_amd.inputs import make_columns

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [0.0, 5e-324, 1e-310])
@pytest.mark.parametrize("batch", [False, True])
def test_zero_inverse_exner(host_tables, value, batch):
    import torch
    ncol, nlev = 70, 24
    ctx = p3x.Context(host_tables)
    stream = torch.cuda.current_stream().cuda_stream
    good = make_columns(ncol, nlev, seed=9)
    bad = {k: v.copy() for k, v in good.items()}
    bad["inv_exner"][3, 5] = value

    def step(inp):
        d, _ = device_fields(inp)
        if batch:
            b = p3x.Batch(ctx, [p3x.column_set(d, ncol, nlev, 300.0, exchange_zeroed=True)],
                          p3x.batch_defaults(precision=p3x.P3X_MIXED))
            b.run(stream)
            status = ctx.sync()
            b.close()
            return status
        ctx.main(d, ncol, nlev, 300.0, precision=p3x.P3X_MIXED, exchange_zeroed=True, stream=stream, async_=True)
        return ctx.sync()

    assert [step(i) for i in (good, bad, good)] == [p3x.P3X_OK, p3x.P3X_ERR_TEMPERATURE, p3x.P3X_OK]
    ctx.close()
