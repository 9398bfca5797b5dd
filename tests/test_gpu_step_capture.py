"""p3x_main inside a captured graph (its kernels count the columns' order anew on every
replay): the replays, with the caller's own work and synchronisations between them,
give the bits of the eager step."""
import numpy as np
import pytest

from p3_compare import FLOAT_FIELDS, device_fields
from scream_amd import p3x
from scream_amd.inputs import make_columns

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [p3x.P3X_FP64, p3x.P3X_MIXED])
@pytest.mark.parametrize("ncol,nlev,lanes", [(300, 72, 0), (2100, 100, 32), (4200, 40, 16)])
def test_capture(host_tables, ncol, nlev, lanes, precision):
    import torch
    ctx = p3x.Context(host_tables)
    ctx.reserve(ncol, nlev)
    inp = make_columns(ncol, nlev, seed=ncol, dry_every=3, evap_every=9)
    d, _ = device_fields(inp)
    start = {k: d[k].clone() for k in p3x.STATE}

    def step(stream):
        ctx.main(d, ncol, nlev, 300.0, precision=precision, exchange_zeroed=True, sed_lanes_per_column=lanes,
                 stream=stream, async_=True)

    def restore():
        for k, v in start.items():
            d[k].copy_(v)

    step(torch.cuda.current_stream().cuda_stream)
    ctx.sync()
    want = {k: d[k].cpu().numpy() for k in FLOAT_FIELDS}
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            step(side.cuda_stream)
    for _ in range(3):
        restore()
        graph.replay()
        torch.cuda.synchronize()
        for k in FLOAT_FIELDS:
            np.testing.assert_array_equal(d[k].cpu().numpy(), want[k], err_msg=k)
    ctx.close()
