"""Steps that keep no column status words (no status array, no check_values, exchange
fields zeroed on entry) give the bits of steps that do: a column's early exits and a
warm clear level's exchange fields come out the same either way."""
import numpy as np
import pytest

from p3_compare import FLOAT_FIELDS, device_fields
from scream_amd import p3x
from scream_amd.inputs import make_columns

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncol,nlev", [(1, 72), (63, 5), (64, 4), (65, 73), (200, 128), (33, 9)])
@pytest.mark.parametrize("precision", [p3x.P3X_FP64, p3x.P3X_MIXED])
@pytest.mark.parametrize("column_major", [False, True])
def test_untracked_step(host_tables, ncol, nlev, precision, column_major):
    import torch
    full = make_columns(ncol, max(nlev, 72), seed=ncol + nlev, dry_every=5, evap_every=4)
    inp = {k: v[-nlev:] for k, v in full.items()}  # the lowest levels: warm clear ones among them
    ctx = p3x.Context(host_tables)
    got = []
    for tracked, zeroed in ((True, False), (True, True), (False, True)):
        d, dbg = device_fields(inp)
        if zeroed:
            for k in p3x.HIST:
                d[k].fill_(float("nan"))  # every entry is written
        if column_major:
            d = {k: v.t().contiguous() if v.dim() == 2 else v for k, v in d.items()}
            dbg = {k: dbg[k] for k in ("col_status", "sed_substeps")}
        ctx.main(d, ncol, nlev, 300.0, precision=precision, debug=dbg if tracked else None,
                 exchange_zeroed=zeroed, stream=torch.cuda.current_stream().cuda_stream,
                 layout=p3x.P3X_COLUMN_MAJOR if column_major else p3x.P3X_LEVEL_MAJOR)
        got.append({k: d[k].cpu().numpy() for k in FLOAT_FIELDS})
    ctx.close()
    for other in got[1:]:
        for k in FLOAT_FIELDS:
            np.testing.assert_array_equal(other[k], got[0][k], err_msg=k)
