"""Tables of more than 4 GB, whose rows 32-bit offsets do not reach from the table's start: rounds with a row
beyond the first 4 GB (rfx::RowWindow) load by 64-bit addresses.  Integer-valued rows, so that sums are exact in any
order."""

import numpy as np
import pytest

from helpers import require_lib

pytestmark = pytest.mark.gpu


def _window_rows(stride: int) -> int:
    """rfx::RowWindow::ROWS of rows of ``stride`` bytes."""
    return (2 ** 32 - max(4096, stride)) // stride


def _rows_to_look_up(spec, stride, rng):
    """Rows around the ends of the table and of every 4 GB of it, and some anywhere."""
    edges = [0, 1, spec.rows - 2, spec.rows - 1]
    window = _window_rows(stride)
    assert spec.rows > window
    for at in range(window, spec.rows, window):
        edges += [at - 1, at, min(at + 1, spec.rows - 1)]
    return np.unique(np.concatenate([edges, rng.integers(0, spec.rows, 40)]))


@pytest.mark.parametrize("spread", ["all windows", "one window"])
def test_rows_beyond_four_gigabytes(spread):
    import torch
    from recflex_amd import prebuilt
    from recflex_amd.rec_modules import FeatEmbed
    from recflex_amd.workloads import row_stride
    wl = prebuilt.model_spec("bigtables").workload
    dev = torch.device("cuda", 0)
    rng = np.random.default_rng(5)
    tables, indices, offsets, want = [], [], [], []
    for f in wl.features:
        stride = row_stride(f.dim, f.data_type)
        rows = _rows_to_look_up(f, stride, rng)
        if spread == "one window":
            rows = rows[rows < _window_rows(stride)]
        # the values of the rows that are looked up; nothing else of the table is written or read
        values = rng.integers(-8, 9, (len(rows), f.dim))
        if f.data_type == "int8":
            codes = rng.integers(0, 256, (len(rows), f.dim))
            content = np.zeros((len(rows), stride), np.uint8)
            content[:, :f.dim] = codes
            content[:, f.dim:f.dim + 4] = np.array([0.5, 3.0], np.float16).view(np.uint8)
            values = codes * 0.5 + 3.0
            table = torch.empty(f.rows, stride, dtype=torch.uint8, device=dev)
        else:
            dtype = torch.float32 if f.data_type == "float" else torch.float16
            content = values.astype(np.float32 if f.data_type == "float" else np.float16)
            table = torch.empty(f.rows, f.dim, dtype=dtype, device=dev)
        table[torch.from_numpy(rows).to(dev)] = torch.from_numpy(content).to(dev)
        lens = rng.poisson(f.mean_bag, wl.batch)
        lens[::9] = 0
        lens[5] = 400                       # beyond its schedule: summed by a whole wavefront
        picks = rng.integers(0, len(rows), lens.sum())
        bag_of = np.repeat(np.arange(wl.batch), lens)
        pooled = np.zeros((wl.batch, f.dim))
        np.add.at(pooled, bag_of, values[picks])
        want.append(pooled)
        tables.append(table)
        indices.append(torch.from_numpy(rows[picks].astype(np.int32)).to(dev))
        offsets.append(torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).to(dev))
    print(f"[case] bigtables, {spread}", flush=True)
    layer = FeatEmbed(dev, embed_tables=tables, librecom=require_lib("bigtables"))
    got = layer.forward_indices(indices, offsets).cpu().numpy()
    # sums of at most a thousand integers and halves below 2^8: exact in fp32
    np.testing.assert_array_equal(got, np.concatenate(want, 1).astype(np.float32))
