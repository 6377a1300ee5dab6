"""CPU: the part sizes of split bags (``rfx_tile_sizes.h``, the functions the device runs): what a size
is counted with is what the batch is cut into, models of equal features fill their rounds of the
grid, and no size is chosen that is dearer, by the same count, than the plain rule's."""

import ctypes

import numpy as np
import pytest

from helpers import PART_COST, bind_tiles_on_cpu, build_tile_model


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    return build_tile_model(str(tmp_path_factory.mktemp("tile_sizes") / "model.so"))


def split_cost(batch, lookups, dim):
    """Traffic of a feature as the emitter counts it: rows and indices, output rows and offsets."""
    return batch * lookups * (4.0 * dim + 4) + batch * (4.0 * dim + 4)


@pytest.mark.parametrize("features, dim, batch, lookups", [
    (8, 64, 16, 20000), (4, 128, 16, 20000), (2, 256, 16, 20000), (16, 64, 16, 20000), (8, 64, 64, 5000),
    (8, 64, 32, 10000), (1, 128, 16, 100000), (16, 32, 8, 40000), (3, 64, 100, 2222), (7, 96, 48, 4321)])
@pytest.mark.parametrize("grid", [2048, 1280, 1024, 304, 100])
def test_equal_features_fill_their_rounds(model, features, dim, batch, lookups, grid):
    """Bags of one cost: the parts of a round are at most ``grid // bags`` per bag, and no size leaves
    a round that a share of the batch in that many rounds would fill."""
    got = bind_tiles_on_cpu(model, [split_cost(batch, lookups, dim)] * features, [-1] * features, batch, grid, 65536)
    if got["counted"] < 0:
        assert got["unit"] == got["rule"]
        return
    bags, bag = features * batch, split_cost(batch, lookups, dim) / batch
    assert got["counted"] == got["tiles"].sum()
    best = min(-(-bags * p // grid) * (bag / p + PART_COST)
               for r in range(1, 5) for p in [max(1, min(64, 2048 // batch, grid * r // bags))]
               if bag / p >= 131072 and (p == 1 or p > 1.25) and bag / p >= 65536)
    # at least as good as the most parts that one, two, three or four rounds hold
    assert got["price"] <= best * (1 + 1e-5), got


def test_random_models_count_what_they_bind_and_never_lose(model):
    rng = np.random.default_rng(1)
    searched = 0
    for _ in range(20000):
        n = int(rng.integers(1, 17))
        grid = int(rng.choice([2048, 1280, 1024, 304, int(rng.integers(1, 4096))]))
        batch = int(np.exp(rng.uniform(0, np.log(4096))))
        tile_size = int(rng.choice([4096, 32768, 65536, 131072, 262144, 300000]))
        # around the window in which sizes are searched: 256 KiB to 1 MiB of traffic per workgroup
        share = np.exp(rng.uniform(np.log(128 * 1024), np.log(2 << 20)))
        weight = rng.random(n) + 0.05 if rng.random() < 0.7 else np.ones(n)
        cost = share * grid * weight / weight.sum()
        gran = np.where(rng.random(n) < 0.75, -1, rng.choice([1, 4, 16, 64], n))
        got = bind_tiles_on_cpu(model, cost, gran, batch, grid, tile_size)
        case = (n, grid, batch, tile_size, cost.tolist(), gran.tolist(), got)
        if got["counted"] < 0:
            assert got["unit"] == got["rule"], case
            continue
        searched += 1
        assert got["counted"] == got["tiles"].sum(), case
        assert got["price"] <= got["rule_price"] * (1 + 1e-6), case
        assert all(t <= 2048 for t, g in zip(got["tiles"], gran) if g == -1 and t > batch), case
    assert searched > 5000


def test_bags_just_below_the_split_limit_do_not_cost_rounds(model):
    """878 bags of a quarter of a megabyte in eight features: left whole in four rounds of 527 KB by a
    search that does not price the plain rule, five rounds of 263 KB by the rule."""
    for mean in range(1000, 2200, 50):
        got = bind_tiles_on_cpu(model, [split_cost(878, mean, 64)] * 8, [-1] * 8, 878, 2048, 65536)
        assert got["price"] <= got["rule_price"] * (1 + 1e-6)


def test_host_restatements_of_the_tile_sizes(model):
    """What the tuner computes on the host is what the device does: the size picked for a batch, and
    what becomes of a size that a library was emitted with."""
    from recflex_amd.tuning import measure
    rng = np.random.default_rng(2)
    cut = 0
    for _ in range(5000):
        total, grid = int(np.exp(rng.uniform(0, np.log(1e11)))), int(rng.integers(0, 4096))
        built = int(rng.choice([4096, 65536, 65537, 131072, 262144, 1 << 20]))
        want = model.model_capped_tile_size(built, ctypes.c_longlong(total), grid)
        assert measure.capped_tile_bytes(built, total, grid) == want
        cut += want < built
        # one bag of one lookup, `total` bytes in all
        off = np.array([0, 1], np.int64)
        auto = model.model_auto_tile_size(ctypes.c_longlong(total), grid)
        assert measure.auto_tile_bytes([off], [total - 1], [1], grid) == auto
    assert cut > 500


def test_tiles_of_a_library_emitted_with_large_tiles():
    """The walk stage's tile counts and the frozen bindings are those of the library that runs: one
    emitted with 256 KiB gives a batch of a few such tiles per workgroup smaller ones."""
    from recflex_amd.tuning.measure import emitted_tile_bytes, tiles_per_feature
    from recflex_amd.tuning.tuner import Tuner, TuneConfig
    off = np.arange(0, 16385 * 10, 10, dtype=np.int64)      # 16 384 bags of 10 lookups
    args = ([off] * 4, [516] * 4, [516] * 4, [4] * 4)       # 89 MiB each
    # 355 MiB on 256 workgroups: 5.5 tiles of 256 KiB each; on 1 280: 64 KiB and more
    assert tiles_per_feature(*args, emitted_tile_bytes(262144), grid_blocks=256) == \
        tiles_per_feature(*args, 262144, grid_blocks=256)
    assert tiles_per_feature(*args, emitted_tile_bytes(262144), grid_blocks=1280) == \
        tiles_per_feature(*args, 65536, grid_blocks=1280) != tiles_per_feature(*args, 262144, grid_blocks=1280)
    assert emitted_tile_bytes(65536) == 65536 and emitted_tile_bytes(0) == 0

    class Sched:
        class meta:
            row_bytes, embed_dim = 512, 128

        @staticmethod
        def TileGranularity(params):
            return 4

    tuner = Tuner.__new__(Tuner)
    tuner.num_feats, tuner.batches = 4, [[(None, off)] for _ in range(4)]
    cfg = TuneConfig(occupancies=[5], gpu_ids=[0], sm_count=256)
    tiles = tuner.sample_tiles([(Sched, None)] * 4, 5, 262144, cfg)
    assert tiles.tolist() == tiles_per_feature(*args, 65536, grid_blocks=1280)


def test_the_sweep_times_the_library_that_ships(monkeypatch, tmp_path):
    """A tile size beyond 64 KiB is tried as the library emitted with it would run each batch."""
    import torch
    from recflex_amd import rec_modules
    from recflex_amd.tuning import measure
    seen = []

    class Layer:
        class lib:
            embed_dims, dtypes = [128] * 4, [0] * 4
            get_max_concurrent_blocks = staticmethod(lambda: 1280)

        def __init__(self, *args, **kwargs):
            pass

        def bind_inputs(self, indices, offsets):
            return offsets

        def forward_indices(self, indices, offsets=None, tile_bytes=0, **kwargs):
            if offsets is None:
                seen.append((indices[0].numel() - 1, tile_bytes))

    monkeypatch.setattr(rec_modules, "FeatEmbed", Layer)
    monkeypatch.setattr(measure, "_pin_gpu", lambda gpu_id: None)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(measure, "make_table", lambda *args, **kwargs: None)
    monkeypatch.setattr(torch.Tensor, "to", lambda self, device: self)
    monkeypatch.setattr(measure, "_timed_launches", lambda run, repeats: run() or 1.0)
    small, large = (np.arange(0, n * 10 + 1, 10, dtype=np.int32) for n in (16384, 163840))
    monkeypatch.setattr(measure, "load_batches", lambda path: [(small, small), (large, large)])
    out = str(tmp_path / "t.txt")
    for size in (0, 32768, 262144):
        seen.clear()
        measure.measure_kernel_events("lib", [(1, 1)] * 4, ["float"] * 4, ["x"] * 4, out, size, 0, 1, 1)
        assert set(seen) == {(16384, min(size, 65536)), (163840, size)}


def test_launch_tile_bytes_counts_as_the_emitter_does():
    """Rows without the padding of int8 tables, indices, output rows and offsets."""
    from recflex_amd import prebuilt
    from recflex_amd.code_emitter.codegen import BAG_FIXED_BYTES, INDEX_BYTES
    from recflex_amd.librecom import RecomLib
    from recflex_amd.tuning import measure
    for name in ("edge", "c5s"):
        lib = RecomLib(prebuilt.ensure_built(name))
        lib.get_max_concurrent_blocks = lambda: 3
        metas = [s.meta for s, _ in prebuilt.model_spec(name).feat_schedules]
        off = [np.array([0, 70000 + 13 * f, 99991], np.int64) for f in range(len(metas))]
        total = measure.batch_traffic(off, [m.row_bytes + INDEX_BYTES for m in metas],
                                      [m.embed_dim * 4 + BAG_FIXED_BYTES for m in metas])
        assert 5 * 3 * 65536 < total
        assert measure.launch_tile_bytes(lib, off, 1 << 30) == measure.capped_tile_bytes(1 << 30, total, 3) < 1 << 30
