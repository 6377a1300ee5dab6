"""GPU parity of a library emitted with outlier tiles (bags found ahead of the kernel and summed
by several workgroups)."""

import numpy as np
import pytest

from helpers import oracle_output, require_lib

pytestmark = pytest.mark.gpu

CAP, PARTS = 4096, 16384      # rfx::kOutlierCap, rfx::kOutlierPartCap


def _inject(rng, wl, indices, offsets, plan):
    """plan: {feature: [extra lookups, ...]} -- each entry lengthens one random bag; an int
    instead of a list lengthens every bag of the feature."""
    indices, offsets = list(indices), list(offsets)
    for f, extras in plan.items():
        lens = np.diff(offsets[f]).astype(np.int64)
        if isinstance(extras, int):
            lens += extras
            extras = []
        for extra in extras:
            lens[rng.integers(0, wl.batch)] += extra
        off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        indices[f] = rng.integers(0, wl.features[f].rows, int(off[-1])).astype(np.int32)
        offsets[f] = off
    return indices, offsets


def _outlier_space(layer):
    """The ticket counters of the parts (rfx::OutlierTickets: eight, 128 bytes apart) and the list
    behind them, at the end of the workspace."""
    ws = layer.workspace.cpu().numpy()
    at = len(ws) - (32 + 4 * CAP + CAP + PARTS + PARTS * 128)
    return ws[at - 8 * 32:at], ws[at:]


@pytest.mark.parametrize("case", ["none", "few", "many", "overflow", "mid", "mid_overflow"])
def test_outlier_tiles_are_bit_exact(case):
    """No outlier at all; a few bags of 300 to 20 000 lookups in features of every kind of
    schedule; some hundred outliers; more than the list holds (4 096), where the launch falls back
    to a wavefront per outlier; some hundred mid-size bags (beyond their schedule's reach, below
    the outlier threshold: they go through the workgroup's list in LDS to whichever wavefront
    has time); every bag of twenty features mid-size, more than that list holds (192 per
    workgroup), where a bag is summed by the wavefront that met it.  Three launches each on one
    workspace, whose list header and arrival counters must be back at zero afterwards.
    Integer-valued tables: bit for bit."""
    import torch
    from recflex_amd import prebuilt
    from recflex_amd.rec_modules import FeatEmbed
    from recflex_amd.workloads import gen_inputs, gen_tables

    spec = prebuilt.model_spec("c3s_outliers")
    wl = spec.workload
    assert wl.table_values == "integer"
    assert sum(type(s).__name__ == "SplitBagSchedule" for s, _ in spec.feat_schedules) == 10
    dev = torch.device("cuda", 0)
    print(f"[case] c3s_outliers {case}: F={wl.num_features} B={wl.batch}", flush=True)
    tables = gen_tables(wl, dev)
    host_tables = [t.cpu().numpy() for t in tables]
    layer = FeatEmbed(dev, embed_tables=tables, librecom=require_lib("c3s_outliers"))
    assert layer.workspace is not None
    rng = np.random.default_rng(len(case))
    base_idx, base_off = gen_inputs(wl)
    for launch in range(3):
        feats = rng.permutation(wl.num_features)
        if case == "none":
            plan = {}
        elif case == "few":
            plan = {int(f): [int(x)] for f, x in zip(feats[:6], (300, 2000, 20000, 4200, 5000, 9000))}
        elif case == "many":
            plan = {int(f): [2000 + 371 * k for k in range(12)] for f in feats[:10]}
        elif case == "overflow":
            plan = {int(f): 2500 for f in feats[:60]}
        elif case == "mid":
            plan = {int(f): [70 + 13 * k for k in range(40)] for f in feats[:12]}
        else:
            plan = {int(f): 90 + 7 * int(f) % 60 for f in feats[:20]}
        indices, offsets = _inject(rng, wl, base_idx, base_off, plan)
        d_idx = [torch.from_numpy(i).to(dev) for i in indices]
        d_off = [torch.from_numpy(o).to(dev) for o in offsets]
        got = layer.forward_indices(d_idx, d_off).cpu().numpy()
        want = oracle_output(wl, host_tables, indices, offsets)
        bad = np.argwhere(got.view(np.uint32) != want.view(np.uint32))
        assert bad.size == 0, f"launch {launch}: {len(bad)} elements differ, first at {bad[:5].tolist()}"
        # the outlier space follows the split regions of every tenth feature: header (32 ints),
        # CAP entries of 4 ints, CAP counters, PARTS part -> entry, PARTS slots of 128 floats
        tickets, ws = _outlier_space(layer)
        assert not ws[:3].any(), f"launch {launch}: list header not cleared: {ws[:6].tolist()}"
        assert not tickets.any(), f"launch {launch}: ticket counters not reset: {tickets[::32].tolist()}"
        assert not ws[32 + 4 * CAP:32 + 5 * CAP].any(), f"launch {launch}: arrival counters not reset"
        # what the launch found: bags beyond their schedule's threshold and 128 KiB of traffic
        # (split-bag features take bags of any length themselves)
        expect = 0
        for (sched, params), feat, off in zip(spec.feat_schedules, wl.features, offsets):
            if sched.LongBagThreshold(params) > 0:
                thr = max(sched.LongBagThreshold(params), -(-131072 // (4 * feat.dim + 4)))
                expect += int((np.diff(off) > thr).sum())
        assert int(ws[3]) == expect, (int(ws[3]), expect)
        if case == "overflow":
            assert expect > CAP
        elif case in ("few", "many"):
            assert 0 < expect <= CAP and int(ws[4]) >= expect


# (bags, workgroups (0: the library's own grid), outlier bags in each of how many features, their
# lookups, ticket counters): one counter where the parts outnumber the workgroups or where there are
# fewer than eight of those, else eight, which a grid that is no multiple of eight shares unevenly;
# batches of one and two rounds of a finding workgroup (2 048 bags, eight a thread), and one beyond
@pytest.mark.parametrize("bags, grid, outliers, feats, lookups, counters", [
    (192, 1, 3, 4, 3000, 1), (192, 7, 3, 4, 3000, 1), (192, 16, 6, 8, 9000, 1), (192, 100, 3, 4, 3000, 8),
    (192, 1003, 12, 10, 6000, 8), (192, 0, 30, 30, 20000, 1), (257, 0, 5, 10, 3000, 8), (2048, 0, 20, 8, 2500, 8),
    (2049, 12, 60, 6, 2500, 1), (4100, 0, 20, 8, 2500, 8)])
def test_outlier_tickets_and_finding(bags, grid, outliers, feats, lookups, counters):
    """Outliers at bags spread over the whole batch, the first and the last one among them, two
    launches on one workspace with other bags each: bit for bit, the list is what the bags' lengths
    say, and every counter is back at zero."""
    import torch
    from recflex_amd import prebuilt
    from recflex_amd.rec_modules import FeatEmbed
    from recflex_amd.workloads import gen_inputs, gen_tables

    spec = prebuilt.model_spec("c3s_outliers")
    wl = spec.workload._replace(batch=bags, features=tuple(
        f._replace(mean_bag=min(f.mean_bag, 3.0)) for f in spec.workload.features))
    dev = torch.device("cuda", 0)
    print(f"[case] c3s_outliers B={bags} grid={grid} {feats} x {outliers} x {lookups}", flush=True)
    tables = gen_tables(wl, dev)
    host_tables = [t.cpu().numpy() for t in tables]
    layer = FeatEmbed(dev, embed_tables=tables, librecom=require_lib("c3s_outliers"))
    workgroups = grid or layer.lib.get_max_concurrent_blocks()
    thresholds = [max(s.LongBagThreshold(p), -(-131072 // (4 * f.dim + 4))) if s.LongBagThreshold(p) > 0 else 0
                  for (s, p), f in zip(spec.feat_schedules, wl.features)]
    listing = [f for f, thr in enumerate(thresholds) if 0 < thr < lookups]
    assert len(listing) >= feats
    rng = np.random.default_rng(bags + grid)
    indices, offsets = map(list, gen_inputs(wl))
    short = [np.diff(o).astype(np.int64) for o in offsets]
    for launch in range(2):
        expect_bags = expect_parts = 0
        chosen = rng.choice(listing, feats, replace=False)
        for f, lens in enumerate(short):
            lens = lens.copy()
            if f in chosen:
                lens[np.linspace(0, bags - 1, outliers).astype(int)] = lookups + rng.integers(0, 300, outliers)
            offsets[f] = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
            indices[f] = rng.integers(0, wl.features[f].rows, int(offsets[f][-1])).astype(np.int32)
            if thresholds[f]:
                long = lens[lens > thresholds[f]]
                expect_bags += len(long)
                expect_parts += int(np.minimum(64, -(-long * (4 * wl.features[f].dim + 4) // 262144)).sum())
        assert 0 < expect_bags <= CAP and expect_parts <= PARTS
        assert counters == (8 if workgroups >= 8 and expect_parts < workgroups else 1)
        got = layer.forward_indices([torch.from_numpy(i).to(dev) for i in indices],
                                    [torch.from_numpy(o).to(dev) for o in offsets], grid_blocks=grid).cpu().numpy()
        want = oracle_output(wl, host_tables, indices, offsets)
        bad = np.argwhere(got.view(np.uint32) != want.view(np.uint32))
        assert bad.size == 0, f"launch {launch}: {len(bad)} elements differ, first at {bad[:5].tolist()}"
        tickets, ws = _outlier_space(layer)
        assert not ws[:3].any() and not tickets.any(), (launch, ws[:3].tolist(), tickets[::32].tolist())
        assert not ws[32 + 4 * CAP:32 + 5 * CAP].any(), f"launch {launch}: arrival counters not reset"
        assert ws[3:5].tolist() == [expect_bags, expect_parts]


def test_outliers_beyond_one_round_of_the_finding_grid():
    """More bags than the finding kernel's 64 workgroups per feature look at in one round of 2 048
    each: nearly all of them empty, long ones at both ends and around the seam."""
    import torch
    from recflex_amd import prebuilt
    from recflex_amd.rec_modules import FeatEmbed
    from recflex_amd.workloads import gen_tables

    spec = prebuilt.model_spec("c3s_outliers")
    wl = spec.workload
    bags, seam = 64 * 2048 + 300, 64 * 2048
    at = np.array([0, 255, 256, 2047, 2048, seam - 1, seam, seam + 257, bags - 1])
    dev = torch.device("cuda", 0)
    print(f"[case] c3s_outliers B={bags}", flush=True)
    tables = gen_tables(wl, dev)
    layer = FeatEmbed(dev, embed_tables=tables, librecom=require_lib("c3s_outliers"))
    rng = np.random.default_rng(9)
    lens = np.zeros(bags, np.int64)
    indices, offsets, few = [], [], []
    for f, (sched, params) in enumerate(spec.feat_schedules):
        lens[at] = 3000 if sched.LongBagThreshold(params) > 0 and wl.features[f].dim >= 32 else 2
        offsets.append(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32))
        indices.append(rng.integers(0, wl.features[f].rows, int(offsets[f][-1])).astype(np.int32))
        few.append(np.concatenate([[0], np.cumsum(lens[at])]).astype(np.int32))
    got = layer.forward_indices([torch.from_numpy(i).to(dev) for i in indices],
                                [torch.from_numpy(o).to(dev) for o in offsets])
    want = oracle_output(wl._replace(batch=len(at)), [t.cpu().numpy() for t in tables], indices, few)
    rows = torch.from_numpy(at).to(dev)
    assert np.array_equal(got[rows].cpu().numpy(), want)
    got[rows] = 0
    assert int(torch.count_nonzero(got)) == 0
    tickets, ws = _outlier_space(layer)
    assert not ws[:3].any() and not tickets.any()
    assert int(ws[3]) == len(at) * sum(int(f[1]) == 3000 for f in few)


@pytest.mark.parametrize("name", ["c4s_outliers", "c5s_outliers"])
@pytest.mark.parametrize("case", ["few", "mid"])
def test_outlier_tiles_on_fp16_and_int8_rows(name, case):
    """The block-wide parts, the workgroup's list of mid-size bags and the wavefront that sums
    them, on fp16 and int8 rows (scale and bias, staged output): a few bags of 300 to 20 000
    lookups, and some hundred bags between their schedule's reach and the outlier threshold.
    Two launches on one workspace; integer-valued tables, bit for bit."""
    import torch
    from recflex_amd import prebuilt
    from recflex_amd.rec_modules import FeatEmbed
    from recflex_amd.workloads import gen_inputs, gen_tables

    spec = prebuilt.model_spec(name)
    wl = spec.workload
    assert wl.table_values == "integer"
    dev = torch.device("cuda", 0)
    print(f"[case] {name} {case}: F={wl.num_features} B={wl.batch}", flush=True)
    tables = gen_tables(wl, dev)
    host_tables = [t.cpu().numpy() for t in tables]
    layer = FeatEmbed(dev, embed_tables=tables, librecom=require_lib(name))
    assert layer.lib.info.outliers == 1 and layer.workspace is not None
    rng = np.random.default_rng(len(name) + len(case))
    base_idx, base_off = gen_inputs(wl)
    for launch in range(2):
        feats = rng.permutation(wl.num_features)
        if case == "few":
            plan = {int(f): [int(x)] for f, x in zip(feats[:6], (300, 2000, 20000, 4200, 5000, 9000))}
        else:
            plan = {int(f): [70 + 13 * k for k in range(30)] for f in feats[:8]}
        indices, offsets = _inject(rng, wl, base_idx, base_off, plan)
        got = layer.forward_indices([torch.from_numpy(i).to(dev) for i in indices],
                                    [torch.from_numpy(o).to(dev) for o in offsets]).cpu().numpy()
        want = oracle_output(wl, host_tables, indices, offsets)
        bad = np.argwhere(got.view(np.uint32) != want.view(np.uint32))
        assert bad.size == 0, f"launch {launch}: {len(bad)} elements differ, first at {bad[:5].tolist()}"
