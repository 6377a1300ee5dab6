"""Schedule templates for the gfx950 fused embedding kernel.

``SCHEDULE_MAPPING`` plays the role of ``globals()`` of the reference's ``examples/tune.py``
(``tune.py:78`` passes it as ``schedule_mapping``): class name in ``schedule_config.txt`` ->
schedule class.
"""

from typing import Dict, NamedTuple, Tuple, Type

from recflex_amd.code_emitter.schedule_base import ScheduleBase, MetaData
from .team import (TeamParams, TeamScheduleBase, ThreadPerBagSchedule, ThreadPerBagParams,
                   SubWavefrontPerBagSchedule, SubWavefrontPerBagParams,
                   WavefrontPerBagSchedule, WavefrontPerBagParams, OneHotBagSchedule,
                   OneHotBagParams, next_pow2)
from .block_per_bag import BlockPerBagSchedule, BlockPerBagParams, SplitBagSchedule
from .reference_names import (OneHotSchedule, OneHotMultiBlockSchedule, WarpPerSampleSchedule,
                              OneBlockMultiSampleSchedule, MultiBlockPerSampleSchedule,
                              ReduceByKeySchedule, OneHotParams, OneHotMultiBlockParams,
                              WarpPerSampleParams, OneBlockMultiSampleParams,
                              MultiBlockPerSampleParams, ReduceByKeyParams)

SCHEDULE_MAPPING: Dict[str, Type[ScheduleBase]] = {
    cls.__name__: cls
    for cls in (ThreadPerBagSchedule, SubWavefrontPerBagSchedule, WavefrontPerBagSchedule,
                OneHotBagSchedule, BlockPerBagSchedule, SplitBagSchedule, OneHotSchedule, OneHotMultiBlockSchedule,
                WarpPerSampleSchedule, OneBlockMultiSampleSchedule,
                MultiBlockPerSampleSchedule, ReduceByKeySchedule)
}

PARAM_TYPES: Dict[str, Type[NamedTuple]] = {
    "ThreadPerBagSchedule": ThreadPerBagParams,
    "SubWavefrontPerBagSchedule": SubWavefrontPerBagParams,
    "WavefrontPerBagSchedule": WavefrontPerBagParams,
    "BlockPerBagSchedule": BlockPerBagParams,
    "SplitBagSchedule": BlockPerBagParams,
    "OneHotBagSchedule": OneHotBagParams,
    "OneHotSchedule": OneHotBagParams,
    "OneHotMultiBlockSchedule": OneHotBagParams,
    "WarpPerSampleSchedule": TeamParams,
    "OneBlockMultiSampleSchedule": TeamParams,
    "MultiBlockPerSampleSchedule": BlockPerBagParams,
    "ReduceByKeySchedule": BlockPerBagParams,
}


def default_schedule(meta: MetaData, mean_bag_len: float = 1.0, block_threads: int = 256,
                     one_hot: bool = False) -> Tuple[ScheduleBase, NamedTuple]:
    """Untuned starting point for one feature from its row size and mean bag length
    (``one_hot``: no bag of the feature is known to hold more than one lookup -- the row-copy
    template): enough
    column lanes that a lane owns one or two 16-byte vectors, lookup lanes only for long bags,
    and eight row vectors in flight per lane, four for fp16 and int8 rows with their 8 or 16
    accumulators per vector, half as many of fp32 and int8 rows where the bags hold few lookups
    (measured at four workgroups per CU, us per launch with half as many in flight and with
    these: 1 000 fp32 features 85 and 79 at 256 samples, 31.9 and 27.6 at 64; 100 fp32 features
    318 and 313 at 6 000; 200 int8 features 1 529 and 1 404 at 16 384, 17.1 and 14.7 at 64.  Eight
    for fp16 rows: 400 features 388 instead of 394 at 512 samples, but 4 624 instead of 4 299 at
    8 192; for int8 rows 13.7 and 1 461.  200 features with bags of 1.8 lookups, 4 096 / 16 384
    samples, half as many and not: fp16 116 / 405 and 110 / 394, int8 126 / 528 and 129 / 540, fp32
    134 / 502 and 132 / 495)."""
    if one_hot:
        sched = OneHotBagSchedule(meta, block_threads)
        return sched, sched.default_params()
    v = meta.row_vectors
    x = min(64, next_pow2(v))
    if v > 1 and x * meta.vec_bytes >= 256 and mean_bag_len < 8:
        x //= 2                      # short bags of wide rows: two vectors per lane
    vpl = -(-v // x)
    acc_floats = vpl * meta.elems_per_vector          # accumulators of one bag per lane
    if mean_bag_len <= 1.5:
        bags = 4 if 4 * acc_floats <= 16 else (2 if 2 * acc_floats <= 16 else 1)
        team = x
        if team == 1:
            return ThreadPerBagSchedule(meta, block_threads), ThreadPerBagParams(1, bags, vpl)
        if team == 64:
            return WavefrontPerBagSchedule(meta, block_threads), WavefrontPerBagParams(64, 1, vpl)
        return (SubWavefrontPerBagSchedule(meta, block_threads),
                SubWavefrontPerBagParams(x, 1, 1, bags, vpl))
    if mean_bag_len >= 96 and meta.payload_bytes >= 512 and vpl * meta.elems_per_vector < 16:
        # long bags of wide rows: fewer column lanes, each with 16 accumulators (4 fp32 or 2 fp16
        # vectors), so that four (two) times as many lookups are in flight per wavefront -- the
        # move the production-build climb makes first on C3 (fp32, D=128) and C4 (fp16, D=256)
        vpl = max(1, 16 // meta.elems_per_vector)
        x = max(1, next_pow2(v) // vpl)
        vpl = -(-v // x)
    if mean_bag_len < 24:
        y = 1
    elif mean_bag_len < 96:
        y = max(1, min(4, 64 // x))
    else:
        y = max(1, 64 // x)
    if mean_bag_len >= 512 and next_pow2(v) >= 4:
        # the whole workgroup on one bag, one row vector per lane -- and several workgroups per
        # bag when the batch holds so few bags that one of them is a good part of a workgroup's
        # share (8 features x 64 bags x 4 000 lookups: 105 us against 203 us with a team per bag);
        # eight lookups in flight per lane for fp32 rows (8 features, 1 bag of 28 000 lookups 17.8 us
        # with four and 16.0, 16 of 20 000 73.5 and 72.2, 128 of 2 000 61.4 and 60.9), four where a
        # lane has more than two vectors of them: eight spill (8 features, 16 bags of 4 000: 512
        # columns 154 us either way, 768 247 with four and 261, 1 024 340 and 382)
        lanes = min(64, next_pow2(v))
        items = 2 if meta.elems_per_vector > 4 else (8 if v <= 2 * lanes else 4)
        return SplitBagSchedule(meta, block_threads), BlockPerBagParams(lanes, items, 4 * block_threads)
    items = max(1, (8 if meta.elems_per_vector <= 4 else 4) // vpl)
    items = 1 << (items.bit_length() - 1)
    if items * y >= 2 * mean_bag_len and meta.elems_per_vector != 8:
        items = max(1, items // 2)
    team = x * y
    if team == 1:
        return ThreadPerBagSchedule(meta, block_threads), ThreadPerBagParams(items, 1, vpl)
    if team == 64:
        return WavefrontPerBagSchedule(meta, block_threads), WavefrontPerBagParams(x, items, vpl)
    return (SubWavefrontPerBagSchedule(meta, block_threads),
            SubWavefrontPerBagParams(x, y, items, 1, vpl))


def schedule_from_config(entry: dict, meta: MetaData, block_threads: int = 256
                         ) -> Tuple[ScheduleBase, NamedTuple]:
    """Inverse of ``CodeEmitter.serialize_config`` for one feature:
    ``{"schedule": ClassName, "params": {...}}`` -> (schedule object, params tuple)."""
    name = entry["schedule"]
    if name not in SCHEDULE_MAPPING:
        raise KeyError(f"unknown schedule class {name!r}")
    return SCHEDULE_MAPPING[name](meta, block_threads), PARAM_TYPES[name](**entry["params"])
